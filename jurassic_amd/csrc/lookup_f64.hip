// FP64 emissivity lookups (intpol_tbl_ega, src/jurassic.c:3799-3891, and
// intpol_tbl_cga, :3710-3795), one independent chain per (ray, channel,
// emitter).
//
// The EGA recurrence couples the segments of one ray only through each
// emitter's own path transmittance tau_path[id][ig]; emitters and channels
// are independent.  So one wavefront handles one (block of 64 rays, channel,
// emitter), a lane per ray, and writes the segment emissivity eps of every
// LOS point to the emissivity buffer; the radiance kernel combines the
// emitters as the reference does (tau_seg *= 1 - eps in emitter order).
//
// A lane keeps tau_path, its table cell and, per corner, the bracket of the
// inverse lookup u(1 - tau_path).  Along a ray consecutive segments mostly
// stay in the same cell and bracket, so:
//  * cell data (pressure bracket, temperature grids and their reciprocal
//    spacings, column sizes) are reloaded only when the cell changes, and a
//    column that the cell keeps takes its bracket along;
//  * a corner's four knots from the previous segment's bracket on are loaded
//    first, and cover the inverse lookup moving up one knot and the grown
//    column the next one (ega_step64); the next point's LOS values are loaded
//    behind them, so that waiting for the knots does not wait for HBM.
// Every search returns the reference's index and the arithmetic is the
// reference's (built with -ffp-contract=off), except that the cell's weights
// multiply by reciprocals kept with the cell where LIN divides (an ulp or so).
// The temperature index truncates such a product too, which may fall on the
// other side of a whole number than the reference's quotient (98 x (1 / 24.5) <
// 4): at a temperature of the grid that is another cell, and one of the two may
// hold no data.  So it divides where the product is close to a whole number
// (the check: 1.73 -> 1.75 ms per call of 10 nadir rays, 14.9 -> 15.0 ms per 512
// x 32 x 12 limb forward model).
// Large batches are bound by instruction issue (512 x 32 x 12 limb paths of
// three emitters: 10.3 ms, 14.9 ms with one walk per lookup and LIN's
// divisions), small ones by the latency of a point: its LOS load, its knots
// and its eight float quotients in series took 4.25 us; with the loads ahead
// and a quad's lanes sharing the quotients it is 0.84 us (10 nadir rays, 2
// channels, 805 points: 3.43 -> 0.67 ms).
#include "jur_device.hpp"

namespace jur {

#define LOSR(f, ip) LOS_AT(los, L, f, ip)

// locate_reg without its clamps: the truncated quotient of t - tg[0] and the
// spacing of the temperatures at tg.
__device__ __forceinline__ int reg_quotient(const double *tg, double t) {
  JUR_FP_EXACT
  return (int)((t - tg[0]) / (tg[1] - tg[0]));
}

// x within 1e-9 above a whole number or 4.8e-7 below one, by the high word of
// its fraction (NaN too).
__device__ __forceinline__ bool near_whole(double x) {
  constexpr unsigned lo = 0x3e112e0b, hi = 0x3fefffff;  // 1e-9, 1 - 2^-21
  return (unsigned)__double2hiint(__builtin_amdgcn_fract(x)) - lo >= hi - lo;
}

// PATH: store the path transmittance tau_path after each segment instead of
// the segment emissivity (the Jacobian restarts any segment from it).
// RL lanes per chain, as in the FP32 lookups: RL = 4 (small batches, where a
// wavefront's chain is the kernel's duration; EGA): each lane of a quad takes
// one corner of the cell, exchanged by DPP; the same operations on the same
// values, so the same bits.  A wavefront then covers a quarter of a block.
template <bool CGA, bool PATH, int RL = 1>
__global__ __launch_bounds__(WAVE) void k_lookup_f64(ModelView M, BatchView B, LosView L,
                                                     EpsView E, const RayInfo *info, int blk0,
                                                     int nblk) {
  JUR_FP_EXACT
  static_assert(RL == 1 || !CGA, "the four-lane chains are the EGA ones");
  const int nd = M.nd, ng = M.ng;
  int bl, rem;
  if (!xcd_block_map(blockIdx.x, nd * ng * RL, nblk, bl, rem)) return;
  const int qtr = rem % RL;
  rem /= RL;
  const int id = rem / ng;
  const int ig = rem - id * ng;
  const int lane = threadIdx.x;
  const int sub = lane % RL;  // the lane's corner (RL = 4)
  const int ln = RL == 1 ? lane : qtr * (WAVE / RL) + lane / RL;  // the ray's lane in its block
  const int ir = (blk0 + bl) * WAVE + ln;
  if (ir >= B.nray) return;
  const TabView &T = M.tab;
  const int tix = ig * nd + id;
  const int npt = T.np[tix];
  if (npt < 30) return;  // eps = 0 for every segment; the consumers know
  const RayInfo R = info[ir];
  if (R.status != JUR_OK) return;

  const double *los = L.los + (size_t)bl * L.cap * L.nfield * WAVE + ln;
  const int npb = E.npb[bl];
  double *out = (double *)E.eps + E.off[bl] + ((size_t)id * ng + ig) * npb * WAVE + ln;
  const int mono = T.mono[tix];
  const int pdir = T.pdir[tix];
  const double *pg = T.p + (size_t)tix * T.TP;
  const int *ntp = T.nt + (size_t)tix * T.TP;
  const double *tgb = T.t + (size_t)tix * T.TP * T.TT;
  const int *nub = T.nu + (size_t)tix * T.TP * T.TT;
  const float2 *knb = T.kn + (size_t)tix * T.TP * T.TT * T.TS + 1;
  const int gtop = T.TU - 2;

  constexpr int NC = RL == 1 ? 4 : 1;  // the lane's corners
  double tp = 1, cu = 0, cp = 0, ct = 0;
  int gi[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) gi[c] = CGA || !mono ? T.TU / 2 : -1;

  // cached cell
  int ipr = -1, it0 = -1, it1 = -1;
  double pa = 0, pb = 0, rp = 0, g00 = 0, r0 = 0, g10 = 0, r1 = 0;  // p bracket, T-grid starts and 1/spacings
  double ta0 = 0, rt0 = 0, ta1 = 0, rt1 = 0;
  int nt0 = 0, nt1 = 0;
  int tq0 = 0;          // first T-grid entry of p row ipr
  bool full = false;    // every corner column has two knots

  double p = 0, t = 0, useg = 0;
  if (R.np > 0) {
    p = LOSR(F_P, 0);
    t = LOSR(F_T, 0);
    useg = LOSR(L.f_u + ig, 0);
  }
  for (int ip = 0; ip < R.np; ip++) {
    const int ipn = ip + 1 < R.np ? ip + 1 : ip;
    if (CGA) {
      cu = cu + useg;
      cp = cp + useg * p;
      ct = ct + useg * t;
    }
    const bool opaque = tp < 1e-9;
    const double pq = CGA ? cp / cu : p;
    const double tq = CGA ? ct / cu : t;
    bool cell = false;
    float4 ka[NC], kb[NC];
    if (!opaque) {
      // pressure bracket (locate_irr): keep the cached one while it holds
      bool keep = false;
      if (ipr >= 0 && pdir != 0) {
        if (pdir > 0)
          keep = (ipr == 0 || !(pa > pq)) && (ipr == npt - 2 || pb > pq);
        else
          keep = (ipr == 0 || !(pa <= pq)) && (ipr == npt - 2 || pb <= pq);
      }
      if (!keep) {
        const int iprev = ipr;
        ipr = (pdir != 0 && ipr >= 0) ? irr_walk(pg, npt, pq, ipr, pdir) : locate_irr(pg, npt, pq);
        // a column that the cell keeps takes its bracket along, a new one
        // extrapolates from the pair
        const bool fwd = ipr == iprev + 1, bwd = ipr == iprev - 1;
        if (fwd || bwd) {
          if constexpr (RL == 1) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
              const int lo = gi[c], hi = gi[c + 2];
              gi[c] = fwd ? hi : 2 * lo - hi;
              gi[c + 2] = fwd ? 2 * hi - lo : lo;
            }
          } else {
            const int o = quad_xor<2>(gi[0]);
            gi[0] = (sub < 2) == fwd ? o : 2 * gi[0] - o;
          }
        }
        pa = pg[ipr];
        pb = pg[ipr + 1];
        rp = 1 / (pb - pa);
        nt0 = ntp[ipr];
        nt1 = ntp[ipr + 1];
        tq0 = ipr * T.TT;
        g00 = tgb[tq0];
        r0 = 1 / (tgb[tq0 + 1] - g00);
        g10 = tgb[tq0 + T.TT];
        r1 = 1 / (tgb[tq0 + T.TT + 1] - g10);
        it0 = it1 = -2;
      }
      cell = nt0 >= 2 && nt1 >= 2;
      if (cell) {
        // locate_reg on the two temperature rows
        const double x0 = (tq - g00) * r0, x1 = (tq - g10) * r1;
        int j0 = (int)x0, j1 = (int)x1;
        if (near_whole(x0) | near_whole(x1)) {
          j0 = reg_quotient(tgb + tq0, tq);
          j1 = reg_quotient(tgb + tq0 + T.TT, tq);
        }
        j0 = j0 < 0 ? 0 : (j0 > nt0 - 2 ? nt0 - 2 : j0);
        j1 = j1 < 0 ? 0 : (j1 > nt1 - 2 ? nt1 - 2 : j1);
        if (j0 != it0 || j1 != it1) {
          const int d0 = j0 - it0, d1 = j1 - it1;
          if constexpr (RL == 1) {
            const int lo0 = gi[0], hi0 = gi[1], lo1 = gi[2], hi1 = gi[3];
            if (d0 == 1) { gi[0] = hi0; gi[1] = 2 * hi0 - lo0; }
            if (d0 == -1) { gi[1] = lo0; gi[0] = 2 * lo0 - hi0; }
            if (d1 == 1) { gi[2] = hi1; gi[3] = 2 * hi1 - lo1; }
            if (d1 == -1) { gi[3] = lo1; gi[2] = 2 * lo1 - hi1; }
          } else {
            const int o = quad_xor<1>(gi[0]);
            const int d = sub < 2 ? d0 : d1;
            if (d == 1) gi[0] = (sub & 1) ? 2 * gi[0] - o : o;
            if (d == -1) gi[0] = (sub & 1) ? o : 2 * gi[0] - o;
          }
          it0 = j0;
          it1 = j1;
          ta0 = tgb[tq0 + it0];
          rt0 = 1 / (tgb[tq0 + it0 + 1] - ta0);
          ta1 = tgb[tq0 + T.TT + it1];
          rt1 = 1 / (tgb[tq0 + T.TT + it1 + 1] - ta1);
          full = nub[tq0 + it0] >= 2 && nub[tq0 + it0 + 1] >= 2 && nub[tq0 + T.TT + it1] >= 2 &&
                 nub[tq0 + T.TT + it1 + 1] >= 2;
        }
        cell = full;
      }
    }
    // the corner's column of the table
    auto column = [&](int c) {
      return (c < 2 ? tq0 + it0 : tq0 + T.TT + it1) + (c & 1);
    };
    if (cell && !CGA && mono) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        gi[c] = gi[c] < -1 ? -1 : (gi[c] > gtop ? gtop : gi[c]);
        const Col k{knb + (size_t)column(RL == 1 ? c : sub) * T.TS};
        ka[c] = k[gi[c]];
        kb[c] = k[gi[c] + 2];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const double pn = LOSR(F_P, ipn), tn = LOSR(F_T, ipn), un = LOSR(L.f_u + ig, ipn);
    __builtin_amdgcn_sched_barrier(0);
    double eps = opaque ? 1 : 0;
    if (cell) {
      double e[4] = {0, 0, 0, 0};
      if (!CGA && mono) {
        const double x = 1 - tp;
        double ec[NC];
        int bad = 0;
#pragma unroll
        for (int c = 0; c < NC; c++) {
          bool ok;
          ec[c] = ega_step64(ka[c], kb[c], x, useg, gi[c], ok);
          bad |= ok ? 0 : 1 << c;
        }
        // the corners left, one at a time for each lane
        while (bad) {
          int c = 0, g = gi[0];
          if constexpr (RL == 1) {
            c = __ffs(bad) - 1;
            g = c == 0 ? gi[0] : (c == 1 ? gi[1] : (c == 2 ? gi[2] : gi[3]));
          }
          const int q = column(RL == 1 ? c : sub);
          const double v = ega_slow64(Col{knb + (size_t)q * T.TS}, nub[q], x, useg, g);
#pragma unroll
          for (int k = 0; k < NC; k++)
            if (k == c) {
              ec[k] = v;
              gi[k] = g;
            }
          bad &= bad - 1;
        }
        if constexpr (RL == 1) {
#pragma unroll
          for (int c = 0; c < 4; c++) e[c] = ec[c];
        } else {
          e[0] = quad_lane<0>(ec[0]);
          e[1] = quad_lane<1>(ec[0]);
          e[2] = quad_lane<2>(ec[0]);
          e[3] = quad_lane<3>(ec[0]);
        }
      } else {
        if constexpr (CGA) {
          if (mono) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
              const int q = column(c);
              float4 r;
              gi[c] = col_walk<0>(Col{knb + (size_t)q * T.TS}, nub[q], cu, gi[c], r);
              e[c] = eps_from_rec(r, cu);
            }
          }
        }
        if (!mono) {
#pragma unroll 1
          for (int c = 0; c < 4; c++) {
            const int q = column(c), n = nub[q];
            const Col k{knb + (size_t)q * T.TS};
            int g2 = 0;
            const double v = CGA ? col_eps(k, n, cu, 0, g2)
                                 : col_eps(k, n, col_u(k, n, 1 - tp, 0, g2) + useg, 0, g2);
            e[0] = c == 0 ? v : e[0];
            e[1] = c == 1 ? v : e[1];
            e[2] = c == 2 ? v : e[2];
            e[3] = c == 3 ? v : e[3];
          }
        }
      }
      const double w0 = (tq - ta0) * rt0, w1 = (tq - ta1) * rt1;
      double e00 = e[0] + (e[1] - e[0]) * w0;
      const double e11 = e[2] + (e[3] - e[2]) * w1;
      e00 = CGA ? logx(pa, e00, pb, e11, pq) : e00 + (e11 - e00) * ((pq - pa) * rp);
      e00 = (e00 < 1) ? e00 : 1;  // MAX(MIN(eps00, 1), 0)
      e00 = (e00 > 0) ? e00 : 0;
      eps = 1 - (1 - e00) / tp;
    }
    tp *= (1 - eps);
    if (sub == 0) out[(size_t)ip * WAVE] = PATH ? tp : eps;
    p = pn;
    t = tn;
    useg = un;
  }
}

void launch_lookup_f64(const ModelView &M, const BatchView &B, const LosView &L, const EpsView &E,
                       const RayInfo *info, int blk0, int nblk, bool path, hipStream_t s) {
  if (M.nd * M.ng == 0) return;
  const size_t chains = (size_t)padded_blocks(nblk) * M.nd * M.ng;
  const dim3 grid(chains), blk(WAVE);
  if (M.formod == 0) {
    if (path) hipLaunchKernelGGL((k_lookup_f64<true, true>), grid, blk, 0, s, M, B, L, E, info, blk0, nblk);
    else hipLaunchKernelGGL((k_lookup_f64<true, false>), grid, blk, 0, s, M, B, L, E, info, blk0, nblk);
  } else if (chains * 4 <= 4096) {
    // small batches: four lanes per chain while that stays within the four
    // wavefronts per SIMD its registers allow
    const dim3 g4(chains * 4);
    if (path) hipLaunchKernelGGL((k_lookup_f64<false, true, 4>), g4, blk, 0, s, M, B, L, E, info, blk0, nblk);
    else hipLaunchKernelGGL((k_lookup_f64<false, false, 4>), g4, blk, 0, s, M, B, L, E, info, blk0, nblk);
  } else {
    if (path) hipLaunchKernelGGL((k_lookup_f64<false, true>), grid, blk, 0, s, M, B, L, E, info, blk0, nblk);
    else hipLaunchKernelGGL((k_lookup_f64<false, false>), grid, blk, 0, s, M, B, L, E, info, blk0, nblk);
  }
}

}  // namespace jur
