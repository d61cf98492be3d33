// FP32 emissivity lookups: the chains of lookup_f64.hip with FP32 table
// interpolation.
//
// Precision plan (budget: 0.01 K brightness temperature against FP64):
//  * The state of a chain is the path emissivity eps_path = 1 - tau_path.
//    The reference's update tau_path *= 1 - eps with eps = 1 - (1 - eps00) /
//    tau_path makes tau_path exactly 1 - eps00, so eps_path = eps00 carries
//    no accumulated rounding, and small emissivities keep full relative
//    precision in float where 1 - tau_path would not.  (It is summed with the
//    rounding error carried; see cell_interp.)
//  * The emissivity-growth step u_eq = u(eps_path), eps00 = eps(u_eq + u_seg)
//    runs along the column's piecewise-linear curve (ega_step_fast): inside a
//    bracket eps00 = eps_path + u_seg deps/du, and across its upper knot it
//    continues with the next slope, so no column density is formed.  (Before,
//    both lookups were evaluated one after the other, relative to the
//    bracket's knot: 62.7 ms per 4096 x 32 x 12 limb batch of three emitters
//    against 51 ms, 27.2 against 19.4 ms for 1000 nadir paths of 256 channels
//    and eight emitters.)
//  * Output is the path emissivity eps_path after each segment (the radiance
//    kernel forms the segment emissivity (eps_i - eps_{i-1}) / (1 - eps_{i-1});
//    the adjoint restarts any segment from eps_{i-1}); 1 marks an opaque
//    path (tau_path below float resolution).
//  * For the FP32 EGA Jacobian over monotone tables (PART), each step also
//    stores its partials d eps_path / d (eps_prev, p, T, u_seg) with the
//    slopes of the brackets it used (see adjoint.hip), so that the reverse
//    chains need no table access.
#include "jur_device.hpp"

namespace jur {

// LOS field f of point ip: wave-uniform block base, 32-bit lane offset
#define LOSR(f, ip) ld32(losb, ((unsigned)(ip) * nfield + (unsigned)(f)) * WAVE + ln)

// The three knots from bracket g of the column with knot 0 at ko on: one
// 24-byte stretch; g is brought into the column's slots.
__device__ __forceinline__ void load_knots(const float2 *knb, int gtop, unsigned ko, int &g, float4 &a, float2 &b) {
  g = g < -1 ? -1 : (g > gtop ? gtop : g);
  const unsigned k = ko + g;
  const char *at = (const char *)knb + (size_t)(k * (unsigned)sizeof(float2));
  const Knots2 v = *(const Knots2 *)at;
  a = make_float4(v.x, v.y, v.z, v.w);
  b = *(const float2 *)(at + 16);
}

// The corners' brackets when the cell moves: a column that the cell keeps
// takes its bracket along, a new one extrapolates from the pair.  fwd, bwd: by
// one pressure; d0, d1: by so many temperatures on its two pressures.
template <int RL>
__device__ __forceinline__ void carry_brackets(int *gi, int sub, bool fwd, bool bwd, int d0, int d1) {
  if constexpr (RL == 1) {
    if (fwd || bwd) {
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const int lo = gi[c], hi = gi[c + 2];
        gi[c] = fwd ? hi : 2 * lo - hi;
        gi[c + 2] = fwd ? 2 * hi - lo : lo;
      }
    }
    const int lo0 = gi[0], hi0 = gi[1], lo1 = gi[2], hi1 = gi[3];
    gi[0] = d0 == 1 ? hi0 : (d0 == -1 ? 2 * lo0 - hi0 : lo0);
    gi[1] = d0 == 1 ? 2 * hi0 - lo0 : (d0 == -1 ? lo0 : hi0);
    gi[2] = d1 == 1 ? hi1 : (d1 == -1 ? 2 * lo1 - hi1 : lo1);
    gi[3] = d1 == 1 ? 2 * hi1 - lo1 : (d1 == -1 ? lo1 : hi1);
  } else {
    const int o2 = quad_xor<2>(gi[0]);
    if (fwd || bwd) gi[0] = (sub < 2) == fwd ? o2 : 2 * gi[0] - o2;
    const int o1 = quad_xor<1>(gi[0]);
    const int d = sub < 2 ? d0 : d1;
    if (d == 1 || d == -1) gi[0] = ((sub & 1) != 0) == (d < 0) ? o1 : 2 * gi[0] - o1;
  }
}

// The four corners' values from the lanes of a quad.
__device__ __forceinline__ void gather_quad(float v, float *out) {
  out[0] = quad_lane<0>(v);
  out[1] = quad_lane<1>(v);
  out[2] = quad_lane<2>(v);
  out[3] = quad_lane<3>(v);
}

template <typename V>
__device__ __forceinline__ V pick(const V *v, int c) {
  return c == 0 ? v[0] : (c == 1 ? v[1] : (c == 2 ? v[2] : v[3]));
}

// The path emissivity from the corners' values (linear in T with weights w0,
// w1 on the cell's two pressures, then in p with wp; MAX(MIN(eps00, 1), 0)):
// their growths over ep with GROW (EGA), added with the rounding error rest of
// the last sum (half an ulp of ep per point would be some 1e-6 of it over a
// path), or the emissivities themselves.  With PART, the step's partials d
// eps_path / d (eps_prev, p, T, u_seg) (the slopes in T and p are those of
// either).
template <bool PART, bool GROW>
__device__ __forceinline__ float cell_interp(const float *ec, const float *dep, const float *deu, float w0, float w1,
                                             float wp, float dt0, float dt1, float dwp, float ep, float &rest,
                                             float4 &dpart) {
  const float a = __builtin_fmaf(ec[1] - ec[0], w0, ec[0]);
  const float b = __builtin_fmaf(ec[3] - ec[2], w1, ec[2]);
  float en = __builtin_fmaf(b - a, wp, a);
  if (GROW) {
    const float y = en + rest;
    en = ep + y;
    rest = y - (en - ep);
  }
  if constexpr (PART) {
    // the bilinear cell weights and their T and p slopes
    const float q0 = 1.f - wp, q1 = wp;
    const float cw[4] = {q0 * (1.f - w0), q0 * w0, q1 * (1.f - w1), q1 * w1};
    const float tw[4] = {-q0 * dt0, q0 * dt0, -q1 * dt1, q1 * dt1};
    const float pw[4] = {-(1.f - w0) * dwp, -w0 * dwp, (1.f - w1) * dwp, w1 * dwp};
    float sdep = 0.f, sdu = 0.f, sdt = 0.f, sdp = 0.f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      sdep += cw[c] * dep[c];
      sdu += cw[c] * deu[c];
      sdt += tw[c] * ec[c];
      sdp += pw[c] * ec[c];
    }
    // a clamped emissivity is constant
    dpart = (en < 0.f || en > 1.f) ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(sdep, sdp, sdt, sdu);
  }
  if (GROW && (en < 0.f || en > 1.f)) rest = 0.f;
  en = (en < 1.f) ? en : 1.f;
  return (en > 0.f) ? en : 0.f;
}

// eps(cu) on one column (CGA), from the knots in hand: the bracket g or the
// next one; ok is false for longer walks and beyond the last knot.  The
// bracket is the one of cu rounded to float, as the knots are (the curve is
// continuous); the distance from its lower knot is taken in FP64.
__device__ __forceinline__ void cga_step_fast(const float4 &a, const float2 &b, double cu, float cuf, int &g,
                                              float &ec, bool &ok) {
  const bool up = cuf >= a.z;
  const float u0 = up ? a.z : a.x, e0 = up ? a.w : a.y, u1 = up ? b.x : a.z, e1 = up ? b.y : a.w;
  ok = cuf >= u0 && cuf < u1;
  ec = e0 + fdiv(e1 - e0, u1 - u0) * (float)(cu - (double)u0);
  if (up) g++;
}

// The general lookup: CGA, tables on different grids, columns that are not
// monotone, cells without data.
// RL lanes per chain as in k_lookup_f32_cell (EGA).  MONO: every table's columns
// are monotone (TabView::all_mono); the bisections cost the others registers.
template <bool CGA, bool PART, int RL, bool MONO>
__global__ __launch_bounds__(WAVE, 4) void k_lookup_f32(ModelView M, BatchView B, LosView L,
                                                     EpsView E, const RayInfo *info, int blk0,
                                                     int nblk) {
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
  const bool wr = sub == 0;
  const int ir = (blk0 + bl) * WAVE + ln;
  if (ir >= B.nray) return;
  const TabView &T = M.tab;
  const int tix = ig * nd + id;
  const int npt = T.np[tix];
  if (npt < 30) return;
  const RayInfo R = info[ir];
  if (R.status != JUR_OK) return;

  // wave-uniform bases (the ray block's LOS and emissivity chain, the
  // table's arrays) with 32-bit per-lane offsets
  const double *losb = L.los + (size_t)bl * L.cap * L.nfield * WAVE;
  const unsigned nfield = L.nfield;
  const int npb = E.npb[bl];
  float *outb = (float *)E.eps + E.off[bl] + ((size_t)id * ng + ig) * npb * WAVE;
  float4 *partb = PART ? E.part + E.off[bl] + ((size_t)id * ng + ig) * npb * WAVE : nullptr;
  const bool mono = MONO || T.mono[tix];
  const int pdir = T.pdir[tix];
  const double *pg = T.p + (size_t)tix * T.TP;
  const int *ntp = T.nt + (size_t)tix * T.TP;
  const size_t tcols = (size_t)T.TP * T.TT;  // (p, T) columns per table
  const double *tgb = T.t + (size_t)tix * tcols;
  const int *nub = T.nu + (size_t)tix * tcols;
  const float2 *knb = T.kn + (size_t)tix * tcols * T.TS;

  float ep = 0.f, rest = 0.f;  // path emissivity and its last sum's rounding error
  double cu = 0, cp = 0, ct = 0;
  constexpr int NC = RL == 1 ? 4 : 1;  // the lane's corners
  int gi[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) gi[c] = -1;
  const int gtop = T.TU - 2;

  // cached cell
  int ipr = -1, it0 = -1, it1 = -1;
  double pa = 0, pb = 0, rpa = 0;
  bool plog = false;
  float wp_scale = 0, g00 = 0, gi0 = 0, g10 = 0, gi1 = 0;
  float ta0 = 0, dt0 = 0, ta1 = 0, dt1 = 0, lpr = 0;
  int nt0 = 0, nt1 = 0;
  bool full = false;  // every corner column has two knots
  unsigned tq0 = 0;  // first T-grid entry of p row ipr

  // LOS values of the current point; the next point's are loaded after the
  // corner records of the current one, so that waiting for the records does
  // not wait for the (HBM) LOS loads as well
  double p = 0, t = 0, useg = 0;
  if (R.np > 0) {
    p = LOSR(F_P, 0);
    t = LOSR(F_T, 0);
    useg = LOSR(L.f_u + ig, 0);
  }
  int ip = 0;
  for (; ip < R.np; ip++) {
    const int ipn = ip + 1 < R.np ? ip + 1 : ip;
    if (CGA) {
      cu += useg;
      cp += useg * p;
      ct += useg * t;
    }
    const double rcu = CGA ? rcp_d(cu) : 0.0;
    const double pq = CGA ? cp * rcu : p;
    const float tq = (float)(CGA ? ct * rcu : t);
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
      carry_brackets<RL>(gi, sub, iprev >= 0 && ipr == iprev + 1, ipr == iprev - 1, 0, 0);
      pa = pg[ipr];
      pb = pg[ipr + 1];
      wp_scale = frcp((float)(pb - pa));
      if (CGA) {
        // LOGX in p where both ratios are positive
        plog = pb / pa > 0;
        lpr = (float)(1.0 / log(pb / pa));
        rpa = 1.0 / pa;
      }
      nt0 = ntp[ipr];
      nt1 = ntp[ipr + 1];
      tq0 = (unsigned)ipr * T.TT;
      const double t00 = ld32(tgb, tq0), t01 = ld32(tgb, tq0 + 1);
      const double t10 = ld32(tgb, tq0 + T.TT), t11 = ld32(tgb, tq0 + T.TT + 1);
      g00 = (float)t00;
      gi0 = frcp((float)(t01 - t00));
      g10 = (float)t10;
      gi1 = frcp((float)(t11 - t10));
      it0 = it1 = -2;
    }
    double pn = p, tn = t, un = useg;
    float4 dpart = make_float4(1.f, 0.f, 0.f, 0.f);  // a cell without data: e_new = e_prev
    if (nt0 >= 2 && nt1 >= 2) {
      int j0 = (int)((tq - g00) * gi0);
      j0 = j0 < 0 ? 0 : (j0 > nt0 - 2 ? nt0 - 2 : j0);
      int j1 = (int)((tq - g10) * gi1);
      j1 = j1 < 0 ? 0 : (j1 > nt1 - 2 ? nt1 - 2 : j1);
      if (j0 != it0 || j1 != it1) {
        carry_brackets<RL>(gi, sub, false, false, j0 - it0, j1 - it1);
        it0 = j0;
        it1 = j1;
        const double a0 = ld32(tgb, tq0 + it0), b0 = ld32(tgb, tq0 + it0 + 1);
        const double a1 = ld32(tgb, tq0 + T.TT + it1), b1 = ld32(tgb, tq0 + T.TT + it1 + 1);
        ta0 = (float)a0;
        dt0 = frcp((float)(b0 - a0));
        ta1 = (float)a1;
        dt1 = frcp((float)(b1 - a1));
        full = ld32(nub, tq0 + it0) >= 2 && ld32(nub, tq0 + it0 + 1) >= 2 && ld32(nub, tq0 + T.TT + it1) >= 2 &&
               ld32(nub, tq0 + T.TT + it1 + 1) >= 2;
      }
      if (full) {
        // the corner's column of the table and its knot 0
        auto column = [&](int c) { return (c < 2 ? tq0 + it0 : tq0 + T.TT + it1) + (c & 1); };
        auto knot0 = [&](int c) { return column(c) * T.TS + 1; };
        const float us = (float)useg, key = ega_key<PART>(ep, rest);
        float e1[NC], dep1[NC], deu1[NC];
        float4 ka[NC];
        float2 kb[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) e1[c] = dep1[c] = deu1[c] = 0.f;
        if (mono) {
#pragma unroll
          for (int c = 0; c < NC; c++) load_knots(knb, gtop, knot0(RL == 1 ? c : sub), gi[c], ka[c], kb[c]);
          __builtin_amdgcn_sched_barrier(0);
        }
        pn = LOSR(F_P, ipn);
        tn = LOSR(F_T, ipn);
        un = LOSR(L.f_u + ig, ipn);
        __builtin_amdgcn_sched_barrier(0);
        int bad = (1 << NC) - 1;
        if (mono) {
          bad = 0;
#pragma unroll
          for (int c = 0; c < NC; c++) {
            bool ok;
            if (CGA) cga_step_fast(ka[c], kb[c], cu, (float)cu, gi[c], e1[c], ok);
            else ega_step_fast<PART>(ka[c], kb[c], ep, rest, key, us, gi[c], e1[c], dep1[c], deu1[c], ok);
            bad |= ok ? 0 : 1 << c;
          }
        }
        // the corners left, one at a time for each lane
        while (bad) {
          const int c = RL == 1 ? __ffs(bad) - 1 : 0;
          const Col col{knb + knot0(RL == 1 ? c : sub)};
          const int n = ld32(nub, column(RL == 1 ? c : sub));
          int g;
          if constexpr (RL == 1) g = pick(gi, c);
          else g = gi[0];
          float e, de = 0.f, du = 0.f;
          if (!mono) {
            e = CGA ? col_eps_bis(col, n, cu) : col_eps_bis(col, n, col_u_bis(col, n, ep) + useg) - ep;
          } else if (CGA) {
            float4 r;
            g = col_walk_f<0>(col, n, (float)cu, g, r);
            e = eps_from_rec_f(r, cu);
            if ((float)cu < r.x) g = -1;
          } else {
            e = ega_step_slow<PART>(col, n, ep, rest, useg, g, de, du);
          }
#pragma unroll
          for (int q = 0; q < NC; q++)
            if (q == c) {
              e1[q] = e;
              gi[q] = g;
              dep1[q] = de;
              deu1[q] = du;
            }
          bad &= bad - 1;
        }
        float ec[4], dep[4], deu[4];
        if constexpr (RL == 1) {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            ec[c] = e1[c];
            dep[c] = dep1[c];
            deu[c] = deu1[c];
          }
        } else {
          gather_quad(e1[0], ec);
          if (PART) {
            gather_quad(dep1[0], dep);
            gather_quad(deu1[0], deu);
          }
        }
        const float w0 = (tq - ta0) * dt0;
        const float w1 = (tq - ta1) * dt1;
        float wp;
        if (CGA)
          wp = (plog && pq * rpa > 0) ? __logf((float)(pq * rpa)) * lpr : (float)(pq - pa) * wp_scale;
        else
          wp = (float)(pq - pa) * wp_scale;
        ep = cell_interp<PART, !CGA>(ec, dep, deu, w0, w1, wp, dt0, dt1, wp_scale, ep, rest, dpart);
      } else {
        pn = LOSR(F_P, ipn);
        tn = LOSR(F_T, ipn);
        un = LOSR(L.f_u + ig, ipn);
      }
    } else {
      pn = LOSR(F_P, ipn);
      tn = LOSR(F_T, ipn);
      un = LOSR(L.f_u + ig, ipn);
    }
    if (wr) {
      st32(outb, (unsigned)ip * WAVE + ln, ep);
      if (PART) st32(partb, (unsigned)ip * WAVE + ln, dpart);
    }
    if (ep >= 1.f) {
      // tau_path below float resolution: every later segment is opaque too
      if (wr)
        for (ip++; ip < R.np; ip++) st32(outb, (unsigned)ip * WAVE + ln, 1.f);
      break;
    }
    p = pn;
    t = tn;
    useg = un;
  }
}

// EGA on tables that share their pressure and temperature grids, monotone and
// without empty cells (LosView::cell): k_ray_points has located the cell of
// every LOS point once for all chains of the ray, and a step is its cell's
// record (columns and weights), the knots and the arithmetic on them.  Same
// operations as the general kernel, so the same bits.
//
// Against the general kernel (which searched the cell again in each chain and
// kept its grids and column sizes in registers: 4 wavefronts per SIMD, 7 here):
// 51.1 -> 33.9 ms per 4096 x 32 x 12 limb batch of three emitters, 19.4 ->
// 12.0 ms for 1000 nadir paths of 256 channels and eight emitters, and for 77
// x 5 limb rays on quads 2.01 -> 1.26 ms.
//
// RL lanes per chain.  RL = 4 (small batches, where a wavefront's chain is
// the kernel's duration): the four lanes of a (ray, channel, emitter) chain
// each take one corner of the cell's step and exchange the corners' results
// by DPP; every lane then does the same operations on the same values as one
// lane would, so the emissivities are the same to the last bit, and the first
// lane writes them.  A wavefront covers a quarter of a 64-ray block.
template <bool PART, int RL>
__global__ __launch_bounds__(WAVE) void k_lookup_f32_cell(ModelView M, BatchView B, LosView L, EpsView E,
                                                          const RayInfo *info, int blk0, int nblk) {
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
  const bool wr = sub == 0;
  const int ir = (blk0 + bl) * WAVE + ln;
  if (ir >= B.nray) return;
  const TabView &T = M.tab;
  const int tix = ig * nd + id;
  if (T.np[tix] < 30) return;
  const RayInfo R = info[ir];
  if (R.status != JUR_OK || R.np <= 0) return;

  // wave-uniform bases with 32-bit per-lane offsets
  const double *losb = L.los + (size_t)bl * L.cap * L.nfield * WAVE;
  const unsigned nfield = L.nfield;
  const unsigned fu = L.f_u + ig;
  constexpr unsigned CW = PART ? 2 : 1;  // float4 per cell record
  const float4 *cellb = L.cell + (size_t)bl * L.cap * CW * WAVE;
  const int npb = E.npb[bl];
  float *outb = (float *)E.eps + E.off[bl] + ((size_t)id * ng + ig) * npb * WAVE;
  float4 *partb = PART ? E.part + E.off[bl] + ((size_t)id * ng + ig) * npb * WAVE : nullptr;
  const float2 *knb = T.kn + (size_t)tix * T.TP * T.TT * T.TS;
  const int *nub = T.nu + (size_t)tix * T.TP * T.TT;
  const int TT = T.TT, TS = T.TS, gtop = T.TU - 2;

  constexpr int NC = RL == 1 ? 4 : 1;  // the lane's corners
  float ep = 0.f, rest = 0.f;  // path emissivity and its last sum's rounding error
  int gi[NC];
  unsigned ko[NC];  // knot 0 of the corners' columns
#pragma unroll
  for (int c = 0; c < NC; c++) {
    gi[c] = -1;
    ko[c] = 1;
  }
  int cell = -1, c00 = -1, c10 = -1;
  auto column = [&](int c) { return (c < 2 ? c00 : c10) + (c & 1); };

  float4 cc = ld32(cellb, ln * CW), ds = PART ? ld32(cellb, ln * CW + 1) : make_float4(0.f, 0.f, 0.f, 0.f);
  double useg = LOSR(fu, 0);
  int ip = 0;
  for (; ip < R.np; ip++) {
    const unsigned ipn = ip + 1 < R.np ? ip + 1 : ip;
    if (__float_as_int(cc.x) != cell) {
      cell = __float_as_int(cc.x);
      const int o00 = c00, o10 = c10;
      c00 = cell & 0xffff;
      c10 = (int)((unsigned)cell >> 16);
      const bool fwd = c00 == o10, bwd = c10 == o00, p = fwd || bwd;
      carry_brackets<RL>(gi, sub, fwd, bwd, p ? 0 : c00 - o00, p ? 0 : c10 - o10);
#pragma unroll
      for (int c = 0; c < NC; c++) ko[c] = (unsigned)column(RL == 1 ? c : sub) * TS + 1;
    }
    float4 ka[NC];
    float2 kb[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) load_knots(knb, gtop, ko[c], gi[c], ka[c], kb[c]);
    __builtin_amdgcn_sched_barrier(0);
    // the next point's inputs behind the knots, so that waiting for the knots
    // does not wait for HBM as well
    const float4 cn = ld32(cellb, (ipn * WAVE + ln) * CW);
    const float4 dn = PART ? ld32(cellb, (ipn * WAVE + ln) * CW + 1) : ds;
    const double un = LOSR(fu, ipn);
    __builtin_amdgcn_sched_barrier(0);
    const float us = (float)useg, key = ega_key<PART>(ep, rest);
    float e1[NC], dep1[NC], deu1[NC];
    int bad = 0;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      bool ok;
      dep1[c] = deu1[c] = 0.f;
      ega_step_fast<PART>(ka[c], kb[c], ep, rest, key, us, gi[c], e1[c], dep1[c], deu1[c], ok);
      if (!ok) {
        if (ega_above<PART>(ka[c], kb[c], ep, rest)) e1[c] = ega_step_above<PART>(ka[c].z, ka[c].w, ep, us, dep1[c], deu1[c]);
        else bad |= 1 << c;
      }
    }
    // the corners left, one at a time for each lane
    while (bad) {
      const int c = RL == 1 ? __ffs(bad) - 1 : 0;
      const int q = column(RL == 1 ? c : sub);
      int g;
      if constexpr (RL == 1) g = pick(gi, c);
      else g = gi[0];
      float de, du;
      const float e = ega_step_slow<PART>(Col{knb + ((unsigned)q * TS + 1)}, nub[q], ep, rest, useg, g, de, du);
#pragma unroll
      for (int k = 0; k < NC; k++)
        if (k == c) {
          e1[k] = e;
          gi[k] = g;
          if (PART) {
            dep1[k] = de;
            deu1[k] = du;
          }
        }
      bad &= bad - 1;
    }
    float ec[4], dep[4], deu[4];
    if constexpr (RL == 1) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        ec[c] = e1[c];
        dep[c] = dep1[c];
        deu[c] = deu1[c];
      }
    } else {
      gather_quad(e1[0], ec);
      if (PART) {
        gather_quad(dep1[0], dep);
        gather_quad(deu1[0], deu);
      }
    }
    float4 dpart;
    ep = cell_interp<PART, true>(ec, dep, deu, cc.y, cc.z, cc.w, ds.x, ds.y, ds.z, ep, rest, dpart);
    if (wr) {
      st32(outb, (unsigned)ip * WAVE + ln, ep);
      if (PART) st32(partb, (unsigned)ip * WAVE + ln, dpart);
    }
    if (ep >= 1.f) {
      // tau_path below float resolution: every later segment is opaque too
      if (wr)
        for (ip++; ip < R.np; ip++) st32(outb, (unsigned)ip * WAVE + ln, 1.f);
      break;
    }
    cc = cn;
    ds = dn;
    useg = un;
  }
}

void launch_lookup_f32(const ModelView &M, const BatchView &B, const LosView &L, const EpsView &E,
                       const RayInfo *info, int blk0, int nblk, hipStream_t s) {
  if (M.nd * M.ng == 0) return;
  const unsigned chains = (unsigned)padded_blocks(nblk) * M.nd * M.ng;
  auto run = [&](auto kernel, int rl) {
    hipLaunchKernelGGL(kernel, dim3(chains * rl), dim3(WAVE), 0, s, M, B, L, E, info, blk0, nblk);
  };
  if (M.formod == 0) {
    M.tab.all_mono ? run(k_lookup_f32<true, false, 1, true>, 1) : run(k_lookup_f32<true, false, 1, false>, 1);
    return;
  }
  // small batches: four lanes per chain while that stays within the
  // wavefronts that run at once (five per SIMD for the kernel with most
  // registers)
  const bool quad = chains <= 5120 / 4;
  if (L.cell) {
    if (quad) E.part ? run(k_lookup_f32_cell<true, 4>, 4) : run(k_lookup_f32_cell<false, 4>, 4);
    else E.part ? run(k_lookup_f32_cell<true, 1>, 1) : run(k_lookup_f32_cell<false, 1>, 1);
  } else if (E.part) {  // partials are stored for monotone tables only
    quad ? run(k_lookup_f32<false, true, 4, true>, 4) : run(k_lookup_f32<false, true, 1, true>, 1);
  } else if (M.tab.all_mono) {
    quad ? run(k_lookup_f32<false, false, 4, true>, 4) : run(k_lookup_f32<false, false, 1, true>, 1);
  } else {
    quad ? run(k_lookup_f32<false, false, 4, false>, 4) : run(k_lookup_f32<false, false, 1, false>, 1);
  }
}

}  // namespace jur
