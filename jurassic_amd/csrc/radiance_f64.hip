// FP64 radiance kernel: combines the per-emitter segment emissivities of the
// lookup kernel with continua and the source function and accumulates
// radiance and transmittance along each line of sight (formod_pencil,
// src/jurassic.c:3233-3334).
//
// One wavefront per (block of 64 rays, channel), lane = ray.  Every segment
// field is read with one coalesced access per wavefront.
//
// The segments' emissivities and source functions do not depend on each
// other, only the sums do.  A small batch, whose duration is one path's, forms
// them on the PW = 8 waves of a workgroup, RAD64_PT points each per round, and
// adds them in path order on the first wave: the same operations in the same
// order as on one wave, so the same bits (0.63 -> 0.1 ms for 10 nadir rays of
// 805 points; joining the sums of chunks, as the FP32 kernel does, would
// round differently from the reference).
//
// Built with -ffp-contract=off; operation order follows the reference,
// except that the per-segment continua and source function multiply by
// reciprocals (1/T, 1/ds, the grid's inverse spacing, constants folded at
// compile time) where the reference divides, and the H2O continuum's power
// and tanh are evaluated through exp/expm1 (jur_device.hpp, CtmChan):
// radiances within a few ulp of the reference expressions.
#include "jur_device.hpp"

namespace jur {

constexpr int RAD64_PT = 8;

#define LOSR(f, ip) LOS_AT(los, L, f, ip)

template <int PW>
__global__ __launch_bounds__(WAVE *PW) void k_radiance_f64(ModelView M, BatchView B, LosView L,
                                                       EpsView E, const RayInfo *info, int blk0,
                                                       int nblk, double *rad_out, double *tau_out) {
  JUR_FP_EXACT
  const int nd = M.nd, ng = M.ng;
  int bl, id;
  if (!xcd_block_map(blockIdx.x, nd, nblk, bl, id)) return;
  const int lane = threadIdx.x % WAVE;
  const int wv = PW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  // lanes without a ray follow the last one (the waves meet at barriers) and
  // write nothing, as do rays that could not be traced, whose atmosphere index
  // may be out of range: they read the first atmosphere
  const bool live = (blk0 + bl) * WAVE + lane < B.nray;
  const int ir = live ? (blk0 + bl) * WAVE + lane : B.nray - 1;
  RayInfo R = info[ir];
  const bool ok = live && R.status == JUR_OK;
  const bool write = ok && wv == 0;
  if (!ok) R.np = 0;

  const atm_t *atm = &B.atm[ok ? B.ray_prof[ir] : 0];
  const ChanInfo C = M.chan[id];
  const double nu = C.nu;
  const double *los = L.los + (size_t)bl * L.cap * L.nfield * WAVE + lane;
  const int npb = E.npb[bl];
  const double *eps_g = (const double *)E.eps + E.off[bl] + (size_t)id * ng * npb * WAVE + lane;
  const double *sr_col = M.sr + (size_t)id * TBLNS;
  const double inv_dst = 1 / (M.st[1] - M.st[0]);

  double kcl = 0;
  if (L.f_cl >= 0 && M.ncl > 0)
    kcl = lin(M.clnu[C.icl], atm->clk[C.icl], M.clnu[C.icl + 1], atm->clk[C.icl + 1], nu);
  double sfeps = 1.0;
  if (M.nsf > 0)
    sfeps = lin(M.sfnu[C.isf], atm->sfeps[C.isf], M.sfnu[C.isf + 1], atm->sfeps[C.isf + 1], nu);
  const bool has_k = C.window < M.nw;
  const CtmChan K = ctm_chan(M.ctm, nu);

  // emitters with a table (the others have eps = 0)
  unsigned gmask = 0;
  for (int g = 0; g < ng; g++)
    if (M.tab.np[g * nd + id] >= 30) gmask |= 1u << g;
  struct Point {
    double p, t, ds, e[4];
  };
  // what a point's arithmetic begins with: p, t, ds and its first four emitters
  auto load = [&](int ip) {
    Point x;
    x.p = LOSR(F_P, ip);
    x.t = LOSR(F_T, ip);
    x.ds = LOSR(F_DS, ip);
#pragma unroll
    for (int g = 0; g < 4; g++) x.e[g] = g < ng && (gmask >> g & 1u) ? eps_g[((size_t)g * npb + ip) * WAVE] : 0.0;
    return x;
  };

  // a = src eps and s = 1 - eps of a segment (0 and 1 for one that adds nothing)
  auto segment = [&](int ip, const Point &x, double &a, double &s) {
    const double p = x.p, t = x.t, ds = x.ds;
    // tau_seg = prod_g (1 - eps_g), emitter order (intpol_tbl_ega)
    double tau_gas = 1;
#pragma unroll
    for (int g = 0; g < 4; g++) tau_gas *= (1 - x.e[g]);
    for (int g = 4; g < ng; g++)
      if (gmask >> g & 1u) tau_gas *= (1 - eps_g[((size_t)g * npb + ip) * WAVE]);

    // formod_continua (src/jurassic.c:3075-3117)
    const double rt = 1 / t, rds = 1 / ds;
    double beta = has_k ? LOSR(L.f_k + C.window, ip) : 0.0;
    if (L.f_cl >= 0) beta += LOSR(L.f_cl, ip) * kcl;
    if (M.ig_co2 >= 0) beta += ctmco2_seg(K, p, t, LOSR(L.f_u + M.ig_co2, ip)) * rds;
    if (M.ig_h2o >= 0)
      beta += ctmh2o_seg(K, nu, p, t, rt, LOSR(F_Q0 + M.ig_h2o, ip), LOSR(L.f_u + M.ig_h2o, ip)) * rds;
    if (M.ctm_n2) beta += ctmn2_seg(K, p, t, rt);
    if (M.ctm_o2) beta += ctmo2_seg(K, p, rt);

    const double src = srcfunc_u(M.st, inv_dst, sr_col, t);
    a = 0;
    s = 1;
    if (tau_gas > 0) {
      const double eps = 1 - tau_gas * exp(-beta * ds);
      a = src * eps;
      s = 1 - eps;
    }
  };

  double rad = 0, tau = 1, drefl = 0;
  // the down-welling sum of the reflection term is accumulated forward:
  // D = sum_i src_i eps_i prod_{k>i} (1 - eps_k)
  auto add = [&](double a, double s) {
    rad += a * tau;
    tau *= s;
    drefl = drefl * s + a;
  };
  if constexpr (PW == 1) {
    for (int ip = 0; ip < R.np; ip++) {
      double a, s;
      segment(ip, load(ip), a, s);
      add(a, s);
    }
  } else {
    extern __shared__ double2 seg[];  // [points of a round][lane]
    constexpr int RP = PW * RAD64_PT;
    for (int r0 = 0; r0 < npb; r0 += RP) {
      const int i0 = r0 + wv * RAD64_PT;
      const int i1 = i0 + RAD64_PT < R.np ? i0 + RAD64_PT : R.np;
      Point nx{};
      if (i0 < i1) nx = load(i0);
      for (int ip = i0; ip < i1; ip++) {
        const Point x = nx;
        nx = load(ip + 1 < i1 ? ip + 1 : ip);
        double2 v;
        segment(ip, x, v.x, v.y);
        seg[(ip - r0) * WAVE + lane] = v;
      }
      __syncthreads();
      if (wv == 0) {
        const int n = R.np - r0 < RP ? R.np - r0 : RP;
        for (int k = 0; k < n; k++) {
          const double2 v = seg[k * WAVE + lane];
          add(v.x, v.y);
        }
      }
      __syncthreads();
    }
  }

  if (!write) return;
  // surface emission, reflection and solar term (src/jurassic.c:3262-3328)
  if (M.sftype >= 1 && R.sft > 0) {
    const double src_sf = srcfunc(M.st, sr_col, R.sft);
    rad += sfeps * src_sf * tau;
    if (M.sftype >= 2 && sfeps < 1) {
      rad += drefl * tau * (1 - sfeps);
      if (M.sftype >= 3 && R.pad > 0)
        rad += 6.764e-5 / (2. * JUR_PI) * C.planck_sun * tau * (1 - sfeps) * tau * R.rcos;
    }
  }
  rad_out[(size_t)ir * nd + id] = rad;
  tau_out[(size_t)ir * nd + id] = tau;
}

void launch_radiance_f64(const ModelView &M, const BatchView &B, const LosView &L, const EpsView &E,
                         const RayInfo *info, int blk0, int nblk, double *rad, double *tau,
                         hipStream_t s) {
  if (M.nd == 0) return;
  const unsigned g = (unsigned)padded_blocks(nblk) * M.nd;
  // eight waves a path while all workgroups run at once (one per CU, whose LDS
  // and registers hold two)
  if (g <= 512)
    hipLaunchKernelGGL(k_radiance_f64<8>, dim3(g), dim3(8 * WAVE), 8 * RAD64_PT * WAVE * sizeof(double2), s, M, B, L, E,
                       info, blk0, nblk, rad, tau);
  else
    hipLaunchKernelGGL(k_radiance_f64<1>, dim3(g), dim3(WAVE), 0, s, M, B, L, E, info, blk0, nblk, rad, tau);
}

}  // namespace jur
