// Ray tracing (FP64) and hydrostatic equilibrium on the device.
//
// k_raytrace marches each line of sight through its own atmosphere exactly as
// raytrace (src/jurassic.c:4201-4438) does and writes the altitude and the
// trapezoid step length of every LOS point: the march is a serial chain of
// FP64 operations per step, so nothing that a step does not need for the next
// one is done in it.  k_ray_finish clips the last step, finds the tangent
// point (tangent_point, src/jurassic.c:5223-5263) and the solar-incidence
// factor of formod_pencil (src/jurassic.c:3297-3326).  k_ray_points then
// fills in the atmosphere at the points, in parallel over them.
// Built with -ffp-contract=off: every operation rounds as in the reference.
#include "jur_device.hpp"

namespace jur {

// Level search of intpol_atm: the bisection of locate_irr, or, for a
// strictly monotone altitude grid, a walk from the previous point's level
// (the LOS moves by a fraction of a level per step), which returns the same
// index.
// anp is atm->np, read once by the caller: a load of it in the march would
// wait (vmcnt) for the LOS stores issued before it.
__device__ __forceinline__ int atm_level(const atm_t *atm, int anp, int zdir, double z, int &g) {
  g = (zdir != 0 && g >= 0) ? irr_walk(atm->z, anp, z, g, zdir) : locate_irr(atm->z, anp, z);
  return g;
}

// A level (index ip) loaded ahead.
struct LevelAhead {
  int ip = -1;
  double z = 0, p = 0, t = 0;
};

// Pressure and temperature interpolation of intpol_atm
// (src/jurassic.c:3685-3706) with the level-pair coefficients cached: LOGY
// evaluates y0 exp(log(y1/y0)/(x1-x0) (x-x0)) and LIN y0 + (y1-y0)/(x1-x0)
// (x-x0); the quotients depend only on the two levels, so keeping them while
// the ray stays between the same levels gives bit-identical values.
struct LevelCache {
  int ip = -1;
  // the altitudes [lo, hi) for which a walk from this pair returns it: its
  // levels', open at the ends of the grid; empty for a grid that is not
  // strictly monotone (search by bisection)
  double lo = 1, hi = 0;
  double z0 = 0, dz = 0, p0 = 0, pq = 0, t0 = 0, tq = 0;
  bool plog = false;
  double z1 = 0, p1 = 0, t1 = 0;
  __device__ __forceinline__ bool holds(double z) const { return lo <= z && z < hi; }
  __device__ __forceinline__ void range(int anp, int zdir) {
    lo = ip == (zdir > 0 ? 0 : anp - 2) ? -INFINITY : (zdir > 0 ? z0 : z1);
    hi = ip == (zdir > 0 ? anp - 2 : 0) ? INFINITY : (zdir > 0 ? z1 : z0);
  }
  // To the pair of z, not held by this one.  A path leaves a pair into its
  // neighbour: that takes one level, loaded ahead when the pair before was
  // entered (a search reads a level at a time, each a round trip to memory
  // behind the march's stores).
  __device__ __forceinline__ void enter(const atm_t *atm, int anp, int zdir, double z, LevelAhead &ah) {
    JUR_FP_EXACT
    bool found = false, up = false;
    if (ip >= 0 && zdir != 0) {
      up = (z >= hi) == (zdir > 0);
      const int f = up ? ip + 2 : ip - 1;
      if (f >= 0 && f < anp) {
        double zf = ah.z, pf = ah.p, tf = ah.t;
        if (ah.ip != f) {
          zf = atm->z[f];
          pf = atm->p[f];
          tf = atm->t[f];
        }
        ip = up ? ip + 1 : ip - 1;
        const double zs = up ? z1 : z0, ps = up ? p1 : p0, ts = up ? t1 : t0;
        z0 = up ? zs : zf;
        p0 = up ? ps : pf;
        t0 = up ? ts : tf;
        z1 = up ? zf : zs;
        p1 = up ? pf : ps;
        t1 = up ? tf : ts;
        range(anp, zdir);
        found = holds(z);
      }
    }
    if (!found) {
      int g = ip;
      ip = atm_level(atm, anp, zdir, z, g);
      z0 = atm->z[ip];
      z1 = atm->z[ip + 1];
      p0 = atm->p[ip];
      p1 = atm->p[ip + 1];
      t0 = atm->t[ip];
      t1 = atm->t[ip + 1];
      if (zdir != 0) range(anp, zdir);
    }
    const int f = up ? ip + 2 : ip - 1;
    ah.ip = f >= 0 && f < anp ? f : ip;
    ah.z = atm->z[ah.ip];
    ah.p = atm->p[ah.ip];
    ah.t = atm->t[ah.ip];
    dz = z1 - z0;
    plog = (p1 / p0 > 0);
    pq = plog ? log(p1 / p0) / dz : (p1 - p0) / dz;
    tq = (t1 - t0) / dz;
  }
  __device__ __forceinline__ double p(double z) const {
    JUR_FP_EXACT
    // (the exponential is taken in either case: without the branch the
    // evaluations at several altitudes overlap)
    const double x = pq * (z - z0), e = exp(plog ? x : 0);
    return plog ? p0 * e : p0 + x;
  }
  __device__ __forceinline__ double t(double z) const {
    JUR_FP_EXACT
    return t0 + tq * (z - z0);
  }
};

// Square root and quotient for the march, where no operand is near the ends
// of the exponent range (radii, unit vectors, pressures over temperatures):
// Goldschmidt's and Newton's iterations from the hardware estimates, each
// ending in a correction by the exact residual, round as sqrt and / do without
// the scaling around them (the compiler's forms take 6 and 3 instructions
// more).
__device__ __forceinline__ double sqrt_mid(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  double s = a * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  s = __builtin_fma(__builtin_fma(-s, s, a), h, s);
  return __builtin_fma(__builtin_fma(-s, s, a), h, s);
}
__device__ __forceinline__ double div_mid(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
  r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// Altitude of a Cartesian point: the z output of cart2geo
// (src/jurassic.c:108-119), for the refraction probes, which use nothing else.
__device__ __forceinline__ double cart2z(const double *x) {
  JUR_FP_EXACT
  return sqrt_mid(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]) - JUR_RE;
}

// sza (src/jurassic.c:5183-5219).
__device__ __forceinline__ double sza(double sec, double lon, double lat) {
  JUR_FP_EXACT
  const double D = sec / 86400 - 0.5;
  const double g = (357.529 + 0.98560028 * D) * (JUR_PI / 180.0);
  const double q = 280.459 + 0.98564736 * D;
  const double L = (q + 1.915 * sin(g) + 0.020 * sin(2 * g)) * (JUR_PI / 180.0);
  const double e = (23.439 - 0.00000036 * D) * (JUR_PI / 180.0);
  const double dec = asin(sin(e) * sin(L));
  const double ra = atan2(cos(e) * sin(L), cos(L));
  const double GMST = 18.697374558 + 24.06570982441908 * D;
  const double LST = GMST + lon / 15;
  const double h = LST / 12 * JUR_PI - ra;
  const double latr = lat * (JUR_PI / 180.0);
  return acos(sin(latr) * sin(dec) + cos(latr) * cos(dec) * cos(h)) * (180.0 / JUR_PI);
}

#define LOSW(f, ip) LOS_AT(base, L, f, ip)
// RL lanes per ray.  RL = 4 (small batches, where a wavefront's march is the
// kernel's duration): the four lanes of a ray march it together and each
// evaluates one of the four refraction probes of a step, which the lanes
// then exchange by DPP; every lane does the same operations on the same
// values, so the LOS is the same to the last bit, and the first lane writes
// it.  A wavefront then covers a quarter of a 64-ray block.
template <int RL>
__global__ __launch_bounds__(WAVE) void k_raytrace(ModelView M, BatchView B, LosView L,
                                                   RayInfo *info, RayTail *tail, int blk0) {
  JUR_FP_EXACT
  const int lane = threadIdx.x;
  const int lb = blockIdx.x / RL;  // ray block of the chunk
  const int rib = RL == 1 ? lane : (blockIdx.x % RL) * (WAVE / RL) + lane / RL;  // ray in the block
  const bool wr = RL == 1 || lane % RL == 0;  // the lane that writes
  const int blk = blk0 + lb;
  const int ir = blk * WAVE + rib;
  if (ir >= B.nray) return;
  double *base = L.los + (size_t)lb * L.cap * L.nfield * WAVE + rib;

  const double *g = B.ray_geom + (size_t)7 * ir;
  const int iprof = B.ray_prof[ir];
  if (iprof < 0 || iprof >= B.nprof || B.atm[iprof].np < 2 || B.atm[iprof].np > NP) {
    RayInfo E{};
    E.status = JUR_ERR_ARG;
    if (wr) info[ir] = E;
    return;
  }
  const atm_t *atm = &B.atm[iprof];
  const double obsz = g[1], obslon = g[2], obslat = g[3];
  const double vpz = g[4], vplon = g[5], vplat = g[6];

  const double h = 0.02, zrefrac = 60;
  double ex0[3], ex1[3], n, ngr[3], norm, x[3], xh[3], xobs[3], xvp[3];
  double z = 1e99, zmax, zmin;
  int np = 0;

  RayInfo R;
  R.np = 0;
  R.status = JUR_OK;
  R.sft = -999;
  R.tpz = vpz;
  R.tplon = vplon;
  R.tplat = vplat;
  R.rcos = 0;
  R.pad = 0;

  // altitude range (gsl_stats_minmax semantics, src/jurassic.c:4223) and
  // monotonicity of the altitude grid
  // (eight levels per round: the loads of a round wait for memory together)
  zmin = zmax = atm->z[0];
  int zasc = 1, zdesc = 1;
  const int anp = atm->np;
  double vl = zmin;
  bool nan = isnan(zmin);
  for (int i0 = 1; i0 < anp && !nan; i0 += 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = atm->z[i0 + k < anp ? i0 + k : anp - 1];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (i0 + k >= anp || nan) continue;
      zmin = v[k] < zmin ? v[k] : zmin;
      zmax = v[k] > zmax ? v[k] : zmax;
      if (!(v[k] > vl)) zasc = 0;
      if (!(v[k] < vl)) zdesc = 0;
      vl = v[k];
      nan = isnan(vl);
    }
  }
  if (nan) {
    zmin = zmax = vl;
    zasc = zdesc = 0;
  }
  const int zdir = zasc ? 1 : (zdesc ? -1 : 0);
  if (M.nsf > 0) {
    zmin = (atm->sfz > zmin) ? atm->sfz : zmin;
    if (atm->sfp > 0) {
      const int ip = locate_irr(atm->p, atm->np, atm->sfp);
      const double zip = lin(log(atm->p[ip]), atm->z[ip], log(atm->p[ip + 1]), atm->z[ip + 1],
                             log(atm->sfp));
      zmin = (zip > zmin) ? zip : zmin;
    }
  }

  if (obsz < zmin) {
    R.status = JUR_ERR_OBSERVER;
    if (wr) info[ir] = R;
    return;
  }
  if (vpz > zmax) {
    if (wr) info[ir] = R;
    return;
  }

  geo2cart(obsz, obslon, obslat, xobs);
  geo2cart(vpz, vplon, vplat, xvp);
  for (int i = 0; i < 3; i++) ex0[i] = xvp[i] - xobs[i];
  norm = sqrt(ex0[0] * ex0[0] + ex0[1] * ex0[1] + ex0[2] * ex0[2]);
  for (int i = 0; i < 3; i++) ex0[i] /= norm;
  for (int i = 0; i < 3; i++) x[i] = xobs[i];

  // entry point of an observer above the atmosphere (bisection to 1 m)
  if (obsz > zmax) {
    double dmax = norm, dmin = 0;
    while (fabs(dmin - dmax) > 0.001) {
      const double d = (dmax + dmin) / 2;
      for (int i = 0; i < 3; i++) x[i] = xobs[i] + d * ex0[i];
      z = cart2z(x);
      if (z <= zmax && z > zmax - 0.001) break;
      if (z < zmax - 0.0005) dmax = d; else dmin = d;
    }
  }

  // Cartesian positions of the points whose longitude and latitude are
  // needed after the march: the first and the last point, and the two
  // neighbours of the first minimum of z (tangent_point); cart2geo of the
  // same x gives the values the reference stores per point.  (A NaN altitude
  // never leaves the range, so its ray ends at the capacity below and has no
  // tangent point.)
  double zprev = 0, xprev[3] = {0, 0, 0}, xb[3] = {0, 0, 0}, xa[3] = {0, 0, 0};
  double zlow = 0, ds_imin = 0, ds_imin1 = 0;
  int imin = 0;
  bool after_pending = false;
  double ds1 = 0, ds2 = 0;  // raw step lengths of the last two points written
  // the level pairs of the point and of its midpoint probes: a point mostly
  // enters the pair that the probes before it were in
  LevelCache lp, lc;
  LevelAhead ahead;
  const double xfirst[3] = {x[0], x[1], x[2]};
  // the lane's probe (RL = 4): the displacements by h along the axes before
  // its own are made and undone as in the serial order below, x + hp - hm
  const int sub = RL == 1 ? 0 : lane % RL;
  const double hp[3] = {sub >= 1 ? h : 0.0, sub >= 2 ? h : 0.0, sub >= 3 ? h : 0.0};
  const double hm[3] = {sub >= 2 ? h : 0.0, sub >= 3 ? h : 0.0, 0.0};
  double *w = base;
  const size_t wstep = (size_t)L.nfield * WAVE;
  double ds;
  for (;;) {
    ds = M.rayds;
    const double radius = sqrt_mid(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
    if (M.raydz > 0) {
      const double rn = div_mid(1, radius);
      for (int i = 0; i < 3; i++) xh[i] = x[i] * rn;
      const double cosa = fabs(ex0[0] * xh[0] + ex0[1] * xh[1] + ex0[2] * xh[2]);
      if (cosa != 0) ds = (M.rayds < M.raydz / cosa) ? M.rayds : M.raydz / cosa;
    }

    z = radius - JUR_RE;  // the z output of cart2geo

    if (z < zmin || z > zmax || np >= L.cap) break;
    // the trapezoid segment length of the point (src/jurassic.c:4410-4411)
    // from its raw step length ds and the previous point's: 0.5 (ds_prev +
    // ds), the first point 0.5 ds (the clip of the last step changes the last
    // two points, which k_ray_finish rewrites)
    const double dtr = np == 0 ? ds * 0.5 : 0.5 * (ds1 + ds);
    if (wr) {
      w[F_Z * WAVE] = z;
      w[F_DS * WAVE] = dtr;
      if (L.f_xe >= 0)
        for (int i = 0; i < 3; i++) {
          w[(size_t)(L.f_xe + i) * WAVE] = x[i];
          w[(size_t)(L.f_xe + 3 + i) * WAVE] = ex0[i];
        }
    }
    w += wstep;
    // MinTrack::add, with the raw step lengths at the minimum and after it
    if (np == 0 || z < zlow) {
      zlow = z;
      imin = np;
      ds_imin = ds;
      for (int i = 0; i < 3; i++) xb[i] = xprev[i];
      after_pending = true;
    } else if (after_pending) {
      for (int i = 0; i < 3; i++) xa[i] = x[i];
      ds_imin1 = ds;
      after_pending = false;
    }
    ds2 = ds1;
    ds1 = ds;
    for (int i = 0; i < 3; i++) xprev[i] = x[i];
    zprev = z;
    np++;

    if (M.refrac && z <= zrefrac) {
      // the refractivity at the point, and at the midpoint and the three
      // probes displaced by h along each axis, in the reference's order (each
      // displacement is undone by subtracting h before the next axis moves);
      // with RL = 4 each lane has its own probe.  The level pairs come first,
      // so that the evaluations overlap.
      constexpr int NQ = RL == 4 ? 1 : 4;
      double zq[NQ], rq[NQ];
      for (int i = 0; i < 3; i++) xh[i] = x[i] + 0.5 * ds * ex0[i];
      if constexpr (RL == 4) {
        for (int i = 0; i < 3; i++) xh[i] = xh[i] + hp[i] - hm[i];
        zq[0] = cart2z(xh);
      } else {
        zq[0] = cart2z(xh);
        for (int i = 0; i < 3; i++) {
          xh[i] += h;
          zq[i + 1] = cart2z(xh);
          xh[i] -= h;
        }
      }
      bool all = true;  // the probes are in their cached pair
      for (int k = 0; k < NQ; k++) all &= lc.holds(zq[k]);
      if (!lp.holds(z)) {
        if (lc.holds(z)) lp = lc;
        else lp.enter(atm, anp, zdir, z, ahead);
      }
      if (RL == 4 && !all) lc.enter(atm, anp, zdir, zq[0], ahead);
      if (RL == 4 || all) {
        for (int k = 0; k < NQ; k++) rq[k] = div_mid(7.753e-05 * lc.p(zq[k]), lc.t(zq[k]));
      } else {
        // probe by probe (not unrolled)
#pragma unroll 1
        for (int k = 0; k < NQ; k++) {
          const double zk = k == 0 ? zq[0] : (k == 1 ? zq[1 % NQ] : (k == 2 ? zq[2 % NQ] : zq[3 % NQ]));
          if (!lc.holds(zk)) lc.enter(atm, anp, zdir, zk, ahead);
          const double v = div_mid(7.753e-05 * lc.p(zk), lc.t(zk));
          rq[0] = k == 0 ? v : rq[0];
          rq[1 % NQ] = k == 1 ? v : rq[1 % NQ];
          rq[2 % NQ] = k == 2 ? v : rq[2 % NQ];
          rq[3 % NQ] = k == 3 ? v : rq[3 % NQ];
        }
      }
      n = 1 + div_mid(7.753e-05 * lp.p(z), lp.t(z));
      for (int i = 0; i < 3; i++) ex1[i] = ex0[i] * n;
      if constexpr (RL == 4) {
        n = quad_lane<0>(rq[0]);
        ngr[0] = (quad_lane<1>(rq[0]) - n) * (1 / h);
        ngr[1] = (quad_lane<2>(rq[0]) - n) * (1 / h);
        ngr[2] = (quad_lane<3>(rq[0]) - n) * (1 / h);
      } else {
        n = rq[0];
        for (int i = 0; i < 3; i++) ngr[i] = (rq[(i + 1) % NQ] - n) * (1 / h);
      }
    } else {
      for (int i = 0; i < 3; i++) {
        ex1[i] = ex0[i];
        ngr[i] = 0;
      }
    }

    for (int i = 0; i < 3; i++) ex1[i] += ds * ngr[i];
    const double rn1 = div_mid(1, sqrt_mid(ex1[0] * ex1[0] + ex1[1] * ex1[1] + ex1[2] * ex1[2]));
    for (int i = 0; i < 3; i++) ex1[i] *= rn1;
    for (int i = 0; i < 3; i++) x[i] += 0.5 * ds * (ex0[i] + ex1[i]);
    for (int i = 0; i < 3; i++) ex0[i] = ex1[i];
  }
  if (!wr) return;
  if (!(z < zmin || z > zmax)) {
    // capacity exceeded: the reference limit NLOS -> error, a smaller
    // working capacity -> the host retries with NLOS
    R.status = (L.cap >= NLOS) ? JUR_ERR_LOS : 100;
    info[ir] = R;
    return;
  }
  // The last step left the altitude range: k_ray_finish clips it to the range
  // and writes the last point (its cart2geo/geo2cart would hold registers for
  // the whole march here).  With no point written the entry search ended
  // outside the range, so there is no previous point to clip to (the reference
  // would read los->z[-1]): the ray has no LOS points.
  R.np = np;
  RayTail *tl = tail + ir;
  if (np > 0) {
    for (int i = 0; i < 3; i++) {
      tl->xprev[i] = xprev[i];
      tl->xcut[i] = x[i];
      tl->ecut[i] = ex0[i];
      tl->xfirst[i] = xfirst[i];
      tl->mt.xbefore[i] = xb[i];
      tl->mt.xafter[i] = xa[i];
    }
    tl->zprev = zprev;
    tl->zcut = z;
    tl->dscut = ds;
    tl->zmin = zmin;
    tl->zmax = zmax;
    tl->ds1 = ds1;
    tl->ds2 = ds2;
    tl->ds_imin = ds_imin;
    tl->ds_imin1 = ds_imin1;
    tl->mt.zlow = zlow;
    tl->mt.imin = imin;
    tl->mt.after_pending = after_pending;
    tl->mt.nan_seen = false;
    tl->zdir = zdir;
  }
  info[ir] = R;
}

// The end of a ray's march (k_raytrace): the step that left the altitude
// range is clipped to it and becomes the last LOS point, as raytrace does
// (src/jurassic.c:4290-4306), then the tangent point, the solar-incidence
// factor and the trapezoid step lengths of the last two points.
__global__ __launch_bounds__(WAVE) void k_ray_finish(ModelView M, BatchView B, LosView L, RayInfo *info,
                                                     const RayTail *tail, int blk0) {
  JUR_FP_EXACT
  const int lane = threadIdx.x;
  const int ir = (blk0 + blockIdx.x) * WAVE + lane;
  if (ir >= B.nray) return;
  RayInfo R = info[ir];
  if (R.status != JUR_OK || R.np == 0) return;
  double *base = L.los + (size_t)blockIdx.x * L.cap * L.nfield * WAVE + lane;
  const atm_t *atm = &B.atm[B.ray_prof[ir]];
  const RayTail T = tail[ir];
  MinTrack mt = T.mt;
  int np = R.np;

  // the last step, clipped to the altitude range
  const int stop = (T.zcut < T.zmin ? 2 : 1);
  const double frac = ((T.zcut < T.zmin ? T.zmin : T.zmax) - T.zprev) / (T.zcut - T.zprev);
  double zd, lon, lat, xh[3], x[3];
  cart2geo(T.xprev, &zd, &lon, &lat);
  geo2cart(T.zprev, lon, lat, xh);
  for (int i = 0; i < 3; i++) x[i] = xh[i] + frac * (T.xcut[i] - xh[i]);
  const double z = cart2z(x);
  // los->ds[np-1] = ds * frac: the raw step length of the last point written
  const int npm = np;
  const double clip = T.dscut * frac;

  if (np >= L.cap) {
    R.status = (L.cap >= NLOS) ? JUR_ERR_LOS : 100;
    info[ir] = R;
    return;
  }
  // the temperature at the clipped point (intpol_atm), for the surface
  LevelCache lc;
  LevelAhead ahead;
  lc.enter(atm, atm->np, T.zdir, z, ahead);
  double t = lc.t(z);
  // trapezoid segment lengths (src/jurassic.c:4410-4411) of the last point
  // written, from its clipped raw length, and of this one (raw length 0);
  // the march wrote those of the others
  LOSW(F_DS, npm - 1) = npm == 1 ? clip * 0.5 : 0.5 * (T.ds2 + clip);
  LOSW(F_Z, np) = z;
  LOSW(F_DS, np) = 0.5 * (clip + 0.0);
  if (L.f_xe >= 0)
    for (int i = 0; i < 3; i++) {
      LOSW(L.f_xe + i, np) = x[i];
      LOSW(L.f_xe + 3 + i, np) = 0.0;
    }
  mt.add(np, z, x, T.xprev);
  np++;
  if (M.nsf > 0 && atm->sft > 0) t = atm->sft;
  R.sft = (stop == 2 ? t : -999);
  R.np = np;

  // tangent_point at the first minimum imin found during the march
  double zl, lonl, latl;
  cart2geo(x, &zl, &lonl, &latl);
  if (mt.imin <= 0 || mt.imin >= np - 1) {
    R.tpz = LOSW(F_Z, np - 1);
    R.tplon = lonl;
    R.tplat = latl;
  } else {
    const double yy0 = LOSW(F_Z, mt.imin - 1);
    const double yy1 = LOSW(F_Z, mt.imin);
    const double yy2 = LOSW(F_Z, mt.imin + 1);
    // the raw step lengths at imin and imin + 1 (tangent_point runs
    // before the trapezoid rule in raytrace)
    auto rawds = [&](int i) {
      return i == npm ? 0.0 : (i == npm - 1 ? clip : (i == mt.imin ? T.ds_imin : T.ds_imin1));
    };
    const double d1 = rawds(mt.imin), d2 = rawds(mt.imin + 1);
    const double x1 = sqrt(d1 * d1 - (yy1 - yy0) * (yy1 - yy0));
    const double x2 = x1 + sqrt(d2 * d2 - (yy2 - yy1) * (yy2 - yy1));
    const double a = 1 / (x1 - x2) * (-(yy0 - yy1) / x1 + (yy0 - yy2) / x2);
    const double b = -(yy0 - yy1) / x1 - a * x1;
    const double c = yy0;
    const double xt = -b / (2 * a);
    double v[3], v0[3], v2[3], dummy;
    R.tpz = a * xt * xt + b * xt + c;
    double lon0, lat0, lon2, lat2;
    cart2geo(mt.xbefore, &dummy, &lon0, &lat0);
    cart2geo(mt.xafter, &dummy, &lon2, &lat2);
    geo2cart(yy0, lon0, lat0, v0);
    geo2cart(yy2, lon2, lat2, v2);
    for (int i = 0; i < 3; i++) v[i] = lin(0.0, v0[i], x2, v2[i], xt);
    cart2geo(v, &dummy, &R.tplon, &R.tplat);
  }

  // solar incidence (formod_pencil, src/jurassic.c:3297-3326)
  if (M.sftype >= 3 && R.sft > 0) {
    const double sza2 = (M.sfsza < 0) ? sza(B.ray_geom[(size_t)7 * ir], lonl, latl) : M.sfsza;
    if (sza2 < 89.999) {
      double x0[3], x1[3];
      geo2cart(LOSW(F_Z, np - 1), lonl, latl, x0);
      double lonf, latf, zf;
      cart2geo(T.xfirst, &zf, &lonf, &latf);
      geo2cart(LOSW(F_Z, 0), lonf, latf, x1);
      for (int i = 0; i < 3; i++) x1[i] -= x0[i];
      const double cosa = (x0[0] * x1[0] + x0[1] * x1[1] + x0[2] * x1[2]) /
                          sqrt(x0[0] * x0[0] + x0[1] * x0[1] + x0[2] * x0[2]) /
                          sqrt(x1[0] * x1[0] + x1[1] * x1[1] + x1[2] * x1[2]);
      R.rcos = cosa / cos(sza2 * (JUR_PI / 180.0));
      R.pad = 1.0;
    }
  }

  info[ir] = R;
}

// The atmosphere at the LOS points (intpol_atm, src/jurassic.c:3685-3706, and
// the column densities, :4410-4419) from their altitudes and trapezoid step
// lengths.  One wavefront per (block of 64 rays, RP_STEPS points): the level
// pair and the quotients of LOGY (p) and LIN (t, q, k) are kept in LDS while a
// lane's points stay between the same two levels.  Writes p, t, the mixing
// ratio of H2O (no kernel reads the others'), extinctions, cloud factor and
// column densities and, for the FP32 forward pass, what its radiance kernel
// reads rounded to float.
//
// In the march these took two divisions, an interpolation per emitter and
// some twenty stores of every step's chain: 1.90 ms for 10 nadir rays (805
// steps, one emitter) against 0.95 + 0.02 here, 4.27 against 1.93 + 0.04 for
// 77 x 5 limb rays of three emitters; for 4096 x 32 of them 7.1 against 3.7 +
// 4.1 ms (bound by the stores).  (The march has since become faster: 0.66, 1.32
// and 2.6 ms; the points of the large batch take 3.7.)
constexpr int RP_STEPS = 16;

__global__ __launch_bounds__(WAVE) void k_ray_points(ModelView M, BatchView B, LosView L, const RayInfo *info,
                                                     const RayTail *tail, int blk0, int nblk, int nchunk) {
  JUR_FP_EXACT
  int bl, chk;
  if (!xcd_block_map(blockIdx.x, nchunk, nblk, bl, chk)) return;
  const int lane = threadIdx.x;
  const int ir = (blk0 + bl) * WAVE + lane;
  if (ir >= B.nray) return;
  const RayInfo R = info[ir];
  if (R.status != JUR_OK) return;
  const int i0 = chk * RP_STEPS;
  const int i1 = i0 + RP_STEPS < R.np ? i0 + RP_STEPS : R.np;
  if (i0 >= i1) return;
  double *base = L.los + (size_t)bl * L.cap * L.nfield * WAVE + lane;
  float *basef = L.losf ? L.losf + (size_t)bl * L.cap * L.nfield * WAVE + lane : nullptr;
  const atm_t *atm = &B.atm[B.ray_prof[ir]];
  const int anp = atm->np, zdir = tail[ir].zdir;
  // q0[ng], q slopes[ng], k0[nw], k slopes[nw]; field-major, lane fastest
  extern __shared__ double lvl[];
#define LV(f) lvl[(f) * WAVE + lane]
  LevelCache lc;
  LevelAhead ahead;
  // the tables' cell of a point (LosView::cell): the pressure bracket and,
  // on its two pressures, the temperature brackets and weights, with the
  // arithmetic of the FP32 lookups (float, reciprocal spacings)
  const TabView &T = M.tab;
  float4 *cell = L.cell ? L.cell + ((size_t)bl * L.cap * WAVE + lane) * L.ncell : nullptr;
  const double *pg = T.p + (size_t)T.ref_tix * T.TP;
  const double *tgb = T.t + (size_t)T.ref_tix * T.TP * T.TT;
  const int *ntp = T.nt + (size_t)T.ref_tix * T.TP;
  const int npt = cell ? T.np[T.ref_tix] : 0, pdir = cell ? T.pdir[T.ref_tix] : 0;
  int ipr = -1;
  double pa = 0, pb = 0;
  float rwp = 0, g00 = 0, gi0 = 0, g10 = 0, gi1 = 0;
  int nt0 = 0, nt1 = 0;
  auto put_cell = [&](double p, double t, int ip) {
    const bool keep = ipr >= 0 && (pdir > 0 ? (ipr == 0 || !(pa > p)) && (ipr == npt - 2 || pb > p)
                                            : (ipr == 0 || !(pa <= p)) && (ipr == npt - 2 || pb <= p));
    if (!keep) {
      ipr = ipr >= 0 ? irr_walk(pg, npt, p, ipr, pdir) : locate_irr(pg, npt, p);
      pa = pg[ipr];
      pb = pg[ipr + 1];
      rwp = frcp((float)(pb - pa));
      nt0 = ntp[ipr];
      nt1 = ntp[ipr + 1];
      const double *tg = tgb + (size_t)ipr * T.TT;
      g00 = (float)tg[0];
      gi0 = frcp((float)(tg[1] - tg[0]));
      g10 = (float)tg[T.TT];
      gi1 = frcp((float)(tg[T.TT + 1] - tg[T.TT]));
    }
    const float tq = (float)t;
    int j0 = (int)((tq - g00) * gi0);
    j0 = j0 < 0 ? 0 : (j0 > nt0 - 2 ? nt0 - 2 : j0);
    int j1 = (int)((tq - g10) * gi1);
    j1 = j1 < 0 ? 0 : (j1 > nt1 - 2 ? nt1 - 2 : j1);
    const int c00 = ipr * T.TT + j0, c10 = (ipr + 1) * T.TT + j1;
    const double ta0 = tgb[c00], ta1 = tgb[c10];
    const float dt0 = frcp((float)(tgb[c00 + 1] - ta0)), dt1 = frcp((float)(tgb[c10 + 1] - ta1));
    float4 *o = cell + (size_t)ip * WAVE * L.ncell;
    o[0] = make_float4(__int_as_float(c00 | c10 << 16), (tq - (float)ta0) * dt0, (tq - (float)ta1) * dt1,
                       (float)(p - pa) * rwp);
    if (L.ncell > 1) o[1] = make_float4(dt0, dt1, rwp, 0.f);
  };
  double z = LOSW(F_Z, i0), ds = LOSW(F_DS, i0);
  for (int ip = i0; ip < i1; ip++) {
    const int ipn = ip + 1 < i1 ? ip + 1 : ip;
    const double zn = LOSW(F_Z, ipn), dsn = LOSW(F_DS, ipn);
    if (!lc.holds(z)) {
      const int old = lc.ip;
      lc.enter(atm, anp, zdir, z, ahead);
      const int l = lc.ip;
      if (l != old) {
        const double dx = lc.dz;
        for (int ig = 0; ig < M.ng; ig++) {
          const double q0 = atm->q[ig][l];
          LV(ig) = q0;
          LV(M.ng + ig) = (atm->q[ig][l + 1] - q0) / dx;
        }
        for (int iw = 0; iw < M.nw; iw++) {
          const double k0 = atm->k[iw][l];
          LV(2 * M.ng + iw) = k0;
          LV(2 * M.ng + M.nw + iw) = (atm->k[iw][l + 1] - k0) / dx;
        }
      }
    }
    const double dzl = z - lc.z0;
    const double p = lc.p(z), t = lc.t(z);
    // the FP32 forward pass reads p, t and u in FP64 in its lookups, and the
    // rounded copies in its radiance kernel
    auto put = [&](int f, double v) {
      if (basef) LOS_AT(basef, L, f, ip) = (float)v;
      else LOSW(f, ip) = v;
    };
    if (cell) {
      put_cell(p, t, ip);
    }
    if (!cell || !basef) {
      LOSW(F_P, ip) = p;
      LOSW(F_T, ip) = t;
    }
    if (basef) {
      put(F_P, p);
      put(F_T, t);
      put(F_DS, ds);
    }
    const double ucol = 10 * p / (JUR_KB * t) * ds;  // column density per unit vmr
    for (int ig = 0; ig < M.ng; ig++) {
      const double q = LV(ig) + LV(M.ng + ig) * dzl;
      if (ig == M.ig_h2o) put(F_Q0 + ig, q);
      LOSW(L.f_u + ig, ip) = q * ucol;
      if (basef && (ig == M.ig_co2 || ig == M.ig_h2o)) put(L.f_u + ig, q * ucol);
    }
    for (int iw = 0; iw < M.nw; iw++) put(L.f_k + iw, LV(2 * M.ng + iw) + LV(2 * M.ng + M.nw + iw) * dzl);
    if (L.f_cl >= 0) {
      const double aux = (M.ncl > 0 && atm->cldz > 0)
                             ? exp(-0.5 * (((z - atm->clz) / atm->cldz) * ((z - atm->clz) / atm->cldz)))
                             : 0.0;
      put(L.f_cl, aux);
    }
    z = zn;
    ds = dsn;
  }
#undef LV
}

// hydrostatic (src/jurassic.c:3520-3582), one lane per atmosphere.
__global__ __launch_bounds__(WAVE) void k_hydrostatic(atm_t *atm, int nprof, double hydz,
                                                      int ig_h2o) {
  JUR_FP_EXACT
  const int ia = blockIdx.x * WAVE + threadIdx.x;
  if (ia >= nprof) return;
  atm_t *a = &atm[ia];
  const double mmair = 28.96456e-3, mmh2o = 18.0153e-3, G0 = 9.80665, RI = 8.3144598;
  const int ipts = 20;
  double dzmin = 1e99, e = 0;
  int ipref = 0;
  for (int ip = 0; ip < a->np; ip++)
    if (fabs(a->z[ip] - hydz) < dzmin) {
      dzmin = fabs(a->z[ip] - hydz);
      ipref = ip;
    }
  for (int ip = ipref + 1; ip < a->np; ip++) {
    double mean = 0;
    for (int i = 0; i < ipts; i++) {
      if (ig_h2o >= 0) e = lin(0.0, a->q[ig_h2o][ip - 1], ipts - 1.0, a->q[ig_h2o][ip], (double)i);
      mean += (e * mmh2o + (1 - e) * mmair) * G0 / RI /
              lin(0.0, a->t[ip - 1], ipts - 1.0, a->t[ip], (double)i) / ipts;
    }
    a->p[ip] = exp(log(a->p[ip - 1]) - mean * 1000 * (a->z[ip] - a->z[ip - 1]));
  }
  for (int ip = ipref - 1; ip >= 0; ip--) {
    double mean = 0;
    for (int i = 0; i < ipts; i++) {
      if (ig_h2o >= 0) e = lin(0.0, a->q[ig_h2o][ip + 1], ipts - 1.0, a->q[ig_h2o][ip], (double)i);
      mean += (e * mmh2o + (1 - e) * mmair) * G0 / RI /
              lin(0.0, a->t[ip + 1], ipts - 1.0, a->t[ip], (double)i) / ipts;
    }
    a->p[ip] = exp(log(a->p[ip + 1]) - mean * 1000 * (a->z[ip] - a->z[ip + 1]));
  }
}

size_t ray_tail_bytes() { return sizeof(RayTail); }

// tail: ray_tail_bytes() per ray of the batch
void launch_raytrace(const ModelView &M, const BatchView &B, const LosView &L, RayInfo *info, void *tail,
                     int blk0, int nblk, hipStream_t s) {
  // small batches: four lanes per ray, a quarter block per wavefront
  if (nblk <= 512)
    hipLaunchKernelGGL(k_raytrace<4>, dim3(4 * nblk), dim3(WAVE), 0, s, M, B, L, info, (RayTail *)tail, blk0);
  else
    hipLaunchKernelGGL(k_raytrace<1>, dim3(nblk), dim3(WAVE), 0, s, M, B, L, info, (RayTail *)tail, blk0);
  hipLaunchKernelGGL(k_ray_finish, dim3(nblk), dim3(WAVE), 0, s, M, B, L, info, (const RayTail *)tail, blk0);
}

// maxnp: the longest LOS of the blocks
void launch_ray_points(const ModelView &M, const BatchView &B, const LosView &L, const RayInfo *info,
                       const void *tail, int blk0, int nblk, int maxnp, hipStream_t s) {
  if (maxnp <= 0) return;
  const int nchunk = (maxnp + RP_STEPS - 1) / RP_STEPS;
  const size_t lds = (size_t)(2 * M.ng + 2 * M.nw) * WAVE * sizeof(double);
  hipLaunchKernelGGL(k_ray_points, dim3(padded_blocks(nblk) * nchunk), dim3(WAVE), lds, s, M, B, L, info,
                     (const RayTail *)tail, blk0, nblk, nchunk);
}

void launch_hydrostatic(atm_t *atm, int nprof, double hydz, int ig_h2o, hipStream_t s) {
  hipLaunchKernelGGL(k_hydrostatic, dim3((nprof + WAVE - 1) / WAVE), dim3(WAVE), 0, s, atm, nprof,
                     hydz, ig_h2o);
}

}  // namespace jur
