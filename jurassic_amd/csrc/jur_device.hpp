// Device helpers of the FP64 path.  Every function keeps the expression
// tree and the float/double promotions of the reference function it names,
// with multiply-add contraction disabled, so that the FP64 kernels agree with
// the reference to rounding.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "jur_internal.hpp"

namespace jur {

#define JUR_FP_EXACT _Pragma("clang fp contract(off)")

// LIN (src/jurassic.h:164-165) on doubles.
__device__ __forceinline__ double lin(double x0, double y0, double x1, double y1, double x) {
  JUR_FP_EXACT
  return y0 + (y1 - y0) / (x1 - x0) * (x - x0);
}

// LIN with float table entries: the slope is formed in float arithmetic, then
// multiplied by the double (x - x0), as C promotion does in the reference.
__device__ __forceinline__ double lin_f(float x0, float y0, float x1, float y1, double x) {
  JUR_FP_EXACT
  const float s = (y1 - y0) / (x1 - x0);
  return (double)y0 + (double)s * (x - (double)x0);
}

// LOGY (src/jurassic.h:174-177).
__device__ __forceinline__ double logy(double x0, double y0, double x1, double y1, double x) {
  JUR_FP_EXACT
  return (y1 / y0 > 0) ? (y0 * exp(log(y1 / y0) / (x1 - x0) * (x - x0))) : lin(x0, y0, x1, y1, x);
}

// LOGX (src/jurassic.h:168-171).
__device__ __forceinline__ double logx(double x0, double y0, double x1, double y1, double x) {
  JUR_FP_EXACT
  return (x / x0 > 0 && x1 / x0 > 0) ? (y0 + (y1 - y0) * log(x / x0) / log(x1 / x0))
                                      : lin(x0, y0, x1, y1, x);
}

// geo2cart (src/jurassic.c:3500-3516).
__device__ __forceinline__ void geo2cart(double z, double lon, double lat, double *x) {
  JUR_FP_EXACT
  const double radius = z + JUR_RE;
  const double latrad = lat / 180. * JUR_PI;
  const double lonrad = lon / 180. * JUR_PI;
  const double coslat = cos(latrad);
  x[0] = radius * coslat * cos(lonrad);
  x[1] = radius * coslat * sin(lonrad);
  x[2] = radius * sin(latrad);
}

// cart2geo (src/jurassic.c:108-119).
__device__ __forceinline__ void cart2geo(const double *x, double *z, double *lon, double *lat) {
  JUR_FP_EXACT
  const double radius = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  *lat = asin(x[2] / radius) * (180.0 / JUR_PI);
  *lon = atan2(x[1], x[0]) * (180.0 / JUR_PI);
  *z = radius - JUR_RE;
}

// locate_irr (src/jurassic.c:4103-4129): bisection, either grid order.
template <typename T>
__host__ __device__ __forceinline__ int locate_irr(const T *xx, int n, double x) {
  int ilo = 0, ihi = n - 1, i = (ihi + ilo) >> 1;
  if ((double)xx[i] < (double)xx[i + 1])
    while (ihi > ilo + 1) {
      i = (ihi + ilo) >> 1;
      if ((double)xx[i] > x) ihi = i; else ilo = i;
    }
  else
    while (ihi > ilo + 1) {
      i = (ihi + ilo) >> 1;
      if ((double)xx[i] <= x) ihi = i; else ilo = i;
    }
  return ilo;
}

// locate_irr by a local walk from a previous index g, for strictly
// monotone grids (dir = +1 ascending, -1 descending).  The result satisfies
// the bisection's end condition, which for a strictly monotone grid has a
// single solution, so it equals locate_irr's.
template <typename T>
__device__ __forceinline__ int irr_walk(const T *xx, int n, double x, int g, int dir) {
  g = g < 0 ? 0 : (g > n - 2 ? n - 2 : g);
  if (dir > 0) {
    while (g > 0 && (double)xx[g] > x) g--;
    while (g < n - 2 && !((double)xx[g + 1] > x)) g++;
  } else {
    while (g > 0 && (double)xx[g] <= x) g--;
    while (g < n - 2 && !((double)xx[g + 1] <= x)) g++;
  }
  return g;
}

// locate_reg (src/jurassic.c:4133-4148).
__device__ __forceinline__ int locate_reg(const double *xx, int n, double x) {
  JUR_FP_EXACT
  const int i = (int)((x - xx[0]) / (xx[1] - xx[0]));
  return i < 0 ? 0 : (i > n - 2 ? n - 2 : i);
}

// ------------------------------------------------------------------
// Column search on a table column of n >= 2 records.
// C selects the searched component: 0 = u (rec.x / rec.z), 1 = eps (rec.y / rec.w).
// Returns i in [0, n-2] with (i == 0 or v_i <= x) and (i == n-2 or v_{i+1} > x),
// which for a non-decreasing column is the index the reference bisection
// locate_tbl (src/jurassic.c:4152-4170) returns.  The walk starts at the
// previous segment's index `g`, which is usually already right.
// ------------------------------------------------------------------
template <int C>
__device__ __forceinline__ float lo_of(const float4 &r) { return C == 0 ? r.x : r.y; }
template <int C>
__device__ __forceinline__ float hi_of(const float4 &r) { return C == 0 ? r.z : r.w; }

template <int C>
__device__ __forceinline__ int col_walk(Col col, int n, double x, int g, float4 &r) {
  g = g < 0 ? 0 : (g > n - 2 ? n - 2 : g);
  r = col[g];
  if (g > 0 && (double)lo_of<C>(r) > x) {
    // answer < g: gallop left to a lower bound, then bisect
    int hi = g, step = 1, lo;
    float4 rl;
    for (;;) {
      int j = hi - step;
      if (j <= 0) { lo = 0; rl = col[0]; break; }
      float4 rj = col[j];
      if ((double)lo_of<C>(rj) <= x) { lo = j; rl = rj; break; }
      hi = j;
      step <<= 1;
    }
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const float4 rm = col[mid];
      if ((double)lo_of<C>(rm) > x) hi = mid; else { lo = mid; rl = rm; }
    }
    r = rl;
    return lo;
  }
  if (g < n - 2 && (double)hi_of<C>(r) <= x) {
    // answer > g: gallop right to an upper bound, then bisect
    int lo = g, step = 1, hi;
    float4 rh;
    for (;;) {
      int j = lo + step;
      if (j >= n - 2) { hi = n - 2; rh = col[n - 2]; break; }
      float4 rj = col[j];
      if ((double)hi_of<C>(rj) > x) { hi = j; rh = rj; break; }
      lo = j;
      step <<= 1;
    }
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const float4 rm = col[mid];
      if ((double)hi_of<C>(rm) > x) { hi = mid; rh = rm; } else lo = mid;
    }
    r = rh;
    return hi;
  }
  return g;
}

// col_walk with the record at the start index already in hand (rg = col[g],
// g in [0, n-2]): the common case, x still inside that bracket, loads nothing.
template <int C>
__device__ __forceinline__ int col_walk_r(Col col, int n, double x, int g, const float4 &rg,
                                          float4 &r) {
  const bool left = g > 0 && (double)lo_of<C>(rg) > x;
  const bool right = g < n - 2 && (double)hi_of<C>(rg) <= x;
  if (!left && !right) {
    r = rg;
    return g;
  }
  return col_walk<C>(col, n, x, g, r);
}

// intpol_tbl_u (src/jurassic.c:3933-3967) evaluated from the bracket record
// r that the walk returned for x on a monotone column: x below the first
// knot leaves the walk at record 0 = (u_0, eps_0, ...), x above the last knot
// at record n-2 = (..., u_{n-1}, eps_{n-1}).
__device__ __forceinline__ double u_from_rec(const float4 &r, double x) {
  JUR_FP_EXACT
  if (x < (double)r.y) return lin_f(0.f, 0.f, r.y, r.x, x);
  if (x > (double)r.w) {
    const double a = log((double)(1.f - r.w)) / (double)r.z;
    return log(1 - x) / a;
  }
  return lin_f(r.y, r.x, r.w, r.z, x);
}

// intpol_tbl_eps (src/jurassic.c:3895-3929) from a bracket record.
__device__ __forceinline__ double eps_from_rec(const float4 &r, double x) {
  JUR_FP_EXACT
  if (x < (double)r.x) return lin_f(0.f, 0.f, r.x, r.y, x);
  if (x > (double)r.z) {
    const double a = log((double)(1.f - r.w)) / (double)r.z;
    return 1 - exp(a * x);
  }
  return lin_f(r.x, r.y, r.z, r.w, x);
}

// col_walk for a float key (the FP32 path): same end condition, float
// comparisons.
template <int C>
__device__ __forceinline__ int col_walk_f(Col col, int n, float x, int g, float4 &r) {
  g = g < 0 ? 0 : (g > n - 2 ? n - 2 : g);
  r = col[g];
  if (g > 0 && lo_of<C>(r) > x) {
    int hi = g, step = 1, lo;
    float4 rl;
    for (;;) {
      int j = hi - step;
      if (j <= 0) { lo = 0; rl = col[0]; break; }
      float4 rj = col[j];
      if (lo_of<C>(rj) <= x) { lo = j; rl = rj; break; }
      hi = j;
      step <<= 1;
    }
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const float4 rm = col[mid];
      if (lo_of<C>(rm) > x) hi = mid; else { lo = mid; rl = rm; }
    }
    r = rl;
    return lo;
  }
  if (g < n - 2 && hi_of<C>(r) <= x) {
    int lo = g, step = 1, hi;
    float4 rh;
    for (;;) {
      int j = lo + step;
      if (j >= n - 2) { hi = n - 2; rh = col[n - 2]; break; }
      float4 rj = col[j];
      if (hi_of<C>(rj) > x) { hi = j; rh = rj; break; }
      lo = j;
      step <<= 1;
    }
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const float4 rm = col[mid];
      if (hi_of<C>(rm) > x) { hi = mid; rh = rm; } else lo = mid;
    }
    r = rh;
    return hi;
  }
  return g;
}

// Fast float reciprocal and division for the FP32 path (v_rcp_f32, 1 ulp):
// the default HIP float division here is IEEE-correct, which the FP64
// path's float slopes need, but the FP32 path does not.
// base[i] with a 32-bit element index: a wave-uniform base plus a per-lane
// 32-bit byte offset, which the compiler addresses as SGPR base + VGPR offset
// without 64-bit arithmetic per lane.  For arrays far below 4 GB (one
// table, one ray block's LOS or emissivities).
template <typename V>
__device__ __forceinline__ V ld32(const V *base, unsigned i) {
  return *(const V *)((const char *)base + (size_t)(i * (unsigned)sizeof(V)));
}
template <typename V>
__device__ __forceinline__ void st32(V *base, unsigned i, V v) {
  *(V *)((char *)base + (size_t)(i * (unsigned)sizeof(V))) = v;
}

__device__ __forceinline__ float frcp(float b) { return __builtin_amdgcn_rcpf(b); }

// 1/x in FP64 to about an ulp: v_rcp_f64 and two Newton steps (five
// instructions against about fifteen for a correctly rounded division), for
// the FP32 Jacobian's sweeps, which need FP64 range and accuracy but not a
// correctly rounded quotient.  x > 0 and finite.
__device__ __forceinline__ double rcp_d(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// tanh(x) for x >= 0 in float: (e - 1)/(e + 1) with e = exp(2x) from the
// hardware exponential (relative error about 1e-7 / x below x = 1, a few
// ulp above; 1 beyond x = 9, where tanhf rounds to 1 too).
__device__ __forceinline__ float tanh_pos_f(float x) {
  if (x > 9.f) return 1.f;
  const float e = __expf(2.f * x);
  return fdiv(e - 1.f, e + 1.f);
}

// The reference bisection itself (for columns that are not monotone).
template <int C>
__device__ __forceinline__ int col_bisect(Col col, int n, double x, float4 &r) {
  int ilo = 0, ihi = n - 1, i;
  while (ihi > ilo + 1) {
    i = (ihi + ilo) >> 1;
    if ((double)lo_of<C>(col[i]) > x) ihi = i; else ilo = i;
  }
  r = col[ilo];
  return ilo;
}

// ---- FP32-path table interpolation (lookup_f32.hip, adjoint.hip) ----
// intpol_tbl_eps from a bracket record, float interpolation.
__device__ __forceinline__ float eps_from_rec_f(const float4 &r, double x) {
  if (x < (double)r.x) return fdiv(r.y, r.x) * (float)x;
  if (x > (double)r.z) return 1.f - __expf(fdiv(__logf(1.f - r.w), r.z) * (float)x);
  return r.y + fdiv(r.w - r.y, r.z - r.x) * (float)(x - (double)r.x);
}

// One EGA growth step on one table column, FP32 path: from the path
// emissivity ep, u_eq = u(ep) (intpol_tbl_u, src/jurassic.c:3933-3967), then
// eps(u_eq + u_seg) (intpol_tbl_eps, :3895-3929).
//
// Both interpolations run on the same piecewise-linear curve through the
// knots, so inside one bracket the step is ep + u_seg s with the bracket's
// slope s = deps/du, and a step that leaves the bracket at its upper knot
// (u_1, e_1) continues from there with the next slope: the part of u_seg
// beyond the knot is (ep + u_seg s_0 - e_1)/s_0, hence e_1 + that s_1.  No
// column density is formed, so nothing cancels and nothing needs FP64.  The
// steps return the growth: the caller adds it with the rounding error of the
// last sum carried, since many steps are below half an ulp of ep.
//
// The slopes jump by some percent from bracket to bracket, and the partials of
// all points before with them, so for the partials (D) a path that meets a
// knot to within half an ulp of ep must be on the side that its sum is on: the
// position on the curve is then ep + rest, rest being the carried error.
// (K of 768 atmospheres x 8 nadir views x 96 channels against FP64, by ep and
// by ep + rest: CO2 5.7e-5 and 1.6e-6, H2O 1.5e-5 and 8.7e-7, O3 7.6e-5 and
// 1.4e-6; of 1500 x 32 limb rays x 12 channels: CO2 2.0e-3 and 1.7e-3, T
// 4.7e-4 and 4.1e-4.)
// The emissivities, continuous across the knots, do not need it (and the
// kernel without the partials would lose a wavefront per SIMD to its
// registers, 4% of its time).
//
// ega_key: the largest float not above the position; the knots are floats, so
// position >= knot is key >= knot.
template <bool D>
__device__ __forceinline__ float ega_key(float ep, float rest) {
  return D ? __int_as_float(__float_as_int(ep) - (rest < 0.f ? 1 : 0)) : ep;
}

// The position's distance from a knot (its sign is exact).
template <bool D>
__device__ __forceinline__ float ega_dist(float ep, float rest, float knot) {
  return D ? (ep - knot) + rest : ep - knot;
}

// ega_step_fast has the three knots k[0..2] from the previous step's bracket
// g on in hand (a = k[0], k[1]; b = k[2]; g = -1: the bracket between the
// origin and the first knot).  It covers ep in the bracket g or g + 1, the
// grown emissivity in the same or (from g) the next one.  ok is false for
// everything else (longer walks, beyond the last knot: the end marks' eps of
// -1 fails the comparisons; flat or vertical brackets: NaN does) and
// ega_step_slow gives the result.  g returns the inverse bracket.  With D,
// dep = d eps / d ep and deu = d eps / d u_seg of the brackets used.
template <bool D>
__device__ __forceinline__ void ega_step_fast(const float4 &a, const float2 &b, float ep, float rest, float key,
                                              float us, int &g, float &ec, float &dep, float &deu, bool &ok) {
  JUR_FP_EXACT  // the multiply-adds as written: every kernel the same bits
  const float de1 = b.y - a.w;
  const float s0 = fdiv(a.w - a.y, a.z - a.x);
  const float s1 = fdiv(de1, b.x - a.z);
  const float ratio = fdiv(s1, s0);
  const bool up = key >= a.w;
  const float s = up ? s1 : s0;
  const float d = ega_dist<D>(ep, rest, up ? b.y : a.w);
  const float over = __builtin_fmaf(us, s, d);  // beyond the bracket's upper knot
  const bool in = over < 0.f;
  ok = a.y <= key && (in || (!up && over * ratio < de1));
  ec = in ? us * s : __builtin_fmaf(over, ratio, -d);
  if (D) {
    dep = in ? 1.f : ratio;
    deu = in ? s : s1;
  }
  if (up) g++;
}

// Above the last knot (a = the bracket that ends at it, b = an end mark;
// paths that have grown past a column's last emissivity, e.g. a limb path
// climbing into thin layers): eps(u) = 1 - exp(c u), c = log(1 - eps_last) /
// u_last, so eps(u_eq + u_seg) = 1 - (1 - ep) exp(c u_seg).
template <bool D>
__device__ __forceinline__ bool ega_above(const float4 &a, const float2 &b, float ep, float rest) {
  return b.y < 0.f && a.w >= 0.f && ega_dist<D>(ep, rest, a.w) > 0.f;
}
template <bool D>
__device__ __forceinline__ float ega_step_above(float u_last, float e_last, float ep, float us, float &dep,
                                                float &deu) {
  JUR_FP_EXACT
  const float c = fdiv(__logf(1.f - e_last), u_last);
  if (D) {
    const float ex = __expf(c * us);
    deu = ex > 0.f ? -c * (1.f - ep) * ex : 0.f;
    dep = ex;
  }
  return -(1.f - ep) * expm1f(c * us);
}

// FP32 path: eps_from_rec_f with its slope.
__device__ __forceinline__ float eps_rec_f_vs(const float4 &r, double x, float &s) {
  if (x < (double)r.x) {
    s = fdiv(r.y, r.x);
    return s * (float)x;
  }
  if (x > (double)r.z) {
    const float a = fdiv(__logf(1.f - r.w), r.z);
    const float ex = __expf(a * (float)x);
    s = ex > 0.f ? -a * ex : 0.f;
    return 1.f - ex;
  }
  s = fdiv(r.w - r.y, r.z - r.x);
  return r.y + s * (float)(x - (double)r.x);
}

// The general step on one monotone column of n knots; the inverse search
// starts at g and g returns its bracket (-1 below the first knot).
template <bool D>
__device__ __forceinline__ float ega_step_slow(Col col, int n, float ep, float rest, double useg, int &g, float &dep,
                                               float &deu) {
  JUR_FP_EXACT
  float4 r, r2;
  const float key = ega_key<D>(ep, rest);
  const int i = col_walk_f<1>(col, n, key, g, r);
  g = key < r.y ? -1 : i;
  if (ega_dist<D>(ep, rest, r.w) > 0.f) return ega_step_above<D>(r.z, r.w, ep, (float)useg, dep, deu);
  // the bracket of the position (through the origin below the first knot) and
  // the knot after it: inside the bracket and up to that knot the operations
  // of ega_step_fast, so the result does not depend on where the search
  // started
  const bool below = key < r.y;
  const float2 k2 = below ? make_float2(r.z, r.w) : col.k[i + 2];
  const float x0 = below ? 0.f : r.x, y0 = below ? 0.f : r.y, x1 = below ? r.x : r.z, y1 = below ? r.y : r.w;
  const float de1 = k2.y - y1;
  const float s0 = fdiv(y1 - y0, x1 - x0), s1 = fdiv(de1, k2.x - x1);
  const float d = ega_dist<D>(ep, rest, y1);
  const float over = __builtin_fmaf((float)useg, s0, d);
  if (over < 0.f) {
    if (D) {
      dep = 1.f;
      deu = s0;
    }
    return (float)useg * s0;
  }
  const float ratio = fdiv(s1, s0);
  if (over * ratio < de1) {
    if (D) {
      dep = ratio;
      deu = s1;
    }
    return __builtin_fmaf(over, ratio, -d);
  }
  // further up: by the column density
  const float su = fdiv(x1 - x0, y1 - y0);
  const float off = __builtin_fmaf(ega_dist<D>(ep, rest, y0), su, (float)useg);
  const double arg = (double)x0 + (double)off;
  float se;
  col_walk_r<0>(col, n, arg, i, r, r2);
  const float e = eps_rec_f_vs(r2, arg, se);
  if (D) {
    deu = se;
    dep = se * su;
  }
  return -ega_dist<D>(ep, rest, e);
}

// Reference-order lookups for columns that are not monotone (bisection).
__device__ __forceinline__ float col_eps_bis(Col col, int n, double x) {
  const float4 r0 = col[0];
  if (x < (double)r0.x) return fdiv(r0.y, r0.x) * (float)x;
  const float4 rl = col[n - 1];
  if (x > (double)rl.x) return 1.f - __expf(fdiv(__logf(1.f - rl.y), rl.x) * (float)x);
  float4 r;
  col_bisect<0>(col, n, x, r);
  return r.y + fdiv(r.w - r.y, r.z - r.x) * (float)(x - (double)r.x);
}

__device__ __forceinline__ double col_u_bis(Col col, int n, float x) {
  const float4 r0 = col[0];
  if (x < r0.y) return (double)(fdiv(r0.x, r0.y) * x);
  const float4 rl = col[n - 1];
  if (x > rl.y) return (double)(log1pf(-x) * fdiv(rl.x, __logf(1.f - rl.y)));
  float4 r;
  col_bisect<1>(col, n, (double)x, r);
  return (double)r.x + (double)(fdiv(r.z - r.x, r.w - r.y) * (x - r.y));
}

// intpol_tbl_eps on one column (src/jurassic.c:3895-3929).
// For a monotone column the local walk runs first and the two boundary
// branches are read off the bracket record it returns: x below the first
// knot can only leave the walk at record 0, which holds (u_0, eps_0), and x
// above the last knot only at record n-2, which holds (u_{n-1}, eps_{n-1}).
// Branch conditions and arithmetic are those of the reference.
__device__ __forceinline__ double col_eps(Col col, int n, double x, int mono, int &g) {
  JUR_FP_EXACT
  float4 r;
  if (mono) {
    g = col_walk<0>(col, n, x, g, r);
    if (x < (double)r.x) return lin_f(0.f, 0.f, r.x, r.y, x);
    if (x > (double)r.z) {
      const double a = log((double)(1.f - r.w)) / (double)r.z;
      return 1 - exp(a * x);
    }
    return lin_f(r.x, r.y, r.z, r.w, x);
  }
  const float4 r0 = col[0];
  if (x < (double)r0.x) return lin_f(0.f, 0.f, r0.x, r0.y, x);
  const float4 rl = col[n - 1];
  if (x > (double)rl.x) {
    const double a = log((double)(1.f - rl.y)) / (double)rl.x;
    return 1 - exp(a * x);
  }
  g = col_bisect<0>(col, n, x, r);
  return lin_f(r.x, r.y, r.z, r.w, x);
}

// intpol_tbl_u on one column (src/jurassic.c:3933-3967), same scheme.
__device__ __forceinline__ double col_u(Col col, int n, double x, int mono, int &g) {
  JUR_FP_EXACT
  float4 r;
  if (mono) {
    g = col_walk<1>(col, n, x, g, r);
    if (x < (double)r.y) return lin_f(0.f, 0.f, r.y, r.x, x);
    if (x > (double)r.w) {
      const double a = log((double)(1.f - r.w)) / (double)r.z;
      return log(1 - x) / a;
    }
    return lin_f(r.y, r.x, r.w, r.z, x);
  }
  const float4 r0 = col[0];
  if (x < (double)r0.y) return lin_f(0.f, 0.f, r0.y, r0.x, x);
  const float4 rl = col[n - 1];
  if (x > (double)rl.y) {
    const double a = log((double)(1.f - rl.y)) / (double)rl.x;
    return log(1 - x) / a;
  }
  g = col_bisect<1>(col, n, x, r);
  return lin_f(r.y, r.x, r.w, r.z, x);
}

// One EGA growth step on one table column, FP64 path: eps(u(x) + u_seg) with
// the reference's operations (u_from_rec and eps_from_rec; below the first
// knot their LIN through the origin is the bracket of the column's origin).
//
// ega_step64 has the four knots from the previous step's bracket g on in hand
// (k01, k23; g = -1: the bracket between the origin and the first knot).  It
// covers x in the bracket g or g + 1 and the grown column in the same or the
// next one; ok is false for everything else (longer walks, beyond the last
// knot, whose end marks fail the comparisons) and ega_slow64 gives the
// result.  g returns the inverse bracket.
__device__ __forceinline__ double ega_step64(const float4 &k01, const float4 &k23, double x, double useg, int &g,
                                             bool &ok) {
  JUR_FP_EXACT
  const bool up = x >= (double)k01.w;
  const float u0 = up ? k01.z : k01.x, e0 = up ? k01.w : k01.y;
  const float u1 = up ? k23.x : k01.z, e1 = up ? k23.y : k01.w;
  const float u2 = up ? k23.z : k23.x, e2 = up ? k23.w : k23.y;
  const double arg = lin_f(e0, u0, e1, u1, x) + useg;
  const bool inb = arg < (double)u1;
  ok = (double)e0 <= x && x < (double)e1 && (double)u0 <= arg && (inb || arg < (double)u2);
  if (up) g++;
  const float ua = inb ? u0 : u1, ea = inb ? e0 : e1, ub = inb ? u1 : u2, eb = inb ? e1 : e2;
  return lin_f(ua, ea, ub, eb, arg);
}

__device__ __forceinline__ double ega_slow64(Col col, int n, double x, double useg, int &g) {
  JUR_FP_EXACT
  float4 r, r2;
  const int i = col_walk<1>(col, n, x, g, r);
  g = x < (double)r.y ? -1 : i;
  const double arg = u_from_rec(r, x) + useg;
  col_walk_r<0>(col, n, arg, i, r, r2);
  return eps_from_rec(r2, arg);
}

// Values of the lanes of a quad (lanes 4k..4k+3) by DPP: of lane K, and of
// the lane that differs in the bits X of its number.
template <int CTRL>
__device__ __forceinline__ int quad_dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float quad_dpp(float v) {
  return __int_as_float(quad_dpp<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double quad_dpp(double v) {
  return __hiloint2double(quad_dpp<CTRL>(__double2hiint(v)), quad_dpp<CTRL>(__double2loint(v)));
}
template <int K, typename V>
__device__ __forceinline__ V quad_lane(V v) { return quad_dpp<K * 0x55>(v); }
template <int X, typename V>
__device__ __forceinline__ V quad_xor(V v) {
  return quad_dpp<(0 ^ X) | (1 ^ X) << 2 | (2 ^ X) << 4 | (3 ^ X) << 6>(v);
}

// ------------------------------------------------------------------
// Continua (formod_continua, src/jurassic.c:3075-3117, with ctmco2
// :886-1744, ctmh2o :1746-2794, ctmn2 :2796-2859, ctmo2 :2861-2918), FP64.
// ------------------------------------------------------------------
// The continua split into a per-channel part (everything that depends only
// on the wavenumber) and a per-segment part, with the reference's
// operations: a radiance kernel evaluates the channel part once per lane
// instead of once per segment.  Two evaluations differ from the reference's
// expressions by a few ulp (radiances within 5e-16 relative), which halves
// the cost of the H2O term:
//  - the self-continuum power pow(cw260/cw296, (296 - T)/36) is
//    exp((296 - T)/36 * ln(cw260/cw296)), the logarithm taken once per
//    channel; for a ratio of 0, infinity or NaN this is what pow gives too,
//    except at exponent 0 (T = 296 K), where pow gives 1 and so does the
//    code;
//  - tanh(x), x = 0.7193876 nu / T > 0, is em / (em + 2) with em =
//    expm1(2x), which loses no digits for small x (1 beyond x = 20, where
//    tanh(x) rounds to 1).
struct CtmChan {
  bool co2, h2o, n2, o2;
  double co2_296, co2_260, co2_230;
  double h2o_slf, h2o_ratio, h2o_frn;  // sfac*cw296, cw260/cw296, cwfrn*fscal
  double h2o_lr;                       // ln(h2o_ratio)
  double n2_b, n2_beta, o2_b, o2_beta;
};

// h2o_ratio^e (the H2O self-continuum temperature power).
__device__ __forceinline__ double ctm_h2o_pow(const CtmChan &k, double e) {
  JUR_FP_EXACT
  return e == 0 ? 1.0 : exp(e * k.h2o_lr);
}

// tanh(x) for x >= 0.
__device__ __forceinline__ double tanh_pos(double x) {
  JUR_FP_EXACT
  if (x > 20) return 1.0;
  const double em = expm1(2 * x);
  return em / (em + 2);
}

__device__ __forceinline__ CtmChan ctm_chan(const CtmView &c, double nu) {
  JUR_FP_EXACT
  CtmChan k;
  k.co2 = k.h2o = k.n2 = k.o2 = false;
  k.co2_296 = k.co2_260 = k.co2_230 = k.h2o_slf = k.h2o_ratio = k.h2o_frn = 0;
  k.h2o_lr = 0;
  k.n2_b = k.n2_beta = k.o2_b = k.o2_beta = 0;
  {
    const double xw = nu / 2 + 1;
    if (xw >= 1 && xw < 2001) {
      const int iw = (int)xw;
      const double dw = xw - iw;
      const double ew = 1 - dw;
      k.co2 = true;
      k.co2_296 = ew * c.co2_296[iw - 1] + dw * c.co2_296[iw];
      k.co2_260 = ew * c.co2_260[iw - 1] + dw * c.co2_260[iw];
      k.co2_230 = ew * c.co2_230[iw - 1] + dw * c.co2_230[iw];
    }
  }
  {
    const double xw = nu / 10 + 1;
    if (xw >= 1 && xw < 2001) {
      const int iw = (int)xw;
      const double dw = xw - iw;
      const double ew = 1 - dw;
      const double cw296 = ew * c.h2o_296[iw - 1] + dw * c.h2o_296[iw];
      const double cw260 = ew * c.h2o_260[iw - 1] + dw * c.h2o_260[iw];
      const double cwfrn = ew * c.h2o_frn[iw - 1] + dw * c.h2o_frn[iw];
      double sfac;
      if (nu <= 820 || nu >= 960) {
        sfac = 1;
      } else {
        const double xx = (nu - 820) / 10;
        const int ix = (int)xx;
        const double dx = xx - ix;
        sfac = (1 - dx) * c.h2o_xfcrev[ix] + dx * c.h2o_xfcrev[ix + 1];
      }
      const double vf2 = (nu - 370) * (nu - 370);
      const double vf6 = vf2 * vf2 * vf2;
      const double fscal = 36100 / (vf2 + vf6 * 1e-8 + 36100) * -.25 + 1;
      k.h2o = true;
      k.h2o_slf = sfac * cw296;
      k.h2o_ratio = cw260 / cw296;
      k.h2o_lr = log(k.h2o_ratio);
      k.h2o_frn = cwfrn * fscal;
    }
  }
  if (!(nu < c.n2_nu[0] || nu > c.n2_nu[97])) {
    const int idx = locate_reg(c.n2_nu, 98, nu);
    k.n2 = true;
    k.n2_b = lin(c.n2_nu[idx], c.n2_b[idx], c.n2_nu[idx + 1], c.n2_b[idx + 1], nu);
    k.n2_beta = lin(c.n2_nu[idx], c.n2_beta[idx], c.n2_nu[idx + 1], c.n2_beta[idx + 1], nu);
  }
  if (!(nu < c.o2_nu[0] || nu > c.o2_nu[89])) {
    const int idx = locate_reg(c.o2_nu, 90, nu);
    k.o2 = true;
    k.o2_b = lin(c.o2_nu[idx], c.o2_b[idx], c.o2_nu[idx + 1], c.o2_b[idx + 1], nu);
    k.o2_beta = lin(c.o2_nu[idx], c.o2_beta[idx], c.o2_nu[idx + 1], c.o2_beta[idx + 1], nu);
  }
  return k;
}

// The per-segment parts take 1/T (rt) where the reference divides by T, and
// divide by constants as products with their reciprocals, folded at compile
// time: an FP64 division costs about fifteen instructions, and a product by
// a reciprocal differs from the quotient by at most an ulp or so.
__device__ __forceinline__ double ctmco2_seg(const CtmChan &k, double p, double t, double u) {
  JUR_FP_EXACT
  if (!k.co2) return 0;
  const double dt230 = t - 230;
  const double dt260 = t - 260;
  const double dt296 = t - 296;
  const double ctw = dt260 * 5.050505e-4 * dt296 * k.co2_230 - dt230 * 9.259259e-4 * dt296 * k.co2_260 +
                     dt230 * 4.208754e-4 * dt260 * k.co2_296;
  return u * (1 / JUR_NA / 1000 / JUR_P0) * p * ctw;
}

__device__ __forceinline__ double ctmh2o_seg(const CtmChan &k, double nu, double p, double t, double rt,
                                             double q, double u) {
  JUR_FP_EXACT
  if (!k.h2o) return 0;
  const double ctwslf = k.h2o_slf * ctm_h2o_pow(k, (296 - t) * (1.0 / (296 - 260)));
  const double a1 = nu * u * tanh_pos(.7193876 * nu * rt);
  const double a2 = 296 * rt;
  const double a3 = p * (1 / JUR_P0) * (q * ctwslf + (1 - q) * k.h2o_frn) * 1e-20;
  return a1 * a2 * a3;
}

__device__ __forceinline__ double ctmn2_seg(const CtmChan &k, double p, double t, double rt) {
  JUR_FP_EXACT
  if (!k.n2) return 0;
  const double q_n2 = 0.79, t0 = 273.0, tr = 296.0;
  const double r = p * (t0 / JUR_P0) * rt;
  return 0.1 * (r * r) * exp(k.n2_beta * (1 / tr - rt)) * q_n2 * k.n2_b *
         (q_n2 + (1 - q_n2) * (1.294 - t * (0.4545 / tr)));
}

__device__ __forceinline__ double ctmo2_seg(const CtmChan &k, double p, double rt) {
  JUR_FP_EXACT
  if (!k.o2) return 0;
  const double q_o2 = 0.21, t0 = 273, tr = 296;
  const double r = p * (t0 / JUR_P0) * rt;
  return 0.1 * (r * r) * exp(k.o2_beta * (1 / tr - rt)) * q_o2 * k.o2_b;
}

// formod_srcfunc (src/jurassic.c:3483-3496) for one channel column of the
// source-function table (sr_col[TBLNS]).
__device__ __forceinline__ double srcfunc(const double *st, const double *sr_col, double t) {
  JUR_FP_EXACT
  const int it = locate_reg(st, TBLNS, t);
  return lin(st[it], sr_col[it], st[it + 1], sr_col[it + 1], t);
}

// srcfunc on the uniform temperature grid with its inverse spacing inv_dst
// in hand (the per-segment form: products instead of the two divisions of
// locate_reg and LIN).
__device__ __forceinline__ double srcfunc_u(const double *st, double inv_dst, const double *sr_col, double t) {
  JUR_FP_EXACT
  int it = (int)((t - st[0]) * inv_dst);
  it = it < 0 ? 0 : (it > TBLNS - 2 ? TBLNS - 2 : it);
  return sr_col[it] + (sr_col[it + 1] - sr_col[it]) * inv_dst * (t - st[it]);
}

// PLANCK (src/jurassic.h:183-184).
__device__ __forceinline__ double planck(double t, double nu) {
  JUR_FP_EXACT
  return JUR_C1 * (nu * nu * nu) / expm1(JUR_C2 * nu / t);
}

// BRIGHT (src/jurassic.h:126-127).
__device__ __forceinline__ double bright(double rad, double nu) {
  JUR_FP_EXACT
  return JUR_C2 * nu / log1p(JUR_C1 * (nu * nu * nu) / rad);
}

// XCD-aware work mapping.  The hardware hands workgroup ids to the 8 XCDs
// round-robin (id % 8).  A ray block's G work items (its channels, or its
// channel-emitter chains) should share one XCD's L2, since they read the
// same LOS data; consecutive ray blocks should go to different XCDs, since
// block cost varies smoothly with geometry (limb ray length grows with
// depth) and contiguous ranges would unbalance the XCDs.  With the grid padded
// to nblk8 = 8 ceil(nblk/8) blocks, workgroup wg maps to block
// 8 (k / G) + x and item k % G, x = wg % 8, k = wg / 8: a bijection in which
// XCD x owns blocks x, x+8, x+16, ...  Returns false for padding groups.
__device__ __forceinline__ bool xcd_block_map(int wg, int G, int nblk, int &blk, int &item) {
  const int x = wg & 7, k = wg >> 3;
  const int q = k / G;
  item = k - q * G;
  blk = q * 8 + x;
  return blk < nblk;
}

__host__ __device__ __forceinline__ int padded_blocks(int nblk) { return (nblk + 7) & ~7; }

// ------------------------------------------------------------------
// Sums along a path in chunks of RAD_CH points (the FP32 radiance kernel): each
// chunk's radiance, transmittance and down-welling sum as if it began the
// path, joined in path order.  The chunks do not depend on each other, so a
// small batch, whose duration is one path's, takes them on the PW waves of a
// workgroup (32 points: a few rounds of 16 waves for the ~800 to 1500 points
// of a path, against a join of three operations); a large one in one wave.
// Both join the same chunks in the same order, so the sums are the same bits.
// ------------------------------------------------------------------
constexpr int RAD_CH = 32;

struct PathSum {
  double rad = 0, tau = 1, drefl = 0;
  __device__ __forceinline__ void append(const PathSum &c) {
    JUR_FP_EXACT
    rad = rad + tau * c.rad;
    drefl = drefl * c.tau + c.drefl;
    tau = tau * c.tau;
  }
  // sum: the path up to this round's PW chunks, c: the wave's chunk
  template <int PW>
  static __device__ __forceinline__ void join(PathSum &sum, double (*part)[3][WAVE], int wv, int lane,
                                              const PathSum &c) {
    if constexpr (PW == 1) {
      sum.append(c);
    } else {
      part[wv][0][lane] = c.rad;
      part[wv][1][lane] = c.tau;
      part[wv][2][lane] = c.drefl;
      __syncthreads();
      if (wv == 0)
        for (int k = 0; k < PW; k++) sum.append(PathSum{part[k][0][lane], part[k][1][lane], part[k][2][lane]});
      __syncthreads();
    }
  }
};

// Runs a kernel of g workgroups with the most waves each, TOP, 4 or 1, that
// stay within `all` waves (what runs at once).
template <int TOP, typename F>
void launch_paths(unsigned g, unsigned all, F run) {
  if (g <= all / TOP) run(std::integral_constant<int, TOP>{});
  else if (g <= all / 4) run(std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 1>{});
}

// ------------------------------------------------------------------
// Ray state handed from the march (raytrace.hip) to its finish and to the
// adjoint of the refracted path (adjoint.hip).
// ------------------------------------------------------------------
// First minimum of z along the LOS (gsl_stats_min_index semantics: a NaN
// ends the search) and the positions of its two neighbours, for
// tangent_point.
struct MinTrack {
  double zlow = 0;
  double xbefore[3] = {0, 0, 0}, xafter[3] = {0, 0, 0};
  int imin = 0;
  bool after_pending = false, nan_seen = false;
  // point np at z, position x; xprev is the position of point np - 1
  __device__ __forceinline__ void add(int np, double z, const double *x, const double *xprev) {
    if (!nan_seen) {
      const bool lower = (np == 0) || z < zlow;
      if (lower) zlow = z;
      if (lower || isnan(z)) {
        imin = np;
        if (np > 0)
          for (int i = 0; i < 3; i++) xbefore[i] = xprev[i];
        after_pending = true;
        nan_seen = isnan(z);
      } else if (after_pending) {
        for (int i = 0; i < 3; i++) xafter[i] = x[i];
        after_pending = false;
      }
    } else if (after_pending) {
      for (int i = 0; i < 3; i++) xafter[i] = x[i];
      after_pending = false;
    }
  }
};

// What the march (k_raytrace) hands to k_ray_finish for a ray with LOS
// points: the step that left the altitude range, which is clipped to it
// there, and the state for the tangent point.
struct RayTail {
  double xprev[3];  // the last point written
  double xcut[3];   // the step beyond the altitude range
  double xfirst[3];
  double zprev, zcut, dscut;  // altitudes of both, step length
  double zmin, zmax;
  double ds1, ds2;            // raw step lengths of the last two points written
  double ds_imin, ds_imin1;   // raw step lengths at the first minimum and after it
  double ecut[3];             // the march direction at the step beyond the range
  MinTrack mt;
  int zdir;
};

}  // namespace jur
