// Analytic culling of Gaussian footprints for the rasterizer and voxelizer.
//
// A (pixel|voxel, Gaussian) pair contributes only if alpha = w exp(-sigma)
// passes |alpha| >= thr with sigma >= 0, where sigma = 1/2 d^T P d.  For a
// positive-definite P that can only happen inside the ellipsoid
// sigma <= s*, s* = ln(|w| / thr).  These helpers walk that ellipsoid as
// slices -> rows -> a segment along the contiguous axis, using the
// completed-square forms
//   2D: sigma = 1/2 a (x - xc(y))^2 + 1/2 (det / a) y^2,      xc = -(b / a) y
//   3D: sigma = 1/2 p00 (x - xc(y, z))^2 + 1/2 a2 (y - yc(z))^2 + 1/2 c3 z^2
// (a2, c3 Schur complements), whose terms are all non-negative, so the
// remaining budget s - (terms so far) carries no cancellation error.  Every
// range is conservative:
//   * s* is enlarged by a relative 1e-3 and an absolute 1e-3;
//   * every interval end is widened by kCullMargin (0.125) pixel/voxel.
// Elements inside a range are still evaluated with the per-element test, so
// culling only removes elements that cannot pass it.  Determinants and Schur
// complements are computed in double.
#pragma once

#include "r2s_common.h"

namespace r2s {

constexpr double kCullMargin = 0.125;
constexpr double kLog2e = 1.4426950408889634074;

// 2^-x: one v_exp_f32 for float (the kernels pre-scale sigma by log2(e), so
// exp(-sigma) = 2^-(sigma log2 e)); the library exp2 for double.
__device__ __forceinline__ float neg_exp2(float x) { return __builtin_amdgcn_exp2f(-x); }
__device__ __forceinline__ double neg_exp2(double x) { return exp2(-x); }

// e[k] = 2^-sl[k] as one run of v_exp_f32 at raised wave priority.
// gfx950 issues the simple vector instructions (FMA, add, multiply, compare,
// select) of two waves of a SIMD together, but v_exp_f32 holds the whole
// vector unit for 8 cycles, and at equal priority the oldest wave runs its
// exps and its arithmetic alone while the others queue up at theirs.  With
// the exps at a higher priority every wave passes them as soon as it gets
// there, and the arithmetic between them pairs.  Measured in registers on
// the raster backward's pixel (two FMAs, exp, compare, select, product, five
// accumulations), 4 or 5 waves per SIMD: 42-48 cycles per pixel with equal
// priorities, 32-33 with exps in runs of 4 to 16 at priority 3 (34 for runs
// of one); on the forward's pixel 25-29 and 20-22.
template <typename T, int N>
__device__ __forceinline__ void neg_exp2_run(const T (&sl)[N], T (&e)[N]) {
  __builtin_amdgcn_s_setprio(3);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    e[k] = neg_exp2(sl[k]);
    asm volatile("" : "+v"(e[k]));  // formed here, not at its use
  }
  __builtin_amdgcn_s_setprio(0);
}

// The per-element alpha test -- sigma >= 0 and |w| exp(-sigma) >= thr, with
// sl = sigma log2(e) -- as one unsigned compare of sl's bit pattern.
// Non-negative values order like their patterns, and every negative value
// (and -0, -inf, a negative NaN) has a larger pattern than any non-negative
// one, so with sl* = log2(|w| / thr) >= 0:
//   sl in [+0, sl*]  <=>  bits(sl) < bits(sl*) + 1.
// Limits by record:
//   * |w| < thr: 0, nothing passes (|alpha| <= |w| for sigma >= 0);
//   * non-finite geometry or a NaN w: the sign bit, so every sl >= +0, +inf
//     and a positive NaN pass -- their alpha is 0 or non-finite, which the
//     reference does not skip either -- and sl < 0 fails, as there.
// It differs from testing exp(-sigma) against thr / |w| only for elements
// whose alpha is within a few ulp of thr.
template <typename T>
struct Bits;
template <>
struct Bits<float> {
  using type = uint32_t;
  static constexpr uint32_t kSign = 0x80000000u;
};
template <>
struct Bits<double> {
  using type = uint64_t;
  static constexpr uint64_t kSign = 0x8000000000000000ull;
};

__device__ __forceinline__ uint32_t bits_of(float x) { return __float_as_uint(x); }
__device__ __forceinline__ uint64_t bits_of(double x) {
  return static_cast<uint64_t>(__double_as_longlong(x));
}

template <typename T>
__device__ __forceinline__ typename Bits<T>::type alpha_limit(T w, bool finite_geometry,
                                                              double thr) {
  const T aw = fabs(w);
  if (aw != aw || !finite_geometry) return Bits<T>::kSign;
  if (!(aw >= static_cast<T>(thr))) return 0;
  // log2(|w| / thr) >= 0 (+inf for an infinite w).
  const T sl_max = fmax(log2(aw) - static_cast<T>(log2(thr)), static_cast<T>(0));
  return bits_of(sl_max) + 1;
}

template <typename T>
__device__ __forceinline__ bool alpha_pass(T sl, typename Bits<T>::type limit) {
  return bits_of(sl) < limit;
}

// acc += w e (e = 2^-sl) where the alpha test passes; a failing pair adds
// nothing, where a select would add w * 0 (NaN for a non-finite w).  In
// float the compare writes the execution mask (`full`, the caller's
// __builtin_amdgcn_read_exec(), restores it): one vector instruction instead
// of a compare and a select, and no wait for a scalar mask.  In double the
// scheduling barrier keeps the branch from being turned into a select.
__device__ __forceinline__ void add_passing(float sl, float e, uint32_t limit, float w, float &acc,
                                            uint64_t full) {
  asm volatile(
      "v_cmpx_gt_u32_e32 vcc, %1, %2\n\t"
      "v_fmac_f32_e32 %0, %3, %4\n\t"
      "s_mov_b64 exec, %5"
      : "+v"(acc)
      : "v"(limit), "v"(sl), "v"(w), "v"(e), "s"(full)
      : "vcc");
}
__device__ __forceinline__ void add_passing(double sl, double e, uint64_t limit, double w,
                                            double &acc, uint64_t) {
  if (alpha_pass(sl, limit)) {
    __builtin_amdgcn_sched_barrier(0);
    acc = fma(w, e, acc);
  }
}

// Bits of a limit kept in a T slot (forward records stage it in LDS).
__device__ __forceinline__ float limit_as_value(uint32_t b) { return __uint_as_float(b); }
__device__ __forceinline__ double limit_as_value(uint64_t b) {
  return __longlong_as_double(static_cast<long long>(b));
}

// Keys of the records of a wave: `rb` is the wave's first record (uniform),
// `r` the lane's; the key of record r is the last k with offsets[k] <= r, or
// 0 where there is none (offsets non-decreasing; any others give some key
// below n_keys).  One uniform search for rb, then a
// uniform walk over the next few keys' first indices; a window holding more
// boundaries than that (empty keys share their successor's first index, so
// a run of them is many boundaries at one index) finishes with a per-lane
// binary search above the walk's last key.
__device__ __forceinline__ uint32_t wave_record_key(const int32_t *__restrict__ offsets,
                                                    uint32_t n_keys, int64_t n_isects, int64_t rb,
                                                    int64_t r) {
  constexpr uint32_t kWalk = 4;
  // 64 evenly spaced keys a round, one per lane: three memory round trips for
  // 2^18 keys, where a binary search's eighteen dependent ones were a few per
  // cent of the waves' time.
  uint32_t lo = 0, hi = n_keys;
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + 63) / 64;
    const uint32_t at = lo + lane_id() * step;
    const bool below = at < hi && static_cast<int64_t>(offsets[at]) <= rb;
    // No lane is below where a caller's offsets start after rb: key 0 then.
    lo += static_cast<uint32_t>(max(static_cast<int>(__popcll(ballot(below))), 1) - 1) * step;
    hi = min(lo + step, hi);
  }
  const int64_t r_last = min(rb + 63, n_isects - 1);
  uint32_t key = lo;
  uint32_t k = lo + 1;
  for (uint32_t step = 0; step < kWalk; ++step, ++k) {
    if (k >= n_keys) return key;
    const int64_t bnd = offsets[k];
    if (bnd > r_last) return key;
    if (r >= bnd) key = k;
  }
  // offsets[key] <= r: the last such key at or above it.
  uint32_t a = key, b = n_keys;
  while (b - a > 1) {
    const uint32_t mid = (a + b) >> 1;
    if (static_cast<int64_t>(offsets[mid]) <= r)
      a = mid;
    else
      b = mid;
  }
  return a;
}

// Square root for culling bounds: the hardware v_sqrt_f32 (about 1 ulp),
// far inside the margins, instead of the correctly rounded expansion.
__device__ __forceinline__ float cull_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double cull_sqrt(double x) { return sqrt(x); }

// Enlarged ln(|w| / thr); the float log is ample against the 1e-3 slack.
__device__ __forceinline__ float sigma_bound(float w_abs, double thr) {
  return (logf(w_abs) - static_cast<float>(log(thr))) * (1.0f + 1e-3f) + 1e-3f;
}
__device__ __forceinline__ double sigma_bound(double w_abs, double thr) {
  return log(w_abs / thr) * (1.0 + 1e-3) + 1e-3;
}

// Integer indices j with (j + 0.5) in [c + lo, c + hi], clamped to [j0, j1].
// Returns false when empty.  Inputs may be non-finite (empty or clamped).
template <typename T>
__device__ __forceinline__ bool index_range(T c, T lo, T hi, int j0, int j1, int &a, int &b) {
  const T flo = ceil(c + lo - static_cast<T>(0.5 + kCullMargin));
  const T fhi = floor(c + hi - static_cast<T>(0.5 - kCullMargin));
  const T cl = fmax(flo, static_cast<T>(j0));
  const T ch = fmin(fhi, static_cast<T>(j1));
  if (!(cl <= ch)) return false;
  a = static_cast<int>(cl);
  b = static_cast<int>(ch);
  return true;
}

// Indices j of [j0, j1] with (j + 0.5 - c - centre)^2 <= 2 budget / p, i.e.
// the segment where 1/2 p (u - centre)^2 <= budget.
template <typename T>
__device__ __forceinline__ bool budget_range(T c, T centre, T budget, T inv_p, int j0, int j1,
                                             int &a, int &b) {
  if (!(budget >= static_cast<T>(0))) return false;
  const T h = sqrt(static_cast<T>(2) * budget * inv_p);
  return index_range<T>(c, centre - h, centre + h, j0, j1, a, b);
}

// 2D footprint of conic (a, b, c) = P for weight |w|.
template <typename T>
struct Cull2 {
  bool ok;   // positive definite and finite: the analytic ranges apply
  T s;       // sigma bound
  T hy;      // half extent along y
  T inv_a;   // 1 / a
  T bx;      // x centre per unit y: xc = -bx y  (b / a)
  T c2;      // det / a: row minimum 1/2 c2 y^2
};

template <typename T>
__device__ __forceinline__ Cull2<T> cull2_setup(T a, T b, T c, T w_abs, double thr) {
  Cull2<T> r;
  const double da = a, db = b, dc = c;
  const double det = da * dc - db * db;
  r.ok = (da > 0.0) && (det > 0.0) && isfinite(det) && isfinite(da) &&
         isfinite(static_cast<double>(w_abs));
  r.s = r.hy = r.inv_a = r.bx = r.c2 = 0;
  if (r.ok) {
    const double s = static_cast<double>(sigma_bound(w_abs, thr));
    r.s = static_cast<T>(s);
    r.hy = static_cast<T>(s > 0.0 ? sqrt(2.0 * s * da / det) : 0.0);
    r.inv_a = static_cast<T>(1.0 / da);
    r.bx = static_cast<T>(db / da);
    r.c2 = static_cast<T>(det / da);
  }
  return r;
}

// 3D footprint of the packed conic q = (p00, p01, p02, p11, p12, p22), axis 0
// of the conic = x (contiguous), 1 = y, 2 = z.
template <typename T>
struct Cull3 {
  bool ok;
  T s;
  T hz;          // half extent along z
  T inv_p;       // 1 / p00
  T a2, inv_a2;  // p11 - p01^2 / p00 and its inverse
  T ky;          // y centre per unit z: yc = -ky z
  T c3;          // det / (p00 a2): slice minimum 1/2 c3 z^2
  // The slice ellipse 1/2 p00 (x - xc)^2 + 1/2 a2 (y - yc)^2 <= budget, with
  // xc = -(kx y + kz z), as vertical chords: at x = xe + u (xe its centre)
  //   1/2 p11 (y - ye + r11 u)^2 + 1/2 e11 u^2 <= budget.
  T kx, kz;      // p01 / p00, p02 / p00
  T r11;         // p01 / p11
  T e11;         // (p00 p11 - p01^2) / p11
  T inv_p11;     // 1 / p11
};

template <typename T>
__device__ __forceinline__ Cull3<T> cull3_setup(const T q[6], T w_abs, double thr) {
  Cull3<T> r;
  const double p00 = q[0], p01 = q[1], p02 = q[2], p11 = q[3], p12 = q[4], p22 = q[5];
  const double m2 = p00 * p11 - p01 * p01;
  const double det = p00 * (p11 * p22 - p12 * p12) - p01 * (p01 * p22 - p12 * p02) +
                     p02 * (p01 * p12 - p11 * p02);
  r.ok = (p00 > 0.0) && (m2 > 0.0) && (det > 0.0) && isfinite(det) && isfinite(m2) &&
         isfinite(static_cast<double>(w_abs));
  r.s = r.hz = r.inv_p = r.a2 = r.inv_a2 = r.ky = r.c3 = 0;
  r.kx = r.kz = r.r11 = r.e11 = r.inv_p11 = 0;
  if (r.ok) {
    // Four reciprocals serve every quotient (a few ulp of double, far
    // inside the margins); the differences of products stay in double.
    const double ip00 = 1.0 / p00, im2 = 1.0 / m2, ip11 = 1.0 / p11, idet = 1.0 / det;
    const double s = static_cast<double>(sigma_bound(w_abs, thr));
    const double a2 = m2 * ip00;
    const double k1 = p12 - p01 * p02 * ip00;
    r.s = static_cast<T>(s);
    r.hz = static_cast<T>(s > 0.0 ? sqrt(2.0 * s * m2 * idet) : 0.0);
    r.inv_p = static_cast<T>(ip00);
    r.a2 = static_cast<T>(a2);
    r.inv_a2 = static_cast<T>(p00 * im2);
    r.ky = static_cast<T>(k1 * p00 * im2);
    r.c3 = static_cast<T>(det * im2);
    r.kx = static_cast<T>(p01 * ip00);
    r.kz = static_cast<T>(p02 * ip00);
    r.r11 = static_cast<T>(p01 * ip11);  // p11 > 0 follows from m2 > 0, p00 > 0
    r.e11 = static_cast<T>(m2 * ip11);
    r.inv_p11 = static_cast<T>(ip11);
  }
  return r;
}

}  // namespace r2s
