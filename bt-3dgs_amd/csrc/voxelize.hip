// Brick-tiled voxelizer: volume = per voxel sum over its brick's Gaussian
// list of opacity * exp(-sigma), sigma = 1/2 d^T conic d, skipping sigma < 0
// and |alpha| < 1e-6 (r2splat/cuda/csrc/VoxelizeToVoxelsFwd.cu:69-221), and
// its VJP (VoxelizeToVoxelsBwd.cu:71-441).
//
// sigma is evaluated along x-rows of a brick: with dy, dz fixed per row,
//   sigma log2(e) = (h0 dx + B) dx + C,  h0 = p00 log2(e) / 2,
// two FMAs per voxel and one v_exp_f32 for exp(-sigma) = 2^-(sigma log2 e).
//
// Forward: one workgroup per brick.  At brick size 8 a lane owns an x-row of
// eight voxels and one to four waves share the brick's list (in a fixed order:
// the result is deterministic); at other sizes a thread owns a voxel and sums
// the list in order, as the reference does.  Records are staged in LDS in
// batches with their conics pre-scaled and read as broadcasts.
//
// Backward: one lane per record of the sorted list, so a wave takes 64
// consecutive records (nearly always of one brick) and the work is balanced
// whatever the list lengths.  All lanes walk the brick-local rows together,
// skipping every slice and row that no lane's alpha-test ellipsoid reaches
// (r2s_cull.h, wave ballots); a lane loads the upstream-gradient row of its
// own brick (lanes of one brick share the cache lines).  Per row a lane accumulates
// the moments s_k = sum(w dx^k), k = 0..2, of w = v exp(-sigma) over passing
// voxels, and per record the ten sums
//   T_k = sum s_k,  Y0 = sum dy s0, Z0 = sum dz s0, Y1 = sum dy s1,
//   Z1 = sum dz s1, YY = sum dy^2 s0, YZ = sum dy dz s0, ZZ = sum dz^2 s0,
// from which the ten partials follow.  They go out through float atomics
// (one-pass form) or as the record's row of a table that r2s_rows.h reduces
// per Gaussian (two-pass form).  The two reference backward variants (per
// voxel, per Gaussian) compute the same sums and share this kernel.
#include "r2s_common.h"
#include "r2s_cull.h"
#include "r2s_rows.h"
#include "r2s_scan.h"

namespace r2s {
namespace {

constexpr double kThr3 = 1e-6;
constexpr int kBwdThreads = 256;
constexpr uint32_t kFwdBatch = 256;

template <typename T>
struct Vec;
template <>
struct Vec<float> {
  using v2 = float2;
  using v4 = float4;
};
template <>
struct Vec<double> {
  using v2 = double2;
  using v4 = double4;
};

struct Brick {
  int oi, oj, ok;  // origin (dim0, dim1, dim2)
  int ni, nj, nk;  // extent inside the volume (0 in bricks of a larger grid)
};

__device__ __forceinline__ Brick brick_of(uint32_t key, uint32_t n2, uint32_t n1, uint32_t ts,
                                          uint32_t D2, uint32_t D1, uint32_t D0) {
  const uint32_t b0 = key / (n1 * n2), rem = key - b0 * (n1 * n2);
  const uint32_t b1 = rem / n2, b2 = rem - b1 * n2;
  Brick b;
  b.oi = static_cast<int>(b0 * ts);
  b.oj = static_cast<int>(b1 * ts);
  b.ok = static_cast<int>(b2 * ts);
  // The grid may be larger than the volume: no wrap below zero.
  b.ni = static_cast<int>(min(ts, D0 - min(D0, b0 * ts)));
  b.nj = static_cast<int>(min(ts, D1 - min(D1, b1 * ts)));
  b.nk = static_cast<int>(min(ts, D2 - min(D2, b2 * ts)));
  return b;
}

// Pre-scaled conic: sigma log2(e) = (h0 dx + h1 dy + h2 dz) dx
//                                  + (h3 dy + h4 dz) dy + h5 dz^2.
template <typename T>
__device__ __forceinline__ void scaled_conic(const T q[6], T h[6]) {
  const T l = static_cast<T>(kLog2e), hl = static_cast<T>(0.5 * kLog2e);
  h[0] = hl * q[0];
  h[1] = l * q[1];
  h[2] = l * q[2];
  h[3] = hl * q[3];
  h[4] = l * q[4];
  h[5] = hl * q[5];
}

// Forward for brick sizes other than 8: one thread per voxel.
template <typename T>
__global__ __launch_bounds__(1024) void voxel_fwd_kernel(
    const T *__restrict__ means3d, const T *__restrict__ conics, const T *__restrict__ opac,
    const int32_t *__restrict__ tile_offsets, const int32_t *__restrict__ flatten_ids,
    int64_t n_isects, uint32_t n_keys, uint32_t koff, int64_t N, uint32_t D2, uint32_t D1,
    uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, T *__restrict__ volume) {
  using V4 = typename Vec<T>::v4;
  extern __shared__ double smem_raw[];
  const uint32_t nt = blockDim.x;
  const uint32_t nb = min(nt, kFwdBatch);  // records staged per batch
  // Per staged record: {mx, my, mz, o}, {h0, h1, h2, h3}, {h4, h5, limit bits, 0}.
  V4 *s_rec = reinterpret_cast<V4 *>(smem_raw);

  const uint32_t key = xcd_swizzle(blockIdx.x, n_keys);  // in the lists (koff: the grid's)
  const Brick b = brick_of(key + koff, n2, n1, ts, D2, D1, D0);
  const uint32_t tid = threadIdx.x;
  const int lk = static_cast<int>(tid % ts);
  const int lj = static_cast<int>((tid / ts) % ts);
  const int li = static_cast<int>(tid / (ts * ts));
  const T half = static_cast<T>(0.5);
  const T py = static_cast<T>(b.oj + lj) + half;
  const T pz = static_cast<T>(b.oi + li) + half;
  const T px = static_cast<T>(b.ok + lk) + half;

  const int64_t start = tile_offsets[key];
  const int64_t end = (key == n_keys - 1) ? n_isects : static_cast<int64_t>(tile_offsets[key + 1]);
  T acc = 0;
  for (int64_t base = start; base < end; base += nb) {
    __syncthreads();
    const int64_t idx = base + tid;
    if (tid < nb && idx < end) {
      int64_t g = flatten_ids[idx];
      V4 mo, h0, h1;
      if (g >= 0 && g < N) {
        T q[6], h[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) q[c] = conics[6 * g + c];
        scaled_conic(q, h);
        mo.x = means3d[3 * g];
        mo.y = means3d[3 * g + 1];
        mo.z = means3d[3 * g + 2];
        mo.w = opac[g];
        h0.x = h[0];
        h0.y = h[1];
        h0.z = h[2];
        h0.w = h[3];
        h1.x = h[4];
        h1.y = h[5];
        // The alpha test's limit on the bits of sl (alpha_limit), kept in h1.z.
        bool fin = isfinite(mo.x) && isfinite(mo.y) && isfinite(mo.z);
#pragma unroll
        for (int c = 0; c < 6; ++c) fin = fin && isfinite(h[c]);
        h1.z = limit_as_value(alpha_limit(mo.w, fin, kThr3));
      } else {  // never passes
        mo.x = mo.y = mo.z = mo.w = 0;
        h0.x = h0.y = h0.z = h0.w = 0;
        h1.x = h1.y = 0;
        h1.z = limit_as_value(static_cast<typename Bits<T>::type>(0));
      }
      h1.w = 0;
      s_rec[3 * tid] = mo;
      s_rec[3 * tid + 1] = h0;
      s_rec[3 * tid + 2] = h1;
    }
    __syncthreads();
    const int cnt = static_cast<int>(min(static_cast<int64_t>(nb), end - base));
    const uint64_t exec = __builtin_amdgcn_read_exec();
    for (int t = 0; t < cnt; ++t) {
      const V4 mo = s_rec[3 * t];
      const V4 h0 = s_rec[3 * t + 1];
      const V4 h1 = s_rec[3 * t + 2];
      const typename Bits<T>::type lim = bits_of(h1.z);
      const T dx = px - mo.x, dy = py - mo.y, dz = pz - mo.z;
      const T B = h0.y * dy + h0.z * dz;
      const T C = (h0.w * dy + h1.x * dz) * dy + h1.y * dz * dz;
      const T sl[1] = {fma(fma(h0.x, dx, B), dx, C)};
      T e[1];
      neg_exp2_run(sl, e);
      add_passing(sl[0], e[0], lim, mo.w, acc, exec);
    }
  }
  if (li < b.ni && lj < b.nj && lk < b.nk)
    volume[static_cast<int64_t>(b.oi + li) * D1 * D2 + static_cast<int64_t>(b.oj + lj) * D2 +
           (b.ok + lk)] = acc;
}

// One backward record in registers.
template <typename T>
struct BwdRecord {
  bool live;     // a valid record whose voxels can pass the alpha test
  T m[3], q[6], h[6], o;
  typename Bits<T>::type lim;  // the alpha test on the bits of sl (alpha_limit)
  Cull3<T> cu;
  int i0, i1;    // slice range (all slices when !cu.ok)
};

// A record's geometry, opacity and alpha limit; every slice of the brick in
// range (no culling).
template <typename T>
__device__ __forceinline__ void load_bwd_record_plain(const T *__restrict__ means3d,
                                                      const T *__restrict__ conics,
                                                      const T *__restrict__ opac, int64_t g,
                                                      int64_t N, bool in_list, const Brick &b,
                                                      BwdRecord<T> &rec) {
  rec.live = in_list && g >= 0 && g < N;
  // Loaded together (one memory round trip), the opacity tested after.
  const int64_t gl = rec.live ? g : 0;
  rec.o = opac[gl];
#pragma unroll
  for (int c = 0; c < 3; ++c) rec.m[c] = means3d[3 * gl + c];
#pragma unroll
  for (int c = 0; c < 6; ++c) rec.q[c] = conics[6 * gl + c];
  // |alpha| <= |o| for sigma >= 0: nothing passes (non-finite o stays live).
  if (fabs(rec.o) < static_cast<T>(kThr3)) rec.live = false;
  rec.cu.ok = false;
  if (!rec.live) {
    rec.o = 0;
    rec.lim = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) rec.m[c] = 0;
#pragma unroll
    for (int c = 0; c < 6; ++c) rec.q[c] = rec.h[c] = 0;
    rec.i0 = 0;
    rec.i1 = -1;
    return;
  }
  scaled_conic(rec.q, rec.h);
  bool fin = true;
#pragma unroll
  for (int c = 0; c < 3; ++c) fin = fin && isfinite(rec.m[c]);
#pragma unroll
  for (int c = 0; c < 6; ++c) fin = fin && isfinite(rec.h[c]);
  rec.lim = alpha_limit(rec.o, fin, kThr3);
  rec.i0 = b.oi;
  rec.i1 = b.oi + b.ni - 1;
}

// As load_bwd_record_plain, with the culling setup and the slice range of
// the record's alpha-test ellipsoid (a record reaching no slice is dead).
template <typename T>
__device__ __forceinline__ void load_bwd_record(const T *__restrict__ means3d,
                                                const T *__restrict__ conics,
                                                const T *__restrict__ opac, int64_t g, int64_t N,
                                                bool in_list, const Brick &b, BwdRecord<T> &rec) {
  load_bwd_record_plain(means3d, conics, opac, g, N, in_list, b, rec);
  if (!rec.live) return;
  rec.cu = cull3_setup(rec.q, fabs(rec.o), kThr3);
  if (rec.cu.ok &&
      !index_range<T>(rec.m[2], -rec.cu.hz, rec.cu.hz, b.oi, b.oi + b.ni - 1, rec.i0, rec.i1))
    rec.live = false;
}

// Moments of one brick row for one record: s0 = sum w, s1 = sum w dx,
// s2 = sum w dx^2 over the row's passing voxels (w = v exp(-sigma)).  vv
// holds the row's upstream gradient (zero beyond the volume).  kGuard: also
// exclude columns k >= nk explicitly -- needed only for records whose sigma
// may be NaN (non-finite geometry passes the alpha test there), for which
// v = 0 would not make w = 0.
template <typename T, int R, bool kExact, bool kGuard>
__device__ __forceinline__ void voxel_row(const BwdRecord<T> &rec, const T (&vv)[R], T dx0,
                                          int nk, int nts, T B, T C, T &s0, T &s1, T &s2) {
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if (!kExact && k >= nts) break;
    const T dx = dx0 + static_cast<T>(k);
    const T sl = (rec.h[0] * dx + B) * dx + C;
    const T e = neg_exp2(sl);
    bool skip = !alpha_pass(sl, rec.lim);
    if (kGuard) skip = skip || k >= nk;
    const T p = vv[k] * e;  // unconditional, not a branch around the load and exp
    const T w = skip ? static_cast<T>(0) : p;
    s0 += w;
    const T wx = w * dx;
    s1 += wx;
    s2 += wx * dx;
  }
}

// Slice range of one record's brick rows: rows j0..j1 of slice dz whose
// voxels (columns dx0 .. dx0 + nk - 1 as offsets from the mean) the
// ellipsoid reaches; empty (j1 < j0) when none.  In the slice, the reached
// part of the ellipse is its intersection with the brick's x-band, a convex
// set, so its rows are one range: the top is the top of the vertical chord
// at the band point nearest the ellipse's topmost point (chord tops are a
// concave function of x), the bottom likewise; every term is a completed
// square, so nothing cancels.  The band is widened by kCullMargin and the
// rows are taken with index_range's margin.
template <typename T>
__device__ __forceinline__ void slice_rows(const BwdRecord<T> &rec, const Brick &b, bool in_slice,
                                           T dz, T dx0, int &j0, int &j1) {
  j0 = b.oj;
  j1 = b.oj + b.nj - 1;
  if (!in_slice) {
    j1 = j0 - 1;
    return;
  }
  if (!rec.cu.ok) return;  // every row
  const Cull3<T> &c = rec.cu;
  const T half = static_cast<T>(0.5), two = static_cast<T>(2);
  const T m = static_cast<T>(kCullMargin);
  const T bud = c.s - half * c.c3 * dz * dz;
  const T ye = -c.ky * dz;
  const T xe = -(c.kx * ye + c.kz * dz);
  const T hy = cull_sqrt(fmax(two * bud * c.inv_a2, static_cast<T>(0)));
  const T ulo = (dx0 - m) - xe;
  const T uhi = (dx0 + static_cast<T>(b.nk - 1) + m) - xe;
  // Topmost point of the ellipse at u = -kx hy, bottommost at +kx hy.
  const T ut = fmin(fmax(-c.kx * hy, ulo), uhi);
  const T ub = fmin(fmax(c.kx * hy, ulo), uhi);
  const T rt = bud - half * c.e11 * ut * ut;
  const T rb = bud - half * c.e11 * ub * ub;
  if (!(bud >= static_cast<T>(0)) || !(rt >= static_cast<T>(0))) {
    j1 = j0 - 1;  // the slice, or the band, misses the ellipse
    return;
  }
  const T top = ye + (cull_sqrt(two * rt * c.inv_p11) - c.r11 * ut);
  const T bot = ye - (cull_sqrt(fmax(two * rb * c.inv_p11, static_cast<T>(0))) + c.r11 * ub);
  if (!index_range<T>(rec.m[1], bot, top, b.oj, b.oj + b.nj - 1, j0, j1)) j1 = j0 - 1;
}

// The rows of a brick of size 8 that one record reaches, as a 64-bit mask:
// bit 8 * slice + row (brick-local).
template <typename T>
__device__ __forceinline__ uint64_t reach_mask(const BwdRecord<T> &rec, const Brick &b, T dx0) {
  const T half = static_cast<T>(0.5);
  uint64_t reach = 0;
#pragma unroll 1
  for (int li = 0; li < 8; ++li) {
    const int i = b.oi + li;
    const bool in_slice = rec.live && li < b.ni && i >= rec.i0 && i <= rec.i1;
    const T dz = (static_cast<T>(i) + half) - rec.m[2];
    int j0, j1;
    slice_rows(rec, b, in_slice, dz, dx0, j0, j1);
    const uint32_t c = j1 >= j0 ? static_cast<uint32_t>(j1 - j0 + 1) : 0u;  // rows j0 - oj ..
    const uint32_t run = c >= 8u ? 0xFFu : ((1u << c) - 1u);
    reach |= static_cast<uint64_t>((run << ((j0 - b.oj) & 7)) & 0xFFu) << (8 * li);
  }
  return reach;
}

// A batch of the forward below whose records reach at least this share of
// their 64 rows on average walks every row: no set to step through, uniform
// reads of the staged records, no transpose; and the wave's next batch does
// so without its masks while half of its records look as large (box_is_dense,
// a few operations a record where the masks take hundreds).  Measured on
// trees (6.8 M records of a 250 x 201 x 173 volume, nearly every row reached)
// 0.974 -> 0.785 ms, 0.883 with every batch's masks formed; and on 2000 large
// Gaussians before 600k tiny ones at 128^3 0.207 -> 0.196 ms, where a wave
// that never looked again took 0.253.  From 5/8 on the same; lists of small
// footprints (0.62 of the rows walked) stay below it.
constexpr int kDenseShareNum = 3, kDenseShareDen = 4;

// Whether a record's alpha-test ellipsoid reaches about that share of its
// brick's rows, from its half-widths along y and z through the mean:
// sigma log2(e) = h3 dy^2 (h5 dz^2) meets the test's limit there.
template <typename T>
__device__ __forceinline__ bool box_is_dense(const BwdRecord<T> &rec, const Brick &b) {
  const T limit = limit_as_value(rec.lim);
  const T hy = cull_sqrt(limit / rec.h[3]), hz = cull_sqrt(limit / rec.h[5]);
  const T zero = 0, eight = 8;
  const T y = rec.m[1] - static_cast<T>(b.oj), z = rec.m[2] - static_cast<T>(b.oi);
  const T ny = fmin(y + hy, eight) - fmax(y - hy, zero);
  const T nz = fmin(z + hz, eight) - fmax(z - hz, zero);
  return ny > zero && nz > zero && ny * nz * kDenseShareDen >= 64 * kDenseShareNum;
}

// Forward at brick size 8 with culled rows.  S waves per brick; lane =
// x-row (slice lane / 8, row lane % 8), its 8 voxels in registers.  Wave w
// takes the batches of 64 records w, w + S, w + 2S, ... of the brick's list
// (a list whose Gaussians differ in size along it is shared out evenly).
// Per batch, each lane loads one record and the rows it reaches
// (reach_mask); a 64 x 64 bit transpose hands each row's lane the set of
// batch records that reach that row; each lane then walks its own set in
// list order, so a record costs a row only where it can pass the alpha
// test, and the rows a record does not reach would only add exact zeros.
// With S = 1 every voxel sums its records in list order (the volume equals
// voxel_fwd_kernel's bit for bit); with S > 1 (long lists: the host picks S
// from the mean list length) the S partial bricks are added in wave order
// through LDS, a fixed order.  reach_out (optional): each record's reach
// mask, stored at its list position for a backward over the same lists.
template <typename T, int S>
__global__ __launch_bounds__(64 * S, sizeof(T) == 4 ? 1 : 3) void voxel_fwd_reach_kernel(
    const T *__restrict__ means3d, const T *__restrict__ conics, const T *__restrict__ opac,
    const int32_t *__restrict__ tile_offsets, const int32_t *__restrict__ flatten_ids,
    int64_t n_isects, uint32_t n_keys, uint32_t koff, int64_t N, uint32_t D2, uint32_t D1,
    uint32_t D0, uint32_t n2, uint32_t n1, T *__restrict__ volume,
    uint64_t *__restrict__ reach_out) {
  constexpr int R = 8;
  using V4 = typename Vec<T>::v4;
  // Per staged record {my, mz, o, h0}, {h1, h2, h3, h4}, {h5, limit bits,
  // 0, 0} and its eight column offsets dx_k = (x_k + 1/2) - mx, the same for
  // every row of the brick: five vector reads per use; the 20-word stride
  // spreads 8 consecutive records over all banks.
  __shared__ V4 s_rec[S][64][5];
  __shared__ T s_part[S > 1 ? S - 1 : 1][R][64];
  const uint32_t key = xcd_swizzle(blockIdx.x, n_keys);  // in the lists (koff: the grid's)
  const Brick b = brick_of(key + koff, n2, n1, R, D2, D1, D0);
  const int lane = static_cast<int>(lane_id());
  const int w = S > 1 ? static_cast<int>(wave_index()) : 0;
  const int li = lane >> 3, lj = lane & 7;
  const T half = static_cast<T>(0.5);
  const T py = static_cast<T>(b.oj + lj) + half;
  const T pz = static_cast<T>(b.oi + li) + half;
  const T px0 = static_cast<T>(b.ok) + half;
  const int64_t l0 = tile_offsets[key];
  const int64_t l1 = (key == n_keys - 1) ? n_isects : static_cast<int64_t>(tile_offsets[key + 1]);
  const int64_t start = l0 + 64 * w, end = l1;
  T acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) acc[k] = 0;
  // Adds batch record t to the lane's row.  The mask the alpha test restores
  // is the caller's (lanes whose set is exhausted stay off).
  const auto add_record = [&](int t, uint64_t exec) {
    const V4 qa = s_rec[w][t][0], qh = s_rec[w][t][1], qr = s_rec[w][t][2];
    const V4 q0 = s_rec[w][t][3], q1 = s_rec[w][t][4];
    const T dxs[R] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    const typename Bits<T>::type lim = bits_of(qr.y);
    const T dy = py - qa.x, dz = pz - qa.y;
    const T B = qh.x * dy + qh.y * dz;
    const T C = (qh.z * dy + qh.w * dz) * dy + qr.x * dz * dz;
    T sl[R], e[R];
#pragma unroll
    for (int k = 0; k < R; ++k) sl[k] = (qa.w * dxs[k] + B) * dxs[k] + C;
    neg_exp2_run(sl, e);
#pragma unroll
    for (int k = 0; k < R; ++k) add_passing(sl[k], e[k], lim, qa.z, acc[k], exec);
  };
  // The ids of the wave's next batch, loaded a batch ahead (one memory round
  // trip fewer before the records' own loads).
  int64_t idx = start + lane;
  int32_t next_id = idx < end ? flatten_ids[idx] : -1;
  bool all_rows = false;  // uniform: the batch before walked every row
  for (int64_t base = start; base < end; base += 64 * S) {
    const bool in = idx < end;
    const int64_t at = idx, g = in ? static_cast<int64_t>(next_id) : -1;
    idx += 64 * S;
    next_id = idx < end ? flatten_ids[idx] : -1;
    const int cnt = static_cast<int>(min(static_cast<int64_t>(64), end - base));
    BwdRecord<T> rec;
    uint64_t reach = 0;
    // Walking a row that a record does not reach adds exact zeros, so a dense
    // batch needs no masks; a caller that takes the masks needs every batch's.
    bool cull = true;
    if (all_rows && reach_out == nullptr) {
      load_bwd_record_plain(means3d, conics, opac, g, N, in, b, rec);
      cull = __popcll(ballot(rec.live && box_is_dense(rec, b))) * 2 < cnt;
    }
    if (cull) {
      load_bwd_record(means3d, conics, opac, g, N, in, b, rec);
      reach = rec.live ? reach_mask(rec, b, px0 - rec.m[0]) : 0ull;
      if (reach_out != nullptr && in) reach_out[at] = reach;
    }
    V4 a, hq, hr, d0, d1;
    a.x = rec.m[1];
    a.y = rec.m[2];
    a.z = rec.o;
    a.w = rec.h[0];
    hq.x = rec.h[1];
    hq.y = rec.h[2];
    hq.z = rec.h[3];
    hq.w = rec.h[4];
    hr.x = rec.h[5];
    hr.y = limit_as_value(rec.live ? rec.lim : static_cast<typename Bits<T>::type>(0));
    hr.z = 0;
    hr.w = 0;
    // The column offsets from the voxel centres x_k + 1/2 = px0 + k (exact),
    // computed once per record instead of once per walked row.
    T dxs[R];
#pragma unroll
    for (int k = 0; k < R; ++k) dxs[k] = (px0 + static_cast<T>(k)) - rec.m[0];
    d0.x = dxs[0];
    d0.y = dxs[1];
    d0.z = dxs[2];
    d0.w = dxs[3];
    d1.x = dxs[4];
    d1.y = dxs[5];
    d1.z = dxs[6];
    d1.w = dxs[7];
    // The wave's LDS operations complete in order: the fences keep the
    // compiler from moving this batch's writes above the previous batch's
    // reads, or the reads below above the writes.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    s_rec[w][lane][0] = a;
    s_rec[w][lane][1] = hq;
    s_rec[w][lane][2] = hr;
    s_rec[w][lane][3] = d0;
    s_rec[w][lane][4] = d1;
    // Walking every row in step costs about kDenseShare of walking each
    // row's own set, record for record (uniform reads, no set to step
    // through, no transpose).
    if (cull) all_rows = wave_sum(__popcll(reach)) * kDenseShareDen >= 64 * cnt * kDenseShareNum;
    uint64_t mine = 0;
    // Bit t of lane r's set: batch record t reaches row r.
    if (!all_rows) mine = transpose_bits64(reach, static_cast<uint32_t>(lane));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (all_rows) {
      const uint64_t exec = __builtin_amdgcn_read_exec();
#pragma unroll 1
      for (int t = 0; t < cnt; ++t) add_record(t, exec);
    } else {
      while (mine != 0ull) {
        const int t = static_cast<int>(__builtin_ctzll(mine));
        mine &= mine - 1ull;
        add_record(t, __builtin_amdgcn_read_exec());
      }
    }
  }
  if constexpr (S > 1) {
    // Waves 1 .. S-1 hand their partial bricks to wave 0, which adds them in
    // wave order.
    if (w > 0) {
#pragma unroll
      for (int k = 0; k < R; ++k) s_part[w - 1][k][lane] = acc[k];
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int ww = 0; ww < S - 1; ++ww) {
#pragma unroll
      for (int k = 0; k < R; ++k) acc[k] += s_part[ww][k][lane];
    }
  }
  if (li < b.ni && lj < b.nj) {
    T *out = volume + static_cast<int64_t>(b.oi + li) * D1 * D2 +
             static_cast<int64_t>(b.oj + lj) * D2 + b.ok;
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k < b.nk) out[k] = acc[k];
  }
}

// The whole brick of one record when every brick of the wave lies inside
// the volume (no column guard).  The column offsets dx_k are the same on
// every row and the column sums W_k = sum over rows of w accumulate per
// column, so T0, T1, T2 follow from W_k once per record and each voxel adds
// three sums (W_k, s0, s1) instead of four.  Rows the record does not reach
// test against a zero limit (every voxel fails), so the upstream
// gradient is loaded without masks.
// kReach: the slices' row ranges come from `reach` (bit 8 * slice + row of
// the reached rows, as voxel_bwd_chunk_kernel computes them) instead of
// slice_rows.  kRuns: a row's exps as one run (neg_exp2_run), where many
// waves share a SIMD.
// v: the gradient at the brick's first voxel, with the given slice and row
// strides; every row 16-byte aligned.
template <typename T, int R, bool kReach = false, bool kRuns = false>
__device__ __forceinline__ void voxel_brick_full(const BwdRecord<T> &rec, const Brick &b,
                                                 const T *__restrict__ v, int64_t plane,
                                                 uint32_t D2, T dx0, T &T0, T &T1, T &T2, T &Y0,
                                                 T &Z0, T &Y1, T &Z1, T &YY, T &YZ, T &ZZ,
                                                 uint64_t reach = 0) {
  using Q = typename Quad<T>::type;
  constexpr int kq = Quad<T>::n;
  T dxk[R], wk[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    dxk[k] = dx0 + static_cast<T>(k);
    wk[k] = 0;
  }
  const T half = static_cast<T>(0.5);
#pragma unroll 1
  for (int li = 0; li < R; ++li) {
    const int i = b.oi + li;
    const bool in_slice = rec.live && i >= rec.i0 && i <= rec.i1;
    if (ballot(in_slice) == 0) continue;
    const T dz = (static_cast<T>(i) + half) - rec.m[2];
    int j0, j1;
    if constexpr (kReach) {
      const uint32_t byte = static_cast<uint32_t>(reach >> (8 * li)) & 0xFFu;
      j0 = b.oj + static_cast<int>(__builtin_ctz(byte | 0x100u));
      j1 = j0 + __popc(byte) - 1;
    } else {
      slice_rows(rec, b, in_slice, dz, dx0, j0, j1);
    }
    const T h4dz = rec.h[4] * dz, h5dzz = rec.h[5] * dz * dz, Bz = rec.h[2] * dz;
    const T *__restrict__ vslice = v + static_cast<int64_t>(li) * plane;
#pragma unroll 1
    for (int lj = 0; lj < R; ++lj) {
      const int j = b.oj + lj;
      const bool in_row = j >= j0 && j <= j1;
      if (ballot(in_row) == 0) continue;
      const T dy = (static_cast<T>(j) + half) - rec.m[1];
      const T B = fma(rec.h[1], dy, Bz);
      const T C = fma(fma(rec.h[3], dy, h4dz), dy, h5dzz);
      const typename Bits<T>::type lim = in_row ? rec.lim : 0;
      const T *__restrict__ vrow = vslice + static_cast<int64_t>(lj) * D2;
      T vv[R];
#pragma unroll
      for (int q = 0; q < R / kq; ++q)
        *reinterpret_cast<Q *>(vv + q * kq) = *reinterpret_cast<const Q *>(vrow + q * kq);
      T s0 = 0, s1 = 0;
      // Explicit FMAs keep the row-invariant products of dx_k from being
      // hoisted into extra registers.
      T sl[R], e[R];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        sl[k] = fma(fma(rec.h[0], dxk[k], B), dxk[k], C);
        if (!kRuns) e[k] = neg_exp2(sl[k]);
      }
      if constexpr (kRuns) neg_exp2_run(sl, e);
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const T dx = dxk[k];
        const T p = vv[k] * e[k];  // unconditional, not a branch around the load and exp
        const T w = alpha_pass(sl[k], lim) ? p : static_cast<T>(0);
        wk[k] += w;
        s0 += w;
        s1 = fma(w, dx, s1);
      }
      const T dys0 = dy * s0, dzs0 = dz * s0;
      Y0 += dys0;
      Z0 += dzs0;
      YY += dy * dys0;
      YZ += dz * dys0;
      ZZ += dz * dzs0;
      Y1 += dy * s1;
      Z1 += dz * s1;
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const T wx = wk[k] * dxk[k];
    T0 += wk[k];
    T1 += wx;
    T2 += wx * dxk[k];
  }
}

// The rows of one record's brick with masked loads, for bricks of any size
// and extent (guard: voxel_row's kGuard, uniform per wave).
template <typename T, int R, bool kExact>
__device__ __forceinline__ void voxel_brick_rows(const BwdRecord<T> &rec, const Brick &b,
                                                 const T *__restrict__ v_vol, int64_t plane,
                                                 uint32_t D2, T dx0, int nts, bool vec, bool guard,
                                                 T &T0, T &T1, T &T2, T &Y0, T &Z0, T &Y1, T &Z1,
                                                 T &YY, T &YZ, T &ZZ) {
  const T half = static_cast<T>(0.5);
  // Rolled loops: unrolled, the slices and rows multiply the registers.
#pragma unroll 1
  for (int li = 0; li < R; ++li) {
    if (!kExact && li >= nts) break;
    const int i = b.oi + li;
    const bool in_slice = rec.live && i >= rec.i0 && i <= rec.i1;
    if (ballot(in_slice) == 0) continue;
    const T dz = (static_cast<T>(i) + half) - rec.m[2];
    // Rows of this slice the lane's ellipsoid can reach.
    int j0, j1;
    slice_rows(rec, b, in_slice, dz, dx0, j0, j1);
    const T h4dz = rec.h[4] * dz, h5dzz = rec.h[5] * dz * dz, Bz = rec.h[2] * dz;
#pragma unroll 1
    for (int lj = 0; lj < R; ++lj) {
      if (!kExact && lj >= nts) break;
      const int j = b.oj + lj;
      const bool in_row = j >= j0 && j <= j1;
      if (ballot(in_row) == 0) continue;
      const T dy = (static_cast<T>(j) + half) - rec.m[1];
      const T B = rec.h[1] * dy + Bz;
      const T C = (rec.h[3] * dy + h4dz) * dy + h5dzz;
      const T *__restrict__ vrow =
          v_vol +
          (in_row ? static_cast<int64_t>(i) * plane + static_cast<int64_t>(j) * D2 : 0) + b.ok;
      T vv[R];
      if (vec)
        load_grad_row<T, R, true>(vrow, in_row, b.nk, nts, vv);
      else
        load_grad_row<T, R, false>(vrow, in_row, b.nk, nts, vv);
      T s0 = 0, s1 = 0, s2 = 0;
      if (guard)
        voxel_row<T, R, kExact, true>(rec, vv, dx0, b.nk, nts, B, C, s0, s1, s2);
      else
        voxel_row<T, R, kExact, false>(rec, vv, dx0, b.nk, nts, B, C, s0, s1, s2);
      T0 += s0;
      T1 += s1;
      T2 += s2;
      const T dys0 = dy * s0, dzs0 = dz * s0;
      Y0 += dys0;
      Z0 += dzs0;
      YY += dy * dys0;
      YZ += dz * dys0;
      ZZ += dz * dzs0;
      Y1 += dy * s1;
      Z1 += dz * s1;
    }
  }
}

// Records in brick order (tile_offsets, flatten_ids; isect_ids optional),
// one lane per record.  kRows = false: each record's ten partials go out
// through global atomics.  kRows = true: they are stored as the row
// isect_src[r] of `rows` (see r2s_rows.h), zeros included.  kExact: the
// brick size equals R (loops fully unrolled); otherwise ts <= R at run time.
template <typename T, int R, bool kExact, bool kRows>
__global__ __launch_bounds__(kBwdThreads) void voxel_bwd_kernel(
    const T *__restrict__ means3d, const T *__restrict__ conics, const T *__restrict__ opac,
    const int32_t *__restrict__ tile_offsets, const int64_t *__restrict__ isect_ids,
    const int32_t *__restrict__ flatten_ids, const int32_t *__restrict__ isect_src,
    int64_t n_isects, uint32_t n_keys, uint32_t koff, int64_t N, const T *__restrict__ v_vol,
    uint32_t D2, uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, bool vec,
    T *__restrict__ v_means, T *__restrict__ v_conics, T *__restrict__ v_opac,
    T *__restrict__ rows) {
  // Consecutive blocks (neighbouring tiles, which share Gaussians) on one XCD.
  const int64_t rb =
      static_cast<int64_t>(xcd_swizzle(blockIdx.x, gridDim.x)) * kBwdThreads + 64 * wave_index();
  if (rb >= n_isects) return;  // uniform per wave
  const int64_t r = rb + lane_id();
  const bool in_list = r < n_isects;
  const int nts = kExact ? R : static_cast<int>(ts);
  uint32_t key;
  bool key_ok = in_list;
  // Issued with the key's load, not after its check (one memory round trip
  // fewer before the record's own loads).
  const int32_t fid = in_list ? flatten_ids[r] : -1;
  if (isect_ids != nullptr) {
    const int64_t k = in_list ? isect_ids[r] : 0;
    key_ok = key_ok && k >= 0 && k < static_cast<int64_t>(n_keys);
    key = key_ok ? static_cast<uint32_t>(k) : 0u;
  } else {
    key = wave_record_key(tile_offsets, n_keys, n_isects, rb, r);
  }
  const int64_t g = key_ok ? static_cast<int64_t>(fid) : -1;
  const Brick b = brick_of(key + koff, n2, n1, static_cast<uint32_t>(nts), D2, D1, D0);
  BwdRecord<T> rec;
  load_bwd_record(means3d, conics, opac, g, N, key_ok, b, rec);
  const T half = static_cast<T>(0.5);
  const T dx0 = (static_cast<T>(b.ok) + half) - rec.m[0];
  const int64_t plane = static_cast<int64_t>(D1) * D2;
  // Columns past the volume matter only for records whose sigma may be
  // non-finite (uniform over the wave).
  const bool guard = ballot(rec.live && !rec.cu.ok && b.nk < nts) != 0;
  T T0 = 0, T1 = 0, T2 = 0, Y0 = 0, Z0 = 0, Y1 = 0, Z1 = 0, YY = 0, YZ = 0, ZZ = 0;
  bool full = false;
  if constexpr (kExact && R % Quad<T>::n == 0)
    full = vec && ballot(b.ni < nts || b.nj < nts || b.nk < nts) == 0;
  if (full && ballot(rec.live) != 0) {
    voxel_brick_full<T, R>(rec, b, v_vol + b.oi * plane + static_cast<int64_t>(b.oj) * D2 + b.ok,
                           plane, D2, dx0, T0, T1, T2, Y0, Z0, Y1, Z1, YY, YZ, ZZ);
  } else if (ballot(rec.live) != 0) {
    voxel_brick_rows<T, R, kExact>(rec, b, v_vol, plane, D2, dx0, nts, vec, guard, T0, T1, T2, Y0,
                                   Z0, Y1, Z1, YY, YZ, ZZ);
  }
  if (!key_ok) return;
  // Per-voxel terms of VoxelizeToVoxelsBwd.cu:409-421 summed over the brick
  // (zero for dead records).
  const T o = rec.o;
  const T *q = rec.q;
  const T gx = o * (q[0] * T1 + q[1] * Y0 + q[2] * Z0);
  const T gy = o * (q[3] * Y0 + q[4] * Z0 + q[1] * T1);
  const T gz = o * (q[5] * Z0 + q[4] * Y0 + q[2] * T1);
  const T g0 = -half * o * T2, g1 = -o * Y1, g2 = -o * Z1;
  const T g3 = -half * o * YY, g4 = -o * YZ, g5 = -half * o * ZZ;
  const T go = T0;
  if (kRows) {
    const T v[10] = {gx, gy, gz, g0, g1, g2, g3, g4, g5, go};
    store_row(rows, isect_src[r], v);
    return;
  }
  if (!rec.live) return;
  if (gx == 0 && gy == 0 && gz == 0 && g0 == 0 && g1 == 0 && g2 == 0 && g3 == 0 && g4 == 0 &&
      g5 == 0 && go == 0)
    return;
  atomic_add(v_means + 3 * g, gx);
  atomic_add(v_means + 3 * g + 1, gy);
  atomic_add(v_means + 3 * g + 2, gz);
  atomic_add(v_conics + 6 * g, g0);
  atomic_add(v_conics + 6 * g + 1, g1);
  atomic_add(v_conics + 6 * g + 2, g2);
  atomic_add(v_conics + 6 * g + 3, g3);
  atomic_add(v_conics + 6 * g + 4, g4);
  atomic_add(v_conics + 6 * g + 5, g5);
  atomic_add(v_opac + g, go);
}

// The row of a record's ten partials: the per-voxel terms of
// VoxelizeToVoxelsBwd.cu:409-421 summed over the brick.
template <typename T>
__device__ __forceinline__ void store_partials(T *__restrict__ rows, int64_t e, T o,
                                               const T (&q)[6], T T0, T T1, T T2, T Y0, T Z0,
                                               T Y1, T Z1, T YY, T YZ, T ZZ) {
  const T half = static_cast<T>(0.5);
  const T v[10] = {o * (q[0] * T1 + q[1] * Y0 + q[2] * Z0),
                   o * (q[3] * Y0 + q[4] * Z0 + q[1] * T1),
                   o * (q[5] * Z0 + q[4] * Y0 + q[2] * T1),
                   -half * o * T2,
                   -o * Y1,
                   -o * Z1,
                   -half * o * YY,
                   -o * YZ,
                   -half * o * ZZ,
                   T0};
  store_row(rows, e, v);
}

// One record's sums over the voxels of its brick inside the volume, one
// voxel at a time (rare: see voxel_bwd_chunk_kernel's `apart`).
// The record is loaded again, so that it need not stay in registers.
template <typename T>
__device__ __forceinline__ void voxel_sums_apart(const T *__restrict__ means3d,
                                                 const T *__restrict__ conics,
                                                 const T *__restrict__ opac, int64_t g, int64_t N,
                                                 const Brick &b, const T *__restrict__ v_vol,
                                                 int64_t plane, uint32_t D2, T &T0, T &T1, T &T2,
                                                 T &Y0, T &Z0, T &Y1, T &Z1, T &YY, T &YZ, T &ZZ) {
  const T half = static_cast<T>(0.5);
  BwdRecord<T> rec;
  load_bwd_record_plain(means3d, conics, opac, g, N, true, b, rec);
  const T dx0 = (static_cast<T>(b.ok) + half) - rec.m[0];
#pragma unroll 1
  for (int q = 0; q < b.ni * b.nj * b.nk; ++q) {
    const int k = q % b.nk, j = b.oj + q / b.nk % b.nj, i = b.oi + q / b.nk / b.nj;
    const T dx = dx0 + static_cast<T>(k);
    const T dy = (static_cast<T>(j) + half) - rec.m[1];
    const T dz = (static_cast<T>(i) + half) - rec.m[2];
    const T B = fma(rec.h[1], dy, rec.h[2] * dz);
    const T C = fma(fma(rec.h[3], dy, rec.h[4] * dz), dy, rec.h[5] * dz * dz);
    const T sl = fma(fma(rec.h[0], dx, B), dx, C);
    if (!alpha_pass(sl, rec.lim)) continue;
    const T w = v_vol[i * plane + static_cast<int64_t>(j) * D2 + b.ok + k] * neg_exp2(sl);
    T0 += w;
    T1 = fma(w, dx, T1);
    T2 = fma(w * dx, dx, T2);
    Y0 = fma(w, dy, Y0);
    Z0 = fma(w, dz, Z0);
    Y1 = fma(w * dx, dy, Y1);
    Z1 = fma(w * dx, dz, Z1);
    YY = fma(w * dy, dy, YY);
    YZ = fma(w * dy, dz, YZ);
    ZZ = fma(w * dz, dz, ZZ);
  }
}

// ------------------------------------------- chunked backward (rows) ---
//
// A wave of 64 records walks the union of its lanes' reached rows, which is
// nearly always every row of the brick, while one record's culled
// ellipsoid reaches about 57 % of them at config 3.  This form lists, per
// wave, the (record, slice, row) items the records reach -- slice by slice,
// row by row, as slice_rows gives them -- and hands them out in chunks of up
// to kChunkRows consecutive items of one record, one chunk per lane and
// round, so lanes spend their steps on reached rows.  The full chunks come
// first, ordered by (chunk index within the record, record), then each
// record's short last chunk, longest first; a round takes as many steps as
// its first (longest) chunk.  Within a round each record appears at most
// once per chunk index, and the chunk sums are added to the record's LDS
// accumulators one chunk index at a time in increasing order, so each
// record's chunks add in index order and the result does not depend on
// scheduling.
//
// The lanes of a step read the gradient rows of different records: loaded
// from memory, 64 lanes times 32 bytes through the vector cache's return path
// each step, that path was busy 92-98 % of the kernel's time.  Staged
// (kStage), a block therefore keeps its bricks' gradients in LDS when its
// records lie in at most kStageBricks consecutive bricks, zero beyond the
// volume, so that ragged volumes walk like any other; a block over more
// bricks reads rows from memory, element by element at the volume's ragged
// ends.  Six bricks and the other arrays take 28 KB, which with 96 VGPRs and
// no scratch keeps five waves per SIMD: 0.484 -> 0.469 ms for 3.2 M records
// of a 256^3 volume (0.426 -> 0.388 given masks), 22.9 -> 21.9 ms for 252 M
// of a 512^3 one (21.3 -> 19.1), 0.231 -> 0.149 ms for 1.0 M of a
// 250 x 201 x 173 one beside the masked walk.  The records' fields reach the
// lanes that walk them by lane shuffles from the registers of the lanes that
// loaded them; staged in LDS (39 KB, four waves) the rows pass took longer.
// Unstaged, for short lists of whole volumes (stage_bricks), the records'
// fields go through LDS and every row comes from memory: 80 VGPRs, 27 KB, six
// waves per SIMD, no barrier.  Its exps stay with their voxels: where few
// waves run, runs of them (neg_exp2_run) only delay the sums after them.

constexpr int kChunkRows = 8;
constexpr int kChunkWaves = 4;
constexpr uint32_t kStageBricks = 6;
// A chunked item costs about 1.3 times a row of the dense walk (indexing,
// the walk, the chunk sums), so a wave whose records reach more than this
// many of their 64 x 64 (record, row) pairs takes the dense walk instead
// (large footprints, e.g. the binary-tree model on a 128^3 volume).
constexpr int kDenseItems = 3072;

__device__ __forceinline__ uint32_t shfl_bits(uint32_t v, int src) {
  return static_cast<uint32_t>(__shfl(static_cast<int>(v), src, 64));
}
__device__ __forceinline__ uint64_t shfl_bits(uint64_t v, int src) {
  return static_cast<uint64_t>(__shfl(static_cast<long long>(v), src, 64));
}

// Chunks of one wave of 64 records of at most 64 rows, in chunks of up to
// kChunkRows.  Where every brick can be read whole, a wave over kDenseItems
// takes the dense walk, and below it has at most one short chunk per record
// beside the full ones (27 KB of LDS, six blocks per CU); staged blocks are
// not the only ones of the staged form, so no smaller bound holds there.
template <bool kStage>
constexpr int kMaxChunks = kStage ? 64 * (64 / kChunkRows) : kDenseItems / kChunkRows + 64;

// Whether a list's backward stages its bricks' gradients (kStage).  Blocks
// whose records lie in too many bricks for it read memory through the general
// code of the staged form, which is slower than the unstaged kernels, so the
// line lies where most blocks stage.
// Ragged volumes, whose other form is voxel_bwd_kernel's masked walk: from
// 256 records per kStageBricks bricks on, the least that fills a block.  At
// 37 records per brick of 250 x 201 x 173 the staged form takes 173 us and
// the masked walk 168, at 54 147 and 230; of 90 x 61 x 77 at 41 36 and 36, at
// 104 22 and 42.
// Whole volumes, whose other form is the unstaged chunked walk: from 64
// records per brick on.  Of 256 x 200 x 176 at 25 records 99 and 81 us, at 56
// 140 and 130 (given masks 128 and 120), of 256^3 at 97 470 and 461 (given
// masks 385 and 420), of 512^3 at 960 22.0 and 22.4 ms (19.2 and 21.0).
// Lists of less than a block per CU wait for the staging's two barriers alone:
// 9k records of a 32^3 volume, 29 and 26 us.  In double the staged form has
// two waves per SIMD instead of three: 1.22 and 1.17 ms at 256^3 without
// masks.
template <typename T>
inline bool stage_bricks(int64_t n_isects, int64_t n_keys, bool whole) {
  if (!whole) return n_isects * kStageBricks >= 64 * kChunkWaves * n_keys;
  return sizeof(T) == 4 && n_isects >= 64 * n_keys && n_isects >= 64 * kChunkWaves * 256;
}

// A record as the lanes that walk it read it from LDS (unstaged form).
template <typename T>
struct ChunkRecord {
  T c[3];  // the brick's first voxel centre minus the mean (x, y, z)
  T h[6];
  typename Bits<T>::type lim;  // 0 for dead records
  uint32_t brick0;             // byte offset of the brick's first voxel in v_vol
};

// kGiven: each record's reach mask comes from `reach` (stored by the forward
// over the same lists, voxel_fwd_reach_kernel) instead of the culling
// setup and the per-slice row ranges.
template <typename T, bool kGiven, bool kStage>
__global__ __launch_bounds__(64 * kChunkWaves, sizeof(T) == 4 ? (kStage ? 5 : 6) : 1)
void voxel_bwd_chunk_kernel(
    const T *__restrict__ means3d, const T *__restrict__ conics, const T *__restrict__ opac,
    const int32_t *__restrict__ tile_offsets, const int64_t *__restrict__ isect_ids,
    const int32_t *__restrict__ flatten_ids, const int32_t *__restrict__ isect_src,
    int64_t n_isects, uint32_t n_keys, uint32_t koff, int64_t N, const T *__restrict__ v_vol,
    uint32_t D2, uint32_t D1, uint32_t D0, uint32_t n2, uint32_t n1, bool vec,
    T *__restrict__ rows, const uint64_t *__restrict__ reach) {
  constexpr int R = kChunkRows;
  constexpr uint32_t kBrick = R * R * R;
  constexpr int kRun = kStage ? R / 2 : 1;  // voxels per run of exps
  using Q = typename Quad<T>::type;
  constexpr int kq = Quad<T>::n;
  __shared__ uint64_t s_rows[kChunkWaves][64];  // reached rows: bit 8 * slice + row
  __shared__ T s_acc[kChunkWaves][10][64];
  // Chunk entries: record lane | first row << 6 | chunk index << 12.
  __shared__ uint16_t s_chunk[kChunkWaves][kMaxChunks<kStage>];
  __shared__ uint32_t s_key_min[kChunkWaves], s_key_max[kChunkWaves];
  __shared__ WordMajor<ChunkRecord<T>, 64> s_rec[kStage ? 1 : kChunkWaves];
  __shared__ __align__(16) T s_v[kStage ? kStageBricks * kBrick : 1];
  const uint32_t w = wave_index(), lane = lane_id();
  // Positions in the list fit 32 bits: n_isects < 2^31 (the caller checks).
  const uint32_t rb = xcd_swizzle(blockIdx.x, gridDim.x) * (64 * kChunkWaves) + 64 * w;
  const uint32_t r = rb + lane;
  const bool in_list = r < n_isects;
  uint32_t key;
  bool key_ok = in_list;
  // Issued with the key's load, not after its check (one memory round trip
  // fewer before the record's own loads).
  const int32_t fid = in_list ? flatten_ids[r] : -1;
  const uint64_t reach_r = kGiven && in_list ? reach[r] : 0ull;
  if (rb >= n_isects) {  // uniform per wave: no records, only its share of the staging
    if constexpr (!kStage) return;
    key_ok = false;
    key = 0;
  } else if (isect_ids != nullptr) {
    const int64_t k = in_list ? isect_ids[r] : 0;
    key_ok = key_ok && k >= 0 && k < static_cast<int64_t>(n_keys);
    key = key_ok ? static_cast<uint32_t>(k) : 0u;
  } else {
    key = wave_record_key(tile_offsets, n_keys, n_isects, rb, r);
  }
  if (!key_ok) key = 0;
  const int64_t plane = static_cast<int64_t>(D1) * D2;
  const int64_t g = key_ok ? static_cast<int64_t>(fid) : -1;
  const Brick b = brick_of(key + koff, n2, n1, R, D2, D1, D0);
  BwdRecord<T> rec;
  if constexpr (kGiven)
    load_bwd_record_plain(means3d, conics, opac, g, N, key_ok, b, rec);
  else
    load_bwd_record(means3d, conics, opac, g, N, key_ok, b, rec);
  // A record whose sigma may be NaN passes the alpha test there whatever the
  // gradient: in a ragged brick, where the walk below also evaluates columns
  // beyond the volume, it is summed apart, voxel by voxel.
  const bool apart = kStage && rec.live && rec.lim == Bits<T>::kSign &&
                     (b.ni < R || b.nj < R || b.nk < R);
  if (apart) rec.live = false;
  const T half = static_cast<T>(0.5);
  const T dx0 = (static_cast<T>(b.ok) + half) - rec.m[0];

  // The record's reached rows; the items are its set bits in increasing order.
  uint64_t reached;
  if constexpr (kGiven)
    reached = key_ok && rec.live ? reach_r : 0ull;
  else
    reached = reach_mask(rec, b, dx0);
  const int n_items = __popcll(reached);
  const bool used = reached != 0 || apart;
  // Staged: the bricks of the block's records that reach a row.  In lists of
  // long thin Gaussians' boxes most records reach none, and a wave of such
  // records is done here: 7.5 G records of a 512^3 volume with 5 % needles take
  // 515 ms, with every block staged and every record loaded again 707 (513 in
  // the unstaged form).
  bool staged = false;
  uint32_t key0 = 0;
  if constexpr (kStage) {
    const uint32_t k_min = wave_min(reached != 0 ? key : 0xffffffffu);
    const uint32_t k_max = wave_max(reached != 0 ? key : 0u);
    if (lane == 0) {
      s_key_min[w] = k_min;
      s_key_max[w] = k_max;
    }
    __syncthreads();
    key0 = s_key_min[0];
    uint32_t key1 = s_key_max[0];
#pragma unroll
    for (uint32_t ww = 1; ww < kChunkWaves; ++ww) {
      key0 = min(key0, s_key_min[ww]);
      key1 = max(key1, s_key_max[ww]);
    }
    staged = key0 <= key1 && key1 - key0 < kStageBricks;  // uniform over the block
    if (staged) {
      for (uint32_t k = key0; k <= key1; ++k) {
        const Brick sb = brick_of(k + koff, n2, n1, R, D2, D1, D0);
        const T *__restrict__ src = v_vol + sb.oi * plane + static_cast<int64_t>(sb.oj) * D2 + sb.ok;
#pragma unroll
        for (uint32_t h = 0; h < kBrick; h += 64 * kChunkWaves) {
          const int q = static_cast<int>(h + threadIdx.x);
          const int i = q >> 6, j = (q >> 3) & 7, c = q & 7;
          s_v[(k - key0) * kBrick + static_cast<uint32_t>(q)] =
              (i < sb.ni && j < sb.nj && c < sb.nk) ? src[i * plane + static_cast<int64_t>(j) * D2 + c]
                                                    : static_cast<T>(0);
        }
      }
      __syncthreads();
    }
    if (rb >= n_isects) return;  // uniform per wave; no barrier follows
  }
  // The row of the lane's record from its sums over the walked rows.  Staged,
  // the record's opacity and conic and every address are loaded or formed
  // again rather than kept in registers through the walk; a record that
  // reaches no row has a zero row and is not loaded again.
  const auto finish = [&](T T0, T T1, T T2, T Y0, T Z0, T Y1, T Z1, T YY, T YZ, T ZZ) {
    if (!key_ok) return;
    if constexpr (kStage) {
      uint32_t at = r, of = key;
      asm volatile("" : "+v"(at), "+v"(of));  // what they give is formed here
      const int64_t gauss = flatten_ids[at];
      if (apart)
        voxel_sums_apart(means3d, conics, opac, gauss, N,
                         brick_of(of + koff, n2, n1, R, D2, D1, D0), v_vol, plane, D2, T0, T1, T2,
                         Y0, Z0, Y1, Z1, YY, YZ, ZZ);
      T o = 0, q[6] = {0, 0, 0, 0, 0, 0};
      if (used) {
        o = opac[gauss];
#pragma unroll
        for (int c = 0; c < 6; ++c) q[c] = conics[6 * gauss + c];
      }
      store_partials(rows, isect_src[at], o, q, T0, T1, T2, Y0, Z0, Y1, Z1, YY, YZ, ZZ);
    } else {
      store_partials(rows, isect_src[r], rec.o, rec.q, T0, T1, T2, Y0, Z0, Y1, Z1, YY, YZ, ZZ);
    }
  };

  if constexpr (kStage) {
    if (ballot(reached != 0) == 0) {  // uniform per wave
      finish(0, 0, 0, 0, 0, 0, 0, 0, 0, 0);
      return;
    }
  }
  // Whole bricks with 16-byte rows: a row is read as vectors.
  const bool whole =
      !kStage || staged || (vec && ballot(b.ni < R || b.nj < R || b.nk < R) == 0);
  if (whole && wave_sum(n_items) > kDenseItems) {  // uniform per wave
    T T0 = 0, T1 = 0, T2 = 0, Y0 = 0, Z0 = 0, Y1 = 0, Z1 = 0, YY = 0, YZ = 0, ZZ = 0;
    if (ballot(rec.live) != 0) {
      if (kStage && staged)
        voxel_brick_full<T, R, true, kStage>(
            rec, b, s_v + (reached != 0 ? key - key0 : 0u) * kBrick, R * R, R, dx0, T0, T1, T2,
            Y0, Z0, Y1, Z1, YY, YZ, ZZ, reached);
      else
        voxel_brick_full<T, R, true, kStage>(
            rec, b, v_vol + b.oi * plane + static_cast<int64_t>(b.oj) * D2 + b.ok, plane, D2, dx0,
            T0, T1, T2, Y0, Z0, Y1, Z1, YY, YZ, ZZ, reached);
    }
    finish(T0, T1, T2, Y0, Z0, Y1, Z1, YY, YZ, ZZ);
    return;
  }
  // The brick's first voxel centre minus the mean.
  const T c1 = (static_cast<T>(b.oj) + half) - rec.m[1];
  const T c2 = (static_cast<T>(b.oi) + half) - rec.m[2];
  const typename Bits<T>::type my_lim = rec.live ? rec.lim : 0;
  s_rows[w][lane] = reached;
  if constexpr (!kStage) {
    ChunkRecord<T> cr;
    cr.c[0] = dx0;
    cr.c[1] = c1;
    cr.c[2] = c2;
#pragma unroll
    for (int c = 0; c < 6; ++c) cr.h[c] = rec.h[c];
    cr.lim = my_lim;
    // Below 2^32: the caller checks the volume's bytes.
    cr.brick0 = ((static_cast<uint32_t>(b.oi) * D1 + static_cast<uint32_t>(b.oj)) * D2 +
                 static_cast<uint32_t>(b.ok)) * static_cast<uint32_t>(sizeof(T));
    s_rec[w].store(static_cast<int>(lane), cr);
  }
#pragma unroll
  for (int c = 0; c < 10; ++c) s_acc[w][c][lane] = 0;
  // Chunk list: the full chunks in (chunk index, record) order, then each
  // record's short last chunk, longest first, so that the rounds of short
  // chunks take as many steps as their longest.  Each record's chunks keep
  // increasing chunk indices.  Byte li of pref: the reached rows of the
  // slices before li (0..56).
  uint64_t pref = 0;
  {
    uint32_t run = 0;
#pragma unroll
    for (int li = 0; li < R; ++li) {
      pref |= static_cast<uint64_t>(run) << (8 * li);
      run += static_cast<uint32_t>(__popc(static_cast<uint32_t>(reached >> (8 * li)) & 0xFFu));
    }
  }
  // The chunk's first row, the t-th set bit (t = 8 q): its slice li is the
  // last whose byte of pref is <= t, found for all eight bytes at once (each
  // byte | 0x80, minus t + 1, keeps its high bit exactly when the byte
  // exceeds t); within a slice the reached rows are contiguous.
  auto entry = [&](uint32_t q) {
    const uint32_t t = q * static_cast<uint32_t>(R);
    constexpr uint64_t kHigh = 0x8080808080808080ull, kOnes = 0x0101010101010101ull;
    const uint64_t above = ((pref | kHigh) - static_cast<uint64_t>(t + 1u) * kOnes) & kHigh;
    const int li = 7 - __popcll(above);
    const uint32_t byte = static_cast<uint32_t>(reached >> (8 * li)) & 0xFFu;
    const uint32_t before = static_cast<uint32_t>(pref >> (8 * li)) & 0xFFu;
    const uint32_t first =
        8u * static_cast<uint32_t>(li) + __builtin_ctz(byte | 0x100u) + (t - before);
    return static_cast<uint16_t>(lane | (first << 6) | (q << 12));
  };
  const int n_full = n_items / R, tail = n_items - n_full * R;
  uint32_t n_list = 0;
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const bool has = n_full > q;
    const uint64_t m = ballot(has);
    if (has)
      s_chunk[w][n_list + static_cast<uint32_t>(__popcll(m & lt))] =
          entry(static_cast<uint32_t>(q));
    n_list += static_cast<uint32_t>(__popcll(m));
  }
#pragma unroll
  for (int len = R - 1; len > 0; --len) {
    const bool has = tail == len;
    const uint64_t m = ballot(has);
    if (has)
      s_chunk[w][n_list + static_cast<uint32_t>(__popcll(m & lt))] =
          entry(static_cast<uint32_t>(n_full));
    n_list += static_cast<uint32_t>(__popcll(m));
  }
  // The wave's LDS operations complete in order, so its own lanes' writes
  // are visible to the reads below; keep the compiler from moving them.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // The two forms apart: the registers of one are not held through the other.
  const auto walk = [&](auto staged_tag) {
    constexpr bool kStaged = decltype(staged_tag)::value;
#pragma unroll 1
    for (uint32_t cb = 0; cb < n_list; cb += 64) {
      const uint32_t ci = cb + lane;
      const bool act = ci < n_list;
      const uint32_t ent = act ? static_cast<uint32_t>(s_chunk[w][ci]) : 0u;
      const uint32_t rl = ent & 63u, pos = (ent >> 6) & 63u, q = ent >> 12;
      T hr[6], cx, cy, cz;
      typename Bits<T>::type r_lim;
      uint32_t at0 = 0, r_key = 0;
      if constexpr (kStage) {
        // The record, from the registers of the lane that loaded it (every
        // lane takes part); the conic scaled as scaled_conic does.
        const int src = static_cast<int>(rl);
        T qr[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) qr[c] = __shfl(rec.q[c], src, 64);
        scaled_conic(qr, hr);
        cx = __shfl(dx0, src, 64);
        cy = __shfl(c1, src, 64);
        cz = __shfl(c2, src, 64);
        r_lim = shfl_bits(my_lim, src);
        r_key = static_cast<uint32_t>(__shfl(static_cast<int>(key), src, 64));
      } else {
        const ChunkRecord<T> cr = s_rec[w].load(static_cast<int>(rl));
#pragma unroll
        for (int c = 0; c < 6; ++c) hr[c] = cr.h[c];
        cx = cr.c[0];
        cy = cr.c[1];
        cz = cr.c[2];
        r_lim = cr.lim;
        at0 = cr.brick0;
      }
      const uint64_t rows_m = s_rows[w][rl];
      const int n_here =
          act ? min(R, __popcll(rows_m) - static_cast<int>(q) * R) : 0;
      // The record's rows from the chunk's first on: the chunk's items are
      // its n_here lowest set bits.
      uint64_t rest = act ? rows_m & (~0ull << pos) : 0ull;
      T dxk[R], wk[R];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        dxk[k] = cx + static_cast<T>(k);
        wk[k] = 0;
      }
      // The brick's gradient: staged, or in the volume.
      const T *__restrict__ vb = v_vol;
      int nk = R;
      if constexpr (kStaged) {
        at0 = rows_m != 0 ? (r_key - key0) * kBrick : 0u;
      } else if constexpr (kStage) {
        const Brick bb = brick_of(r_key + koff, n2, n1, R, D2, D1, D0);
        vb += bb.oi * plane + static_cast<int64_t>(bb.oj) * D2 + bb.ok;
        nk = bb.nk;
      }
      T Y0 = 0, Z0 = 0, Y1 = 0, Z1 = 0, YY = 0, YZ = 0, ZZ = 0;
      // The round's longest chunk is its first (lane 0 is always active).
      const int steps = __builtin_amdgcn_readfirstlane(n_here);
#pragma unroll 1
      for (int st = 0; st < steps; ++st) {
        const bool item = st < n_here;
        // The next row (bit 63 when none is left: a step without an item
        // still reads a row of the record's own brick and tests against a zero
        // limit).
        const uint32_t p = static_cast<uint32_t>(__builtin_ctzll(rest | (1ull << 63)));
        rest &= rest - 1ull;
        const uint32_t li = p >> 3, lj = p & 7u;
        // The row centre's offsets from the mean as the columns' (dxk): the
        // brick corner's offset plus the row's index in the brick.
        const T dz = static_cast<T>(li) + cz;
        const T dy = static_cast<T>(lj) + cy;
        const T B = fma(hr[1], dy, hr[2] * dz);
        const T C = fma(fma(hr[3], dy, hr[4] * dz), dy, hr[5] * dz * dz);
        typename Bits<T>::type lim = item ? r_lim : 0;
        if constexpr (kStage) asm volatile("" : "+v"(lim));  // one select, not an AND per voxel
        T vv[R];
        if constexpr (kStaged) {
          const T *vrow = s_v + (at0 + p * R);
#pragma unroll
          for (int c = 0; c < R / kq; ++c)
            *reinterpret_cast<Q *>(vv + c * kq) = *reinterpret_cast<const Q *>(vrow + c * kq);
        } else {
          const T *__restrict__ vrow;
          if constexpr (kStage) {
            vrow = vb + (li * plane + static_cast<int64_t>(lj) * D2);
          } else {
            // Two full-rate multiply-adds: li, lj < 8 and the strides in bytes
            // below 2^24 (the caller checks).
            uint32_t at = __umul24(lj, D2 * static_cast<uint32_t>(sizeof(T))) + at0;
            asm volatile("" : "+v"(at));  // not two products and a sum
            at += __umul24(li, D1 * D2 * static_cast<uint32_t>(sizeof(T)));
            vrow = reinterpret_cast<const T *>(reinterpret_cast<const char *>(v_vol) + at);
          }
          if (!kStage || whole) {
#pragma unroll
            for (int c = 0; c < R / kq; ++c)
              *reinterpret_cast<Q *>(vv + c * kq) = *reinterpret_cast<const Q *>(vrow + c * kq);
          } else {
            // Columns beyond the volume read zero; the rows and slices beyond
            // it are reached by no record, only by a step without an item.
            const int n = item ? nk : 0;
#pragma unroll
            for (int k = 0; k < R; ++k) vv[k] = k < n ? vrow[k] : static_cast<T>(0);
          }
        }
        T s0 = 0, s1 = 0;
#pragma unroll
        for (int h = 0; h < R; h += kRun) {
          T sl[kRun], e[kRun];
#pragma unroll
          for (int k = 0; k < kRun; ++k)
            sl[k] = fma(fma(hr[0], dxk[h + k], B), dxk[h + k], C);
          if constexpr (kRun > 1)
            neg_exp2_run(sl, e);
          else
            e[0] = neg_exp2(sl[0]);
#pragma unroll
          for (int k = 0; k < kRun; ++k) {
            // A failing voxel adds an exact zero whatever its upstream gradient
            // (a non-finite one included), as when the voxel is skipped.  The
            // product is formed unconditionally: as an operand of the
            // conditional it would become a branch around its load and exp.
            const T p = vv[h + k] * e[k];
            const T wv = alpha_pass(sl[k], lim) ? p : static_cast<T>(0);
            wk[h + k] += wv;
            s0 += wv;
            s1 = fma(wv, dxk[h + k], s1);
          }
        }
        const T dys0 = dy * s0, dzs0 = dz * s0;
        Y0 += dys0;
        Z0 += dzs0;
        YY = fma(dy, dys0, YY);
        YZ = fma(dz, dys0, YZ);
        ZZ = fma(dz, dzs0, ZZ);
        Y1 = fma(dy, s1, Y1);
        Z1 = fma(dz, s1, Z1);
      }
      T t0 = 0, t1 = 0, t2 = 0;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const T wx = wk[k] * dxk[k];
        t0 += wk[k];
        t1 += wx;
        t2 += wx * dxk[k];
      }
      const T sums[10] = {t0, t1, t2, Y0, Z0, Y1, Z1, YY, YZ, ZZ};
      // One chunk index at a time, in increasing order: the records of one
      // index are distinct, and each record's chunks are added in index order.
      uint32_t qmask = 0;
#pragma unroll
      for (int b = 0; b < R; ++b)
        if (ballot(act && q == static_cast<uint32_t>(b)) != 0) qmask |= 1u << b;
#pragma unroll 1
      for (uint32_t mq = qmask; mq != 0u; mq &= mq - 1u) {
        const uint32_t qq = static_cast<uint32_t>(__builtin_ctz(mq));
        if (act && q == qq) {
#pragma unroll
          for (int c = 0; c < 10; ++c) s_acc[w][c][rl] += sums[c];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
  };
  if (kStage && staged)
    walk(std::true_type{});
  else
    walk(std::false_type{});
  T a[10];
#pragma unroll
  for (int c = 0; c < 10; ++c) a[c] = s_acc[w][c][lane];
  finish(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9]);
}

// n0 brick layers of lists from layer z0 on (the whole grid: z0 = 0 and
// n0 ts >= D0; a z-slab: z0 + n0 layers within the grid).
int check_voxel_args(int64_t n_isects, int64_t N, uint32_t D2, uint32_t D1, uint32_t D0,
                     uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0, const char *name,
                     uint32_t z0 = 0, bool slab = false) {
  R2S_REQUIRE(N >= 0 && N <= kInt32Max, "%s: bad size N=%lld", name, (long long)N);
  // ts <= 10 first: ts^3 in 32 bits wraps for ts >= 1626.
  R2S_REQUIRE(ts > 0 && ts <= 10 && ts * ts * ts <= 1024,
              "%s: tile_size must be positive with tile_size**3 <= 1024", name);
  R2S_REQUIRE(n_isects >= 0 && n_isects <= kInt32Max, "%s: bad n_isects", name);
  R2S_REQUIRE(static_cast<uint64_t>(n2) * ts >= D2 && static_cast<uint64_t>(n1) * ts >= D1 &&
                  (slab || static_cast<uint64_t>(n0) * ts >= D0),
              "%s: brick grid does not cover the volume", name);
  R2S_REQUIRE(!slab || (static_cast<uint64_t>(z0) + n0) * ts < static_cast<uint64_t>(D0) + ts,
              "%s: brick layers [%u, %u) outside the volume", name, z0, z0 + n0);
  R2S_REQUIRE(static_cast<uint64_t>(n2) * ts <= 0x7fffffffull &&
                  static_cast<uint64_t>(n1) * ts <= 0x7fffffffull &&
                  static_cast<uint64_t>(n0) * ts <= 0x7fffffffull,
              "%s: brick grid too large", name);
  R2S_REQUIRE(static_cast<uint64_t>(n2) * n1 * (static_cast<uint64_t>(z0) + n0) <=
                  0x7fffffffull,
              "%s: too many bricks", name);
  return R2S_OK;
}

template <typename T>
void launch_voxel_fwd(const T *means3d, const T *conics, const T *opac,
                      const int32_t *tile_offsets, const int32_t *flatten_ids, int64_t n_isects,
                      uint32_t n_keys, uint32_t koff, int64_t N, uint32_t D2, uint32_t D1,
                      uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, T *volume,
                      hipStream_t stream) {
  const uint32_t nt = ts * ts * ts;
  const size_t smem =
      min(nt, kFwdBatch) * (3 * sizeof(typename Vec<T>::v4));
  voxel_fwd_kernel<T><<<dim3(n_keys), dim3(nt), smem, stream>>>(
      means3d, conics, opac, tile_offsets, flatten_ids, n_isects, n_keys, koff, N, D2, D1, D0, ts,
      n2, n1, volume);
}

// slab: the lists are those of brick layers [z0, z0 + n0) (keys relative to
// layer z0) and only that z-range of the whole volume is written.
template <typename T>
int voxel_fwd_impl(const T *means3d, const T *conics, const T *opac,
                   const int32_t *tile_offsets, const int32_t *flatten_ids, int64_t n_isects,
                   int64_t N, uint32_t D2, uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2,
                   uint32_t n1, uint32_t n0, T *volume, r2s_stream_t st, uint32_t z0 = 0,
                   bool slab = false, uint64_t *reach = nullptr) {
  clear_error();
  const char *name = "voxelize_to_voxels_fwd";
  R2S_RETURN_IF(check_voxel_args(n_isects, N, D2, D1, D0, ts, n2, n1, n0, name, z0, slab));
  R2S_REQUIRE(reach == nullptr || ts == 8, "%s: reach masks need tile_size 8", name);
  // Voxel slices [i0, i1) of the layers' z-range.
  const int64_t i0 = static_cast<int64_t>(z0) * ts;
  const int64_t i1 = slab ? std::min<int64_t>(static_cast<int64_t>(z0 + n0) * ts, D0) : D0;
  const int64_t plane = static_cast<int64_t>(D2) * D1;
  const int64_t n_vox = plane * (i1 - i0);
  if (n_vox <= 0) return R2S_OK;
  R2S_REQUIRE(volume != nullptr, "%s: null volume", name);
  hipStream_t stream = as_stream(st);
  if (N == 0 || n_isects == 0)
    return device_fill<T>(volume + i0 * plane, n_vox, static_cast<T>(0), stream, name);
  R2S_REQUIRE(means3d && conics && opac && tile_offsets && flatten_ids, "%s: null pointer", name);
  const uint32_t n_keys = n2 * n1 * n0, koff = z0 * n1 * n2;
  if (ts == 8) {
    // Waves per brick from the mean list length: one up to 192 records (3
    // batches), then 2, then 4 from 384, so that long lists (large
    // footprints, few bricks) are shared out.
    const int64_t per_brick = n_isects / n_keys;
    const dim3 grid(n_keys);
#define R2S_VOXEL_FWD_REACH(S)                                                                  \
  voxel_fwd_reach_kernel<T, S><<<grid, dim3(64 * S), 0, stream>>>(                              \
      means3d, conics, opac, tile_offsets, flatten_ids, n_isects, n_keys, koff, N, D2, D1, D0,  \
      n2, n1, volume, reach)
    if (per_brick < 192)
      R2S_VOXEL_FWD_REACH(1);
    else if (per_brick < 384)
      R2S_VOXEL_FWD_REACH(2);
    else
      R2S_VOXEL_FWD_REACH(4);
#undef R2S_VOXEL_FWD_REACH
  } else {
    launch_voxel_fwd<T>(means3d, conics, opac, tile_offsets, flatten_ids, n_isects, n_keys, koff,
                        N, D2, D1, D0, ts, n2, n1, volume, stream);
  }
  return check_launch(name);
}

template <typename T, int R, bool kExact>
void launch_voxel_bwd(const T *means3d, const T *conics, const T *opac,
                      const int32_t *tile_offsets, const int64_t *isect_ids,
                      const int32_t *flatten_ids, const int32_t *isect_src, int64_t n_isects,
                      uint32_t n_keys, uint32_t koff, int64_t N, const T *v_vol, uint32_t D2,
                      uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, bool vec,
                      T *v_means, T *v_conics, T *v_opac, T *rows, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(ceil_div(n_isects, kBwdThreads)));
  if (rows != nullptr)
    voxel_bwd_kernel<T, R, kExact, true><<<grid, dim3(kBwdThreads), 0, stream>>>(
        means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, isect_src, n_isects, n_keys,
        koff, N, v_vol, D2, D1, D0, ts, n2, n1, vec, v_means, v_conics, v_opac, rows);
  else
    voxel_bwd_kernel<T, R, kExact, false><<<grid, dim3(kBwdThreads), 0, stream>>>(
        means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, isect_src, n_isects, n_keys,
        koff, N, v_vol, D2, D1, D0, ts, n2, n1, vec, v_means, v_conics, v_opac, rows);
}

int64_t voxel_rows_bytes(int64_t n_isects, int dtype_bytes) {
  return n_isects * row_stride<10>() * static_cast<int64_t>(dtype_bytes);
}

// Second pass of the two-pass backward: per-Gaussian sums of the rows.
template <typename T>
int voxel_reduce_impl(const T *rows, const int32_t *emit_ids, int64_t n_isects, int64_t N,
                      T *v_means, T *v_conics, T *v_opac, r2s_stream_t st) {
  const char *name = "voxelize_to_voxels_bwd (row reduction)";
  R2S_REQUIRE(N >= 0 && N <= kInt32Max && n_isects >= 0 && n_isects <= kInt32Max,
              "%s: bad size", name);
  if (N == 0) return R2S_OK;
  R2S_REQUIRE(v_means && v_conics && v_opac, "%s: null output", name);
  R2S_REQUIRE(n_isects == 0 || (rows && emit_ids), "%s: null pointer", name);
  R2S_REQUIRE(reinterpret_cast<uintptr_t>(rows) % 16 == 0, "%s: rows not 16-byte aligned", name);
  RowTargets<T, 10> tg = {{v_means, v_means + 1, v_means + 2, v_conics, v_conics + 1,
                           v_conics + 2, v_conics + 3, v_conics + 4, v_conics + 5, v_opac},
                          {3, 3, 3, 6, 6, 6, 6, 6, 6, 1}};
  launch_row_reduce(rows, emit_ids, n_isects, N, tg, as_stream(st));
  return check_launch(name);
}

// two_pass: emit_ids / isect_src / ws give the two-pass form (r2s_rows.h);
// rows_only stops after the first pass (the rows are left in ws).
template <typename T>
int voxel_bwd_impl(const T *means3d, const T *conics, const T *opac,
                   const int32_t *tile_offsets, const int64_t *isect_ids,
                   const int32_t *flatten_ids, const int32_t *emit_ids,
                   const int32_t *isect_src, int64_t n_isects, const T *v_vol, int64_t N,
                   uint32_t D2, uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1,
                   uint32_t n0, T *v_means, T *v_conics, T *v_opac, void *ws, size_t ws_bytes,
                   bool two_pass, r2s_stream_t st, bool rows_only = false, uint32_t z0 = 0,
                   bool slab = false, const uint64_t *reach = nullptr) {
  clear_error();
  const char *name = two_pass   ? "voxelize_to_voxels_bwd (two-pass)"
                     : isect_ids ? "voxelize_to_voxels_bwd_per_gaussian"
                                 : "voxelize_to_voxels_bwd";
  R2S_RETURN_IF(check_voxel_args(n_isects, N, D2, D1, D0, ts, n2, n1, n0, name, z0, slab));
  R2S_REQUIRE(reach == nullptr || ts == 8, "%s: reach masks need tile_size 8", name);
  if (N == 0) return R2S_OK;
  const int64_t n_vox = static_cast<int64_t>(D2) * D1 * D0;
  if (n_isects == 0 || n_vox == 0) {  // the two-pass form still stores its (zero) outputs
    if (!two_pass || rows_only) return R2S_OK;
    return voxel_reduce_impl<T>(nullptr, nullptr, 0, N, v_means, v_conics, v_opac, st);
  }
  R2S_REQUIRE(tile_offsets && flatten_ids, "%s: null brick lists", name);
  R2S_REQUIRE(means3d && conics && opac && v_vol, "%s: null pointer", name);
  R2S_REQUIRE(rows_only || (v_means && v_conics && v_opac), "%s: null output", name);
  T *rows = nullptr;
  if (two_pass) {
    R2S_REQUIRE(isect_src && (rows_only || emit_ids), "%s: null emit_ids / isect_src", name);
    const int64_t need = voxel_rows_bytes(n_isects, sizeof(T));
    if (ws == nullptr || static_cast<int64_t>(ws_bytes) < need) {
      set_error("%s: workspace of %zu bytes, %lld required", name, ws_bytes, (long long)need);
      return R2S_EWORKSPACE;
    }
    R2S_REQUIRE(reinterpret_cast<uintptr_t>(ws) % 16 == 0, "%s: workspace not 16-byte aligned",
                name);
    rows = static_cast<T *>(ws);
  }
  const uint32_t n_keys = n2 * n1 * n0, koff = z0 * n1 * n2;
  hipStream_t stream = as_stream(st);
  // 16-byte loads of gradient rows when every row segment starts aligned.
  const bool vec = vec_rows_ok<T>(v_vol, D2, ts);
#define R2S_VOXEL_BWD_R(RR, EXACT)                                                             \
  launch_voxel_bwd<T, RR, EXACT>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids,  \
                                 isect_src, n_isects, n_keys, koff, N, v_vol, D2, D1, D0, ts,  \
                                 n2, n1, vec, v_means, v_conics, v_opac, rows, stream)
  const int64_t elem = static_cast<int64_t>(sizeof(T));
  // The unstaged chunks read whole bricks at 32-bit offsets and 24-bit strides.
  const bool whole = vec && D2 % 8 == 0 && D1 % 8 == 0 && D0 % 8 == 0 &&
                     n2 * 8 == D2 && n1 * 8 == D1 &&
                     (static_cast<int64_t>(z0) + n0) * 8 <= D0 &&
                     n_vox * elem <= (int64_t{1} << 32) &&
                     static_cast<int64_t>(D1) * D2 * elem < (int64_t{1} << 24);
  const bool stage = stage_bricks<T>(n_isects, n_keys, whole);
  if (ts == 8 && rows != nullptr && (stage || whole)) {
    const dim3 grid(static_cast<uint32_t>(ceil_div(n_isects, 64 * kChunkWaves)));
#define R2S_VOXEL_BWD_CHUNK(GIVEN, STAGE)                                                       \
  voxel_bwd_chunk_kernel<T, GIVEN, STAGE><<<grid, dim3(64 * kChunkWaves), 0, stream>>>(         \
      means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, isect_src, n_isects, n_keys, \
      koff, N, v_vol, D2, D1, D0, n2, n1, vec, rows, reach)
    if (reach != nullptr && stage)
      R2S_VOXEL_BWD_CHUNK(true, true);
    else if (reach != nullptr)
      R2S_VOXEL_BWD_CHUNK(true, false);
    else if (stage)
      R2S_VOXEL_BWD_CHUNK(false, true);
    else
      R2S_VOXEL_BWD_CHUNK(false, false);
#undef R2S_VOXEL_BWD_CHUNK
  } else if (ts == 8)
    R2S_VOXEL_BWD_R(8, true);
  else if (ts == 4)
    R2S_VOXEL_BWD_R(4, true);
  else if (ts < 4)
    R2S_VOXEL_BWD_R(4, false);
  else if (ts < 8)
    R2S_VOXEL_BWD_R(8, false);
  else
    R2S_VOXEL_BWD_R(16, false);
#undef R2S_VOXEL_BWD_R
  R2S_RETURN_IF(check_launch(name));
  if (!two_pass || rows_only) return R2S_OK;
  return voxel_reduce_impl<T>(rows, emit_ids, n_isects, N, v_means, v_conics, v_opac, st);
}

}  // namespace
}  // namespace r2s

extern "C" {

int64_t r2s_voxelize_bwd_workspace_bytes(int64_t n_isects, int dtype_bytes) {
  if (n_isects <= 0 || (dtype_bytes != 4 && dtype_bytes != 8)) return 0;
  return r2s::voxel_rows_bytes(n_isects, dtype_bytes);
}

#define R2S_VOXEL_API(SUF, T)                                                                  \
  int r2s_voxelize_fwd_##SUF(const T *means3d, const T *conics, const T *opac,                 \
                             const int32_t *tile_offsets, const int32_t *flatten_ids,          \
                             int64_t n_isects, int64_t N, uint32_t D2, uint32_t D1,            \
                             uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0,  \
                             T *volume, r2s_stream_t st) {                                     \
    return r2s::voxel_fwd_impl<T>(means3d, conics, opac, tile_offsets, flatten_ids, n_isects,  \
                                  N, D2, D1, D0, ts, n2, n1, n0, volume, st);                  \
  }                                                                                            \
  int r2s_voxelize_bwd_##SUF(const T *means3d, const T *conics, const T *opac,                 \
                             const int32_t *tile_offsets, const int64_t *isect_ids,            \
                             const int32_t *flatten_ids, int64_t n_isects, const T *v_vol,     \
                             int64_t N, uint32_t D2, uint32_t D1, uint32_t D0, uint32_t ts,    \
                             uint32_t n2, uint32_t n1, uint32_t n0, T *v_means, T *v_conics,   \
                             T *v_opac, r2s_stream_t st) {                                     \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  nullptr, nullptr, n_isects, v_vol, N, D2, D1, D0, ts, n2,    \
                                  n1, n0, v_means, v_conics, v_opac, nullptr, 0, false, st);   \
  }                                                                                            \
  int r2s_voxelize_bwd_emit_##SUF(                                                             \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *emit_ids,           \
      const int32_t *isect_src, int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2,      \
      uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0,            \
      T *v_means, T *v_conics, T *v_opac, void *ws, size_t ws_bytes, r2s_stream_t st) {        \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  emit_ids, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2, \
                                  n1, n0, v_means, v_conics, v_opac, ws, ws_bytes, true, st);  \
  }                                                                                            \
  int r2s_voxelize_fwd_reach_##SUF(const T *means3d, const T *conics, const T *opac,           \
                                   const int32_t *tile_offsets, const int32_t *flatten_ids,    \
                                   int64_t n_isects, int64_t N, uint32_t D2, uint32_t D1,      \
                                   uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1,         \
                                   uint32_t n0, T *volume, uint64_t *reach, r2s_stream_t st) { \
    return r2s::voxel_fwd_impl<T>(means3d, conics, opac, tile_offsets, flatten_ids, n_isects,  \
                                  N, D2, D1, D0, ts, n2, n1, n0, volume, st, 0, false, reach); \
  }                                                                                            \
  int r2s_voxelize_bwd_emit_reach_##SUF(                                                       \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *emit_ids,           \
      const int32_t *isect_src, int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2,      \
      uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0,            \
      const uint64_t *reach, T *v_means, T *v_conics, T *v_opac, void *ws, size_t ws_bytes,    \
      r2s_stream_t st) {                                                                       \
    if (reach == nullptr) {                                                                    \
      r2s::clear_error();                                                                      \
      r2s::set_error("voxelize_to_voxels_bwd (two-pass): null reach masks");                   \
      return R2S_EINVAL;                                                                       \
    }                                                                                          \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  emit_ids, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2, \
                                  n1, n0, v_means, v_conics, v_opac, ws, ws_bytes, true, st,   \
                                  false, 0, false, reach);                                     \
  }                                                                                            \
  int r2s_voxelize_fwd_slab_##SUF(const T *means3d, const T *conics, const T *opac,            \
                                  const int32_t *tile_offsets, const int32_t *flatten_ids,     \
                                  int64_t n_isects, int64_t N, uint32_t D2, uint32_t D1,       \
                                  uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1,          \
                                  uint32_t z0, uint32_t nz, T *volume, r2s_stream_t st) {      \
    return r2s::voxel_fwd_impl<T>(means3d, conics, opac, tile_offsets, flatten_ids, n_isects,  \
                                  N, D2, D1, D0, ts, n2, n1, nz, volume, st, z0, true);        \
  }                                                                                            \
  int r2s_voxelize_bwd_emit_slab_##SUF(                                                        \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *emit_ids,           \
      const int32_t *isect_src, int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2,      \
      uint32_t D1, uint32_t D0, uint32_t ts, uint32_t n2, uint32_t n1, uint32_t z0,            \
      uint32_t nz, T *v_means, T *v_conics, T *v_opac, void *ws, size_t ws_bytes,              \
      r2s_stream_t st) {                                                                       \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  emit_ids, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2, \
                                  n1, nz, v_means, v_conics, v_opac, ws, ws_bytes, true, st,   \
                                  false, z0, true);                                            \
  }

#define R2S_VOXEL_STAGE_API(SUF, T)                                                            \
  int r2s_voxelize_bwd_rows_##SUF(                                                             \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *isect_src,          \
      int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2, uint32_t D1, uint32_t D0,      \
      uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0, void *rows, size_t rows_bytes,       \
      r2s_stream_t st) {                                                                       \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  nullptr, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2,  \
                                  n1, n0, nullptr, nullptr, nullptr, rows, rows_bytes, true,   \
                                  st, true);                                                   \
  }                                                                                            \
  int r2s_voxelize_bwd_rows_reach_##SUF(                                                       \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *isect_src,          \
      int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2, uint32_t D1, uint32_t D0,      \
      uint32_t ts, uint32_t n2, uint32_t n1, uint32_t n0, const uint64_t *reach, void *rows,   \
      size_t rows_bytes, r2s_stream_t st) {                                                    \
    if (reach == nullptr) {                                                                    \
      r2s::clear_error();                                                                      \
      r2s::set_error("voxelize_to_voxels_bwd (two-pass): null reach masks");                   \
      return R2S_EINVAL;                                                                       \
    }                                                                                          \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  nullptr, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2,  \
                                  n1, n0, nullptr, nullptr, nullptr, rows, rows_bytes, true,   \
                                  st, true, 0, false, reach);                                  \
  }                                                                                            \
  int r2s_voxelize_bwd_rows_slab_##SUF(                                                        \
      const T *means3d, const T *conics, const T *opac, const int32_t *tile_offsets,           \
      const int64_t *isect_ids, const int32_t *flatten_ids, const int32_t *isect_src,          \
      int64_t n_isects, const T *v_vol, int64_t N, uint32_t D2, uint32_t D1, uint32_t D0,      \
      uint32_t ts, uint32_t n2, uint32_t n1, uint32_t z0, uint32_t nz, void *rows,             \
      size_t rows_bytes, r2s_stream_t st) {                                                    \
    return r2s::voxel_bwd_impl<T>(means3d, conics, opac, tile_offsets, isect_ids, flatten_ids, \
                                  nullptr, isect_src, n_isects, v_vol, N, D2, D1, D0, ts, n2,  \
                                  n1, nz, nullptr, nullptr, nullptr, rows, rows_bytes, true,   \
                                  st, true, z0, true);                                         \
  }                                                                                            \
  int r2s_voxelize_bwd_reduce_##SUF(const T *rows, const int32_t *emit_ids, int64_t n_isects,  \
                                    int64_t N, T *v_means, T *v_conics, T *v_opac,             \
                                    r2s_stream_t st) {                                         \
    r2s::clear_error();                                                                        \
    return r2s::voxel_reduce_impl<T>(rows, emit_ids, n_isects, N, v_means, v_conics, v_opac,   \
                                     st);                                                      \
  }

R2S_VOXEL_STAGE_API(f32, float)
R2S_VOXEL_STAGE_API(f64, double)

#undef R2S_VOXEL_STAGE_API

R2S_VOXEL_API(f32, float)
R2S_VOXEL_API(f64, double)

#undef R2S_VOXEL_API

}  // extern "C"
