// Projective point-to-plane ICP on the device.
//
// Reference: CorrespondenceSearch::match, IcpCorrespondence::from_match and
// IcpNormalEquations::accumulate (include/kinectfusion/icp_correspondence.hpp:
// 44-294); the whole-level device loop (src/kinectfusion/cuda/
// icp_correspondence.cu:216-343) with its host epilogue
// (src/kinectfusion/icp_optimizer.cpp:82-169).
//
// One kernel per Gauss-Newton / LM trial (icp_step_kernel):
//  * every workgroup reduces the partial rows that the step before wrote, in a
//    fixed order with Kahan-compensated FP32, and its first wave runs that
//    step's trial on the sums: FP64 pivoted LDL^T solve, caps, Rodrigues
//    increment and pose composition, convergence and failure latches.  All
//    do the same work, so no launch and no device-scope fence stands between a
//    trial and the next sweep (such a fence in every sweep workgroup writes
//    back the L2 and costs more than the sweep itself);
//  * then every thread matches its pixels (up to five at a time, without
//    branches, their memory reads in flight together) and keeps the 29
//    per-correspondence terms (21 J^T J, 6 J^T r, distance, r^2) in FP32
//    registers;
//  * a wave reduces them by halves, the four waves of a workgroup combine in a
//    fixed order through LDS, and each workgroup writes one partial row -- no
//    float atomics, so the sums do not depend on scheduling.
// What bounds it: latency, not rate.  A 640 x 480 sweep reads 20 MB (4 us of a
// copy's rate) with one wave per SIMD; back to back, a launch costs 2.2 us
// before it does anything and 4.4 us with its reads from another die.  A step
// takes 14 us (sweep 5, trial 5) where the sweep and the one-thread trial as
// two launches took 20, and a level of 10 steps, 3 of them active, 85 us for
// 122.  kf_icp_track_maps over 640 x 480 maps: 112 us for 168.
// Once a level's status latches (converged or failed) the remaining steps pass
// the record on and return.  The stability spectrum (FP64) is checked once per
// level, by its last kernel, as in the reference's device loop.  A pass that
// usually exits at once runs each level in one launch instead
// (icp_level_kernel).
#include <cstddef>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "kf_internal.hpp"

// Partial rows of the allocation-free reduction (kf_icp_reduce_static): one
// row of 32 floats per sweep workgroup, at most 256 workgroups (32 KiB).
// Each device holds its own copy for the life of the process; host code
// reaches it only through the address hipGetSymbolAddress returns for the
// current device (static_scratch_rows below), never through this name.
static __device__ __align__(256) float scratch[256 * 32];

namespace kf {
namespace {

constexpr int kSums = 29;
constexpr int kPartialStride = 32;
constexpr int kMaxBlocks = 256;  // partial rows staged in 32 KB of LDS

struct Maps {
  const float4* __restrict__ lv;
  const float4* __restrict__ ln;
  const float4* __restrict__ mv;
  const float4* __restrict__ mn;
  int lw, lh, mw, mh;
  Intr k;
};

// match() (icp_correspondence.hpp:44-110) in two halves so that a thread
// can keep the memory reads of several pixels in flight together, and without
// branches, so that the arithmetic of several pixels overlaps as well: a wave
// has its SIMD to itself, and nothing else hides its latencies.
// Front: transform the live vertex and project it into the model maps; false
// (and model pixel 0) when rejected before the model read.
__device__ inline bool match_front(const Maps& m, const Rigid& cam, const Rigid& mod, V3 lv, V3 ln, V3& src,
                                   size_t& mi) {
  src = xform(cam, lv);
  const V3 sim = xform(mod, src);
  float u, v;
  project(m.k, sim, u, v);
  const float col = roundf(u), row = roundf(v);  // lround into [0, size); a NaN fails
  const bool ok = finite3(lv) && finite3(ln) && finite3(sim) && sim.z > 0.0F && col >= 0.0F &&
                  col < static_cast<float>(m.mw) && row >= 0.0F && row < static_cast<float>(m.mh);
  mi = ok ? static_cast<size_t>(static_cast<int>(row)) * m.mw + static_cast<int>(col) : 0;
  return ok;
}

// Back: with the model vertex and normal read, the distance and normal
// tests and the point-to-plane row (J, residual), zero if there is no match.
__device__ inline bool match_back(const Rigid& cam, float max_dist, float min_dot, bool ok, V3 ln, V3 src, V3 mv,
                                  V3 mn, float* J, float& res, float& dist) {
  const V3 r = rot(cam, ln);
  const float len = norm3(r);
  const V3 q = div3(r, len);
  const bool unit = len > 0.0F;
  const V3 sn = mk3(unit ? q.x : 0.0F, unit ? q.y : 0.0F, unit ? q.z : 0.0F);
  const float d = norm3(sub3(src, mv));
  ok = ok && finite3(mv) && finite3(mn) && !(d > max_dist) && !(dot3(sn, mn) < min_dot);
  const V3 r3 = cross3(src, mn);
  const float e = dot3(mn, sub3(mv, src));
  J[0] = ok ? r3.x : 0.0F;
  J[1] = ok ? r3.y : 0.0F;
  J[2] = ok ? r3.z : 0.0F;
  J[3] = ok ? mn.x : 0.0F;
  J[4] = ok ? mn.y : 0.0F;
  J[5] = ok ? mn.z : 0.0F;
  res = ok ? e : 0.0F;
  dist = ok ? d : 0.0F;
  return ok;
}

// Pixels a thread matches per pass (grid-stride order): their live reads,
// then their model reads, are issued together; the terms are added in pixel
// order (a rejected pixel adds +0, which changes no sum: none is ever -0).
// Five fill the widest grid's share of a 640 x 480 level in one pass; a grid
// whose threads have one or two pixels each takes a pass of that size (with
// five, a 160 x 120 sweep took 8.0 us for 4.8: four fifths of it on nothing).
template <int Batch>
struct LiveBatch {
  V3 v[Batch], n[Batch];
};

__device__ inline int sweep_base(int blk) {
  return blk * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
}

// The live pixels of a pass, the last one again past the end.
template <int Batch>
__device__ __forceinline__ void read_live(const Maps& m, int base, int stride, LiveBatch<Batch>& live) {
  const int last = m.lw * m.lh - 1;
#pragma unroll
  for (int j = 0; j < Batch; ++j) {
    const int p = min(base + j * stride, last);
    live.v[j] = ld3(m.lv[p]);
    live.n[j] = ld3(m.ln[p]);
  }
}

// Per-workgroup sweep: sums of block `blk`'s pixels (of `nblk` sweeping
// blocks) into partial[blk].  live: the first pass's pixels, read by the
// caller (ahead of whatever it waits for).
template <int Batch>
__device__ __forceinline__ void sweep_block(const Maps& m, const Rigid& cam, const Rigid& mod, float max_dist,
                                            float min_dot, float* __restrict__ partial, float (*lds)[kSums + 1],
                                            int blk, int nblk, LiveBatch<Batch>& live) {
  float s[kSums];
#pragma unroll
  for (int i = 0; i < kSums; ++i) s[i] = 0.0F;
  unsigned int cnt = 0;
  const int n = m.lw * m.lh;
  const int stride = nblk * static_cast<int>(blockDim.x);
  for (int base = sweep_base(blk); base < n;) {
    V3 src[Batch], mv[Batch], mn[Batch];
    size_t mi[Batch];
    bool ok[Batch];
#pragma unroll
    for (int j = 0; j < Batch; ++j) {
      ok[j] = match_front(m, cam, mod, live.v[j], live.n[j], src[j], mi[j]);
      ok[j] = ok[j] && base + j * stride < n;
    }
#pragma unroll
    for (int j = 0; j < Batch; ++j) {
      mv[j] = ld3(m.mv[mi[j]]);
      mn[j] = ld3(m.mn[mi[j]]);
    }
#pragma unroll
    for (int j = 0; j < Batch; ++j) {
      float J[6], res, dist;
      ok[j] = match_back(cam, max_dist, min_dot, ok[j], live.n[j], src[j], mv[j], mn[j], J, res, dist);
      int e = 0;
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = r; c < 6; ++c, ++e) s[e] += J[r] * J[c];
#pragma unroll
      for (int r = 0; r < 6; ++r) s[21 + r] += J[r] * res;
      s[27] += dist;
      s[28] += res * res;
      cnt += ok[j] ? 1U : 0U;
    }
    base += Batch * stride;
    if (base < n) read_live(m, base, stride, live);
  }
  // The wave's sums: at each step a lane keeps half of its values and takes
  // the other lanes' halves of them, so 32 exchanges reduce all 30 (a
  // butterfly of every value takes 180); each value is the same tree of
  // pairwise sums over lanes 32, 16, ..., 1 apart.  Lane 2 i ends with value i.
  // The count is summed as a float, exact below 2^24.
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float lo = s[i], hi = i + 16 < kSums ? s[i + 16] : (i + 16 == kSums ? static_cast<float>(cnt) : 0.0F);
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 8]), false, false);
    v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int half = 4; half > 0; half >>= 1) {  // lanes 8, 4 and 2 apart
    const bool upper = (lane & (2 * half)) != 0;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const float keep = upper ? v[i + half] : v[i], give = upper ? v[i] : v[i + half];
      v[i] = keep + __shfl_xor(give, 2 * half);
    }
  }
  v[0] += __shfl_xor(v[0], 1);
  if ((lane & 1) == 0 && lane <= 2 * kSums) lds[wave][lane >> 1] = v[0];
  __syncthreads();
  if (threadIdx.x < kSums) {
    const int i = threadIdx.x;
    partial[blk * kPartialStride + i] = (lds[0][i] + lds[1][i]) + (lds[2][i] + lds[3][i]);
  } else if (threadIdx.x == kSums) {
    unsigned int c = 0;
    for (int w = 0; w < 4; ++w) c += static_cast<unsigned int>(lds[w][kSums]);
    partial[blk * kPartialStride + kSums] = __uint_as_float(c);
  }
}

// Kahan-compensated FP32 sum of the partial rows.  The rows are first
// staged in LDS with coalesced loads.  Column c (29 sums and the count) is
// split over 8 threads: part q adds rows q, q + 8, ... with Kahan, then
// thread c adds the 8 part sums (net of their compensations) in order
// q = 0..7.  The order is fixed, so the result does not depend on scheduling.
// (256 threads; the reads apart, so that a caller can issue them ahead.)
using Quad = float __attribute__((ext_vector_type(4)));  // stays in registers (a float4 array goes to scratch)
struct RowBatch {
  Quad v[kMaxBlocks * kPartialStride / 4 / 256];
};

__device__ __forceinline__ void read_rows(const float* __restrict__ partial, int nblocks, RowBatch& rows) {
  const int last = nblocks * kPartialStride / 4 - 1;
#pragma unroll
  for (int j = 0; j < kMaxBlocks * kPartialStride / 4 / 256; ++j)  // every row in flight at once
    rows.v[j] = reinterpret_cast<const Quad*>(partial)[min(static_cast<int>(threadIdx.x) + j * 256, last)];
}

__device__ __forceinline__ void combine_rows(const RowBatch& batch, int nblocks, float* out) {
  __shared__ __align__(16) float rows[kMaxBlocks * kPartialStride];
  __shared__ float part_sum[8][kPartialStride];
  __shared__ float part_comp[8][kPartialStride];
  __shared__ unsigned part_cnt[8];
#pragma unroll
  for (int j = 0; j < kMaxBlocks * kPartialStride / 4 / 256; ++j)  // past nblocks: never read
    reinterpret_cast<Quad*>(rows)[static_cast<int>(threadIdx.x) + j * 256] = batch.v[j];
  __syncthreads();
  const int col = threadIdx.x & 31, q = threadIdx.x >> 5;  // 256 threads: 32 columns x 8 parts
  float sum = 0.0F, comp = 0.0F;
  unsigned cnt = 0;
  if (col < kSums) {
    for (int b = q; b < nblocks; b += 8) {
      const float y = rows[b * kPartialStride + col] - comp;
      const float t = sum + y;
      comp = (t - sum) - y;
      sum = t;
    }
  } else if (col == kSums) {
    for (int b = q; b < nblocks; b += 8) cnt += __float_as_uint(rows[b * kPartialStride + kSums]);
  }
  part_sum[q][col] = sum;
  part_comp[q][col] = comp;
  if (col == kSums) part_cnt[q] = cnt;
  __syncthreads();
  if (threadIdx.x < kSums) {
    float s2 = 0.0F, c2 = 0.0F;
    for (int k = 0; k < 8; ++k) {
      const float y = (part_sum[k][threadIdx.x] - part_comp[k][threadIdx.x]) - c2;
      const float t = s2 + y;
      c2 = (t - s2) - y;
      s2 = t;
    }
    out[threadIdx.x] = s2;
  } else if (threadIdx.x == kSums) {
    unsigned c = 0;
    for (int k = 0; k < 8; ++k) c += part_cnt[k];
    out[kSums] = __uint_as_float(c);
  }
}

__device__ __forceinline__ void combine_partials(const float* __restrict__ partial, int nblocks, float* out) {
  RowBatch rows;
  read_rows(partial, nblocks, rows);
  combine_rows(rows, nblocks, out);
}

// FP64 LDL^T with symmetric diagonal pivoting (largest remaining |d| first),
// the factorisation Eigen::LDLT uses in the reference host solve
// (icp_optimizer.cpp:391): a pivot with |d| <= DBL_MIN contributes a zero
// solution component, so a damped semidefinite system still solves; the
// solve fails only on a non-finite solution.
//
// By a wave: lane 8 r + c holds element (r, c) of the matrix, column 6 the
// right-hand side (so the forward substitution runs along with the
// elimination) and column 7 the row's place in the solution.  A lane divides
// for itself the two factors that its element's update takes; one thread
// eliminating alone spends 21 divisions and the swaps of every pivot one
// after the other.  A whole trial takes 7400 cycles, 9000 that way (12000
// with the steps unrolled or the solution in scratch memory).  Every operation is the scalar form's, in its order.  A
// solution that is not finite leaves x (in LDS) as it was.
__device__ inline void wave_sync() {  // LDS writes of a wave's lanes before the others' reads
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline double lane_value(double v, int lane) {  // lane: the same in every lane
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u), lane));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), lane));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

__device__ inline double shuffled(double v, int address) {  // address: 4 times the lane
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(address, static_cast<int>(u)));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(address, static_cast<int>(u >> 32)));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// The place of the largest |diagonal| element from k on, the first of equal
// ones; a NaN is never larger, and nothing is larger than one at k.  Almost
// always the upper halves alone decide, in scalar registers.
__device__ __forceinline__ int pivot_of(double a, int lane, int k) {
  const uint32_t high = static_cast<uint32_t>(__builtin_bit_cast(uint64_t, a) >> 32) & 0x7FFFFFFFU;
  const bool diagonal = (lane >> 3) == (lane & 7) && (lane >> 3) >= k && lane < 46;
  const uint32_t key = diagonal ? high : 0U;
  uint32_t most = 0;
#pragma unroll
  for (int i = 0; i < 6; ++i)
    most = max(most, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key), 9 * i)));
  const uint64_t at = __ballot(key == most);
  if (most != 0 && most < 0x7FF00000U && __builtin_popcountll(at) == 1) return __builtin_ctzll(at) >> 3;
  int piv = k;
  double best = fabs(lane_value(a, 9 * k));
#pragma unroll 1
  for (int i = k + 1; i < 6; ++i) {
    const double v = fabs(lane_value(a, 9 * i));
    if (v > best) {
      best = v;
      piv = i;
    }
  }
  return __builtin_amdgcn_readfirstlane(piv);
}

__device__ __forceinline__ bool solve6(const double* eq, int damping_mode, double scale, double* x) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int row = lane >> 3, col = lane & 7;
  const int hi = max(row, col), lo = min(row, col);
  const bool rhs = col == 6;
  double a = eq[row < 6 && col < 6 ? lo * 6 - lo * (lo - 1) / 2 + hi - lo : 21 + min(row, 5)];
  a = col == 7 ? static_cast<double>(row) : a;
  if (damping_mode != 0) {
    const double damped = a + (damping_mode == 1 ? scale : scale * a);
    a = col == row ? damped : a;
  }
  double quotient = 0.0;  // (row, 6): y / d
  int upper_at = 4 * (8 * (rhs ? row : min(hi, 5)));
  int lower_at = 4 * (rhs ? 6 : 8 * min(lo, 5));
  const int lower_step = rhs ? 32 : 4;
#pragma unroll 1
  for (int k = 0; k < 6; ++k) {
    const int piv = pivot_of(a, lane, k);
    if (piv != k) {  // the rows and the columns k and piv change places
      const int from_row = row == k ? piv : (row == piv ? k : row);
      const int from_col = col == k ? piv : (col == piv ? k : col);
      a = shuffled(a, 4 * (8 * from_row + from_col));
    }
    const double d = lane_value(a, 9 * k);
    const bool zero = fabs(d) <= 2.2250738585072014e-308;
    // below the pivot: a -= (l_hi d) l_lo, and the right-hand side less l y
    const double upper = shuffled(a, upper_at);
    const double lower = shuffled(a, lower_at);
    upper_at += 4;
    lower_at += lower_step;
    const double l = zero ? 0.0 : upper / d;  // (row, 6): of this row
    const double q = zero ? 0.0 : lower / d;  // (row, 6): y_k / d
    const double less = (rhs ? l : l * d) * (rhs ? lower : q);
    const bool inside = row > k && row < 6;
    if (rhs && row == k) quotient = q;
    if (inside && col == k) a = l;
    if (inside && col > k && col < 7) a -= less;
  }
  double z[6], own = 0.0;
  bool ok = true;
#pragma unroll
  for (int i = 5; i >= 0; --i) {
    double v = lane_value(quotient, 8 * i + 6);
#pragma unroll
    for (int j = i + 1; j < 6; ++j) v -= lane_value(a, 8 * j + i) * z[j];
    z[i] = v;
    own = row == i ? v : own;
    ok = ok && isfinite(v);
  }
  if (ok && col == 7 && row < 6) x[static_cast<int>(a)] = own;
  wave_sync();
  return ok;
}

// pose <- exp([w]) pose in FP64 (Rodrigues; left-multiplied world-frame
// increment, icp_optimizer.cpp:286), by a wave: a lane writes an element.
__device__ __forceinline__ void compose_increment(const double* x, double angle, double* pose) {
  const double wx = x[0], wy = x[1], wz = x[2];  // angle: their length
  double R[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  if (angle > 1.0e-12) {
    const double ux = wx / angle, uy = wy / angle, uz = wz / angle;
    double s, c;
    sincos(angle, &s, &c);
    const double oc = 1.0 - c;
    R[0] = c + ux * ux * oc;
    R[1] = ux * uy * oc - uz * s;
    R[2] = ux * uz * oc + uy * s;
    R[3] = uy * ux * oc + uz * s;
    R[4] = c + uy * uy * oc;
    R[5] = uy * uz * oc - ux * s;
    R[6] = uz * ux * oc - uy * s;
    R[7] = uz * uy * oc + ux * s;
    R[8] = c + uz * uz * oc;
  }
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int r = (lane >> 2) & 3, c = lane & 3;
  const double r0 = r == 0 ? R[0] : (r == 1 ? R[3] : R[6]);
  const double r1 = r == 0 ? R[1] : (r == 1 ? R[4] : R[7]);
  const double r2 = r == 0 ? R[2] : (r == 1 ? R[5] : R[8]);
  const double t = x[3 + min(r, 2)];
  double out = r0 * pose[c] + r1 * pose[4 + c] + r2 * pose[8 + c];
  if (c == 3) out += t;
  wave_sync();  // every lane has read the pose
  if (lane < 12) pose[lane] = out;
}

__device__ __noinline__ void sym_eig6(const double* eq, double* ev);

// check_system_stability (icp_optimizer.cpp:319-347) on FP64 sums.
__device__ bool stable_from_eigenvalues(const double* ev, const DeviceIcpParams& p, double* min_eig, double* cond);

__device__ bool stable_system(const double* eq, long long count, const DeviceIcpParams& p,
                              double* min_eig, double* cond) {
  if (count < p.min_corr) return false;
  __shared__ double ev[6];  // a wave's lanes write the same values
  sym_eig6(eq, ev);
  return stable_from_eigenvalues(ev, p, min_eig, cond);
}

__device__ bool stable_from_eigenvalues(const double* ev, const DeviceIcpParams& p, double* min_eig, double* cond) {
  double mn = ev[0], mx = ev[0];
  for (int i = 0; i < 6; ++i) {
    if (!isfinite(ev[i])) return false;
    mn = fmin(mn, ev[i]);
    mx = fmax(mx, ev[i]);
  }
  if (min_eig != nullptr) *min_eig = mn;
  if (!(mn > 0.0 && mx > 0.0)) return false;
  if (cond != nullptr) *cond = mx / mn;
  return mn >= static_cast<double>(p.min_eig) && mx / mn <= static_cast<double>(p.max_cond);
}

// One trial on the combined sums (solve_update_kernel semantics), by the first
// wave of a workgroup, its record and the sums in LDS.  A failing trial
// reports kUnconstrainedSystem when the undamped system is unstable, as the
// reference host loop vetoes before solving (icp_optimizer.cpp:263-270).
__device__ __forceinline__ void run_trial(IcpTrial* t, const DeviceIcpParams& p, const float* sums32) {
  const int lane = static_cast<int>(threadIdx.x);
  const double sum = lane < kSums ? static_cast<double>(sums32[lane]) : 0.0;
  const long long count = static_cast<long long>(__float_as_uint(sums32[kSums]));
  if (count < p.min_corr) {
    if (lane < kSums) t->eq[lane] = sum;
    if (lane == 0) {
      t->eq_count = count;
      t->status = 2;
    }
    return;
  }
  const int trials = t->trials;
  double lambda = trials == 0 ? static_cast<double>(p.lambda0) : t->lambda;
  const bool damping = p.damping_mode != 0;
  const bool adaptive = damping && p.adaptive != 0;
  bool accepted = true;
  long long eq_count = count;
  double eq = sum;
  if (adaptive) {
    const double cost = static_cast<double>(sums32[28]) / static_cast<double>(count);
    accepted = trials == 0 || cost <= t->best_cost;
    wave_sync();  // every lane has read what lane 0 writes
    if (accepted) {
      if (lane < kSums) t->best_eq[lane] = sum;
      if (lane < 16) t->best_pose[lane] = t->pose[lane];
      if (lane == 0) {
        t->best_cost = cost;
        t->best_count = count;
      }
      lambda = fmax(lambda * p.dec, static_cast<double>(p.lmin));
    } else {
      if (lane < 16) t->pose[lane] = t->best_pose[lane];
      if (lane == 0) ++t->rejected;
      lambda = fmin(lambda * p.inc, static_cast<double>(p.lmax));
      if (lane < kSums) eq = t->best_eq[lane];
      eq_count = t->best_count;
    }
  }
  wave_sync();
  if (lane < kSums) t->eq[lane] = eq;
  wave_sync();
  const int attempts = damping ? 8 : 1;
  __shared__ double x[6];
  double scale = lambda, ut = 0.0, ang = 0.0;
  bool solved = false;
  for (int a = 0; a < attempts; ++a) {
    if (solve6(t->eq, p.damping_mode, scale, x)) {
      solved = true;
      lambda = scale;
      ang = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
      ut = sqrt(x[3] * x[3] + x[4] * x[4] + x[5] * x[5]);
      if (!damping || (ut <= p.max_t && ang <= p.max_r)) break;
    }
    scale = fmin(scale * p.inc, static_cast<double>(p.lmax));
  }
  int status = 0;
  if (!solved || ut > p.max_t || ang > p.max_r) {
    const bool unstable = !damping && !stable_system(t->eq, eq_count, p, nullptr, nullptr);
    status = unstable ? 5 : (solved ? 4 : 3);
  } else {
    compose_increment(x, ang, t->pose);
    if (accepted && ut < p.min_t && ang < p.min_r) status = 1;
  }
  if (lane == 0) {
    t->eq_count = eq_count;
    t->trials = trials + 1;
    t->lambda = lambda;
    if (solved) {
      t->update_t = ut;
      t->update_r = ang;
    }
    t->status = status;
  }
}

template <typename State>
__device__ void finish_level_block(IcpState* st, const State* t, const DeviceIcpParams& p, int level, float check_rms);

// The trial fields of a level's state, and their return (a whole workgroup of
// at least 32 threads; the caller synchronises).
template <typename To, typename From>
__device__ inline void copy_trial(To* to, const From* from) {
  const int i = static_cast<int>(threadIdx.x);
  if (i < 16) {
    to->pose[i] = from->pose[i];
    to->best_pose[i] = from->best_pose[i];
  }
  if (i < kSums) {
    to->eq[i] = from->eq[i];
    to->best_eq[i] = from->best_eq[i];
  }
  if (i == 0) {
    to->best_cost = from->best_cost;
    to->lambda = from->lambda;
    to->update_t = from->update_t;
    to->update_r = from->update_r;
    to->eq_count = from->eq_count;
    to->best_count = from->best_count;
    to->status = from->status;
    to->trials = from->trials;
    to->rejected = from->rejected;
  }
}

// One step of a level: the previous step's trial (its reduction and FP64
// solve), then this step's correspondence sweep.  Every workgroup solves the
// same trial for itself from the same rows, so a trial needs no launch of its
// own and no fence: a step reads the rows and the trial record the step before
// wrote (one of two, in turn) and writes the other.  Two launches per trial
// took 2 launch latencies and, once a level had latched, 2 empty launches.
__device__ inline void copy_record(IcpTrial* to, const IcpTrial* from) {  // by 256 threads
  static_assert(sizeof(IcpTrial) % 4 == 0 && sizeof(IcpTrial) / 4 <= 256, "a word per thread");
  if (threadIdx.x < sizeof(IcpTrial) / 4)
    reinterpret_cast<uint32_t*>(to)[threadIdx.x] = reinterpret_cast<const uint32_t*>(from)[threadIdx.x];
}

// The rows of step k.
__device__ inline float* step_rows(float* rows, int k) { return rows + (k & 1) * kMaxBlocks * kPartialStride; }

// The trial that follows a step, its record in LDS, from the step's rows.
__device__ __forceinline__ void solve_step(const DeviceIcpParams& p, const RowBatch& rows, int nblocks, IcpTrial* t,
                                  float* combined) {
  combine_rows(rows, nblocks, combined);
  __syncthreads();
  if (threadIdx.x < 64) run_trial(t, p, combined);
  __syncthreads();
}

// What a step reads -- the record and the rows of the step before, then the
// live pixels -- is in flight before the work that waits for it, as each read
// comes from another die's memory (about a microsecond).
template <int Batch>
__global__ void __launch_bounds__(256) icp_step_kernel(Maps m, DeviceIcpParams p, IcpState* st,
                                                        float* __restrict__ rows, int k) {
  __shared__ float lds[4][kSums + 1];
  __shared__ float combined[kSums + 1];
  __shared__ IcpTrial t;
  const int blk = static_cast<int>(blockIdx.x), nblk = static_cast<int>(gridDim.x);
  const int failed = st->frame_failed;
  const Rigid mod = rigid_from12(st->model_inv);
  LiveBatch<Batch> live;
  Rigid cam;
  if (k == 0) {
    cam = rigid_from_pose64(st->pose);
    if (failed != 0) return;
    read_live(m, sweep_base(blk), nblk * static_cast<int>(blockDim.x), live);
    if (blk == 0) copy_trial(&st->trial[0], st);  // the level's start as the first record
  } else {
    RowBatch before;
    read_rows(step_rows(rows, k - 1), nblk, before);
    copy_record(&t, &st->trial[(k - 1) & 1]);
    __syncthreads();
    if (failed != 0) return;
    const bool latched = t.status != 0;  // the record is passed on
    if (!latched) {
      read_live(m, sweep_base(blk), nblk * static_cast<int>(blockDim.x), live);
      solve_step(p, before, nblk, &t, combined);
    }
    if (blk == 0) copy_record(&st->trial[k & 1], &t);
    if (t.status != 0) return;
    cam = rigid_from_pose64(t.pose);
  }
  sweep_block(m, cam, mod, p.max_dist, p.min_dot, step_rows(rows, k), lds, blk, nblk, live);
}

// The end of a level after its last step (one workgroup): the last trial, the
// record's fields back in the state, the stability check and result, and the
// learned warm start's check.
__global__ void __launch_bounds__(256) icp_finish_steps_kernel(DeviceIcpParams p, IcpState* st,
                                                                float* __restrict__ rows, int nblocks, int steps,
                                                                int level, float check_rms) {
  __shared__ float combined[kSums + 1];
  __shared__ IcpTrial t;
  RowBatch before;
  read_rows(step_rows(rows, steps - 1), nblocks, before);
  copy_record(&t, &st->trial[(steps - 1) & 1]);
  const int failed = st->frame_failed;
  __syncthreads();
  if (failed == 0) {
    if (t.status == 0) solve_step(p, before, nblocks, &t, combined);
    copy_trial(st, &t);
    __syncthreads();
  }
  finish_level_block(st, &t, p, level, check_rms);
}

// Ticket protocol: returns true in the workgroup that finished last, after
// which the partial rows of every workgroup are visible (device-scope
// release before the ticket, acquire after it).
__device__ inline bool last_block(unsigned int* ticket) {
  __shared__ bool is_last;
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) is_last = atomicAdd(ticket, 1U) == gridDim.x - 1U;
  __syncthreads();
  if (is_last) __threadfence();
  return is_last;
}

// A whole level in one launch, for a pass whose levels usually exit at once
// (the learned warm start's fallback, when the learned run was kept): the
// workgroups run the level's trials in step.  Each trial: every workgroup
// sweeps its pixels into its partial row; the last to finish (ticket
// protocol) reduces them, solves, and publishes the trial by advancing an
// epoch word with a device-scope release; the others wait for the epoch
// with a device-scope acquire.  The grid is at most kMaxBlocks workgroups,
// all resident at once (checked on the host).  A wait that outlasts
// timeout_ticks of the 100 MHz wall clock (far beyond any trial by default)
// gives up: the workgroup marks the frame failed (it is then neither
// integrated nor reported tracked), counts the event in st->sync_timeouts
// for the host to report, and exits, so every wave ends.  The ticket a
// timed-out launch leaves short is reset when the next level begins.
// st->level_sync: [0] ticket, [1] epoch (only ever advanced: a launch reads
// its base before any workgroup can advance it).
template <int Batch>
__global__ void __launch_bounds__(256) icp_level_kernel(Maps m, DeviceIcpParams p, IcpState* st,
                                                        float* __restrict__ partial, long long timeout_ticks,
                                                        int iterations, int level) {
  __shared__ float lds[4][kSums + 1];
  __shared__ float combined[kSums + 1];
  __shared__ IcpTrial t;
  __shared__ float xf[24];
  __shared__ int go, timed_out;
  if (st->frame_failed) return;
  unsigned int* sync = st->level_sync;
  const unsigned int base = __hip_atomic_load(&sync[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
  for (int it = 0; it < iterations; ++it) {
    if (threadIdx.x == 0) {
      go = st->status == 0 ? 1 : 0;  // latched: the level is done
      if (go != 0) {
        for (int i = 0; i < 12; ++i) {
          xf[i] = static_cast<float>(st->pose[i]);
          xf[12 + i] = st->model_inv[i];
        }
      }
    }
    __syncthreads();
    if (go == 0) break;
    const Rigid cam = rigid_from12(xf), mod = rigid_from12(xf + 12);
    LiveBatch<Batch> live;
    read_live(m, sweep_base(blockIdx.x), static_cast<int>(gridDim.x * blockDim.x), live);
    sweep_block(m, cam, mod, p.max_dist, p.min_dot, partial, lds, static_cast<int>(blockIdx.x),
                static_cast<int>(gridDim.x), live);
    const unsigned int target = base + static_cast<unsigned int>(it) + 1U;
    if (last_block(&sync[0])) {
      copy_trial(&t, st);
      combine_partials(partial, gridDim.x, combined);
      __syncthreads();
      if (threadIdx.x < 64) run_trial(&t, p, combined);
      __syncthreads();
      copy_trial(st, &t);
      __syncthreads();
      if (threadIdx.x == 0) {
        sync[0] = 0U;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_store(&sync[1], target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
    } else {
      if (threadIdx.x == 0) {
        timed_out = 0;
        const long long t0 = wall_clock64();
        while (static_cast<int>(__hip_atomic_load(&sync[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) - target) <
               0) {
          if (wall_clock64() - t0 > timeout_ticks) {
            timed_out = 1;
            st->frame_failed = 1;
            st->failed_level = level;
            atomicAdd(&st->sync_timeouts, 1);
            break;
          }
          __builtin_amdgcn_s_sleep(2);
        }
      }
      __syncthreads();
      if (timed_out != 0) return;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
  }
  if (blockIdx.x == 0) finish_level_block(st, st, p, level, 0.0F);
}

// Single sweep with explicit float transforms (kf_icp_reduce), then its
// reduction into st->sums32.
template <int Batch>
__global__ void __launch_bounds__(256) icp_sweep_kernel(Maps m, Rigid cam, Rigid mod, float max_dist,
                                                         float min_dot, float* __restrict__ partial) {
  __shared__ float lds[4][kSums + 1];
  LiveBatch<Batch> live;
  read_live(m, sweep_base(blockIdx.x), static_cast<int>(gridDim.x * blockDim.x), live);
  sweep_block(m, cam, mod, max_dist, min_dot, partial, lds, static_cast<int>(blockIdx.x),
              static_cast<int>(gridDim.x), live);
}

// The reduction into the host's mirror of the state (mapped memory, seen by
// the host once the stream is synchronised): a copy of the state took as long
// as the sweep and the reduction together.
__global__ void __launch_bounds__(256) icp_combine_kernel(const IcpState* st, const float* __restrict__ partial,
                                                           int nblocks, IcpState* __restrict__ host) {
  __shared__ float combined[kSums + 1];
  const int timeouts = st->sync_timeouts;
  combine_partials(partial, nblocks, combined);
  __syncthreads();
  if (threadIdx.x <= kSums) host->sums32[threadIdx.x] = combined[threadIdx.x];
  if (threadIdx.x == 32) host->sync_timeouts = timeouts;
}

// The same reduction into caller memory: the 29 sums widened to FP64 and the
// correspondence count (kf_icp_reduce_static).
__global__ void __launch_bounds__(256) icp_combine_out_kernel(const float* __restrict__ partial, int nblocks,
                                                               double* __restrict__ sums,
                                                               int64_t* __restrict__ count) {
  __shared__ float combined[kSums + 1];
  combine_partials(partial, nblocks, combined);
  __syncthreads();
  if (threadIdx.x < kSums) sums[threadIdx.x] = static_cast<double>(combined[threadIdx.x]);
  else if (threadIdx.x == kSums) *count = static_cast<int64_t>(__float_as_uint(combined[kSums]));
}

// FP64 cyclic Jacobi eigenvalues of the symmetric 6x6 system.
__device__ __noinline__ void sym_eig6(const double* eq, double* ev) {
  double a[6][6];
  int e = 0;
  for (int r = 0; r < 6; ++r)
    for (int c = r; c < 6; ++c, ++e) {
      a[r][c] = eq[e];
      a[c][r] = eq[e];
    }
  // Sweeps stop once the off-diagonal mass is below (1e-16)^2 of the
  // diagonal's: the eigenvalues are then exact to ~1e-16 of the norm.
  for (int sweep = 0; sweep < 32; ++sweep) {
    double off = 0.0, diag = 0.0;
#pragma unroll
    for (int d = 0; d < 6; ++d) diag += a[d][d] * a[d][d];
#pragma unroll
    for (int pp = 0; pp < 6; ++pp)
#pragma unroll
      for (int q = pp + 1; q < 6; ++q) off += a[pp][q] * a[pp][q];
    if (off <= 1.0e-32 * diag) break;
#pragma unroll
    for (int pp = 0; pp < 6; ++pp)
#pragma unroll
      for (int q = pp + 1; q < 6; ++q) {
        if (a[pp][q] == 0.0) continue;
        const double theta = (a[q][q] - a[pp][pp]) / (2.0 * a[pp][q]);
        const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double c = 1.0 / sqrt(t * t + 1.0);
        const double s = t * c;
#pragma unroll
        for (int k2 = 0; k2 < 6; ++k2) {
          const double akp = a[k2][pp], akq = a[k2][q];
          a[k2][pp] = c * akp - s * akq;
          a[k2][q] = s * akp + c * akq;
        }
#pragma unroll
        for (int k2 = 0; k2 < 6; ++k2) {
          const double apk = a[pp][k2], aqk = a[q][k2];
          a[pp][k2] = c * apk - s * aqk;
          a[q][k2] = s * apk + c * aqk;
        }
      }
  }
  for (int i = 0; i < 6; ++i) ev[i] = a[i][i];
}

// The same eigenvalues computed by one wave (the stability check at the end
// of a level), in two steps:
//  * lane 0 reduces the system to tridiagonal form by four Householder
//    reflections H = I - beta v v^T, each applied as A - v w^T - w v^T with
//    p = beta A v, K = beta (v . p) / 2, w = p - K v (every index a
//    compile-time constant, so the matrix stays in registers);
//  * 60 lanes multisect the six eigenvalues: the 10 lanes of eigenvalue k
//    probe 10 interior points of its interval (initially the Gershgorin
//    interval of the tridiagonal matrix), each counting the eigenvalues below
//    its point by the sign changes of the Sturm sequence p_0 = 1,
//    p_1 = d_0 - x, p_i = (d_{i-1} - x) p_{i-1} - e_{i-2}^2 p_{i-2}
//    (division-free; magnitudes stay far inside the FP64 range for these
//    systems), and keep the sub-interval where the count passes k.  Sixteen
//    rounds shrink the interval by 11^16, to the rounding of the
//    tridiagonal matrix's norm.
// Backward stable: the eigenvalues agree with a full-precision solver to
// ~1e-15 of the norm (a CPU emulation of these steps checks it against
// numpy on condition numbers up to 1e8).  A non-finite system gives NaN.
constexpr int kSectRounds = 16;
constexpr int kSectProbes = 10;

__device__ inline int sturm_count_below(const double (&d)[6], const double (&e2)[5], double x) {
  double p_prev = 1.0, p = d[0] - x;
  bool neg = p < 0.0 || p == 0.0;  // a zero takes the sign opposite to its predecessor (+1)
  int changes = neg ? 1 : 0;
#pragma unroll
  for (int i = 1; i < 6; ++i) {
    const double p_next = (d[i] - x) * p - e2[i - 1] * p_prev;
    const bool n_neg = p_next == 0.0 ? !neg : p_next < 0.0;
    changes += n_neg != neg ? 1 : 0;
    neg = n_neg;
    p_prev = p;
    p = p_next;
  }
  return changes;
}

__device__ void sym_eig6_wave(const double* eq, double* ev) {
  __shared__ double tri[11];  // d[6], e[5]
  const int lane = threadIdx.x & 63;
  if (lane == 0) {
    double a[6][6];
    {
      int idx = 0;
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = r; c < 6; ++c, ++idx) {
          a[r][c] = eq[idx];
          a[c][r] = eq[idx];
        }
    }
    double d[6], e[5];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double n2 = 0.0;
#pragma unroll
      for (int i = k + 1; i < 6; ++i) n2 += a[i][k] * a[i][k];
      double alpha = sqrt(n2);
      if (a[k + 1][k] > 0.0) alpha = -alpha;
      double v[6];
#pragma unroll
      for (int i = k + 1; i < 6; ++i) v[i] = a[i][k];
      v[k + 1] -= alpha;
      double vn = 0.0;
#pragma unroll
      for (int i = k + 1; i < 6; ++i) vn += v[i] * v[i];
      e[k] = alpha;
      d[k] = a[k][k];
      if (vn > 0.0) {
        const double beta = 2.0 / vn;
        double pv[6], w[6];
        double kk = 0.0;
#pragma unroll
        for (int i = k + 1; i < 6; ++i) {
          double acc = 0.0;
#pragma unroll
          for (int j = k + 1; j < 6; ++j) acc += a[i][j] * v[j];
          pv[i] = beta * acc;
          kk += v[i] * pv[i];
        }
        kk *= 0.5 * beta;
#pragma unroll
        for (int i = k + 1; i < 6; ++i) w[i] = pv[i] - kk * v[i];
#pragma unroll
        for (int i = k + 1; i < 6; ++i)
#pragma unroll
          for (int j = k + 1; j < 6; ++j) a[i][j] -= v[i] * w[j] + w[i] * v[j];
      }
    }
    d[4] = a[4][4];
    d[5] = a[5][5];
    e[4] = a[5][4];
#pragma unroll
    for (int i = 0; i < 6; ++i) tri[i] = d[i];
#pragma unroll
    for (int i = 0; i < 5; ++i) tri[6 + i] = e[i];
  }
  wave_sync();
  double d[6], e2[5];
  bool finite = true;
  double lo = 1.0e308, hi = -1.0e308;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    d[i] = tri[i];
    finite = finite && isfinite(d[i]);
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const double ei = tri[6 + i];
    finite = finite && isfinite(ei);
    e2[i] = ei * ei;
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {  // Gershgorin discs of the tridiagonal matrix
    const double r = (i > 0 ? fabs(tri[5 + i]) : 0.0) + (i < 5 ? fabs(tri[6 + i]) : 0.0);
    lo = fmin(lo, d[i] - r);
    hi = fmax(hi, d[i] + r);
  }
  const double pad = (hi - lo) * 1.0e-12 + 1.0e-300;
  lo -= pad;
  hi += pad;
  const int k = lane / kSectProbes, j = lane % kSectProbes + 1;  // eigenvalue, probe (lanes < 60)
  for (int round = 0; round < kSectRounds; ++round) {
    const double step = (hi - lo) * (1.0 / (kSectProbes + 1));
    const bool above = k < 6 && sturm_count_below(d, e2, lo + step * j) > k;
    const unsigned long long votes = __ballot(above);
    const unsigned group = k < 6 ? static_cast<unsigned>((votes >> (kSectProbes * k)) & 0x3FFULL) : 0U;
    const int first = group != 0U ? __builtin_ctz(group) + 1 : kSectProbes + 1;  // first probe above
    const double nlo = first > 1 ? lo + step * (first - 1) : lo;
    const double nhi = first <= kSectProbes ? lo + step * first : hi;
    lo = nlo;
    hi = nhi;
  }
  if (k < 6 && j == 1) ev[k] = finite ? 0.5 * (lo + hi) : __builtin_nan("");
  wave_sync();
}

struct Pose64 {
  double m[16];
};

// A level between maps of the caller's: the model maps' pose and the start.
__global__ void __launch_bounds__(64) icp_begin_maps_kernel(IcpState* st, Pose64 model, Pose64 start) {
  const int i = static_cast<int>(threadIdx.x);
  if (i == 0) st->frame_failed = 0;
  if (i < 16) st->pose[i] = model.m[i];
  __syncthreads();
  if (i == 0) icp_begin_level(st, 0);
  __syncthreads();
  if (i < 16) {
    st->pose[i] = start.m[i];
    st->level_pose0[i] = start.m[i];
    st->best_pose[i] = start.m[i];
  }
}

// The state into the host's mirror (mapped memory; all but the steps' records,
// its end); then, after a standalone track, the context's own pose back.
__global__ void __launch_bounds__(256) icp_publish_kernel(IcpState* st, IcpState* __restrict__ host, int restore) {
  constexpr unsigned words = offsetof(IcpState, trial) / 8;
  static_assert(offsetof(IcpState, trial) % 8 == 0, "copied in 8-byte words");
  for (unsigned i = threadIdx.x; i < words; i += blockDim.x)
    reinterpret_cast<uint64_t*>(host)[i] = reinterpret_cast<const uint64_t*>(st)[i];
  if (restore == 0) return;
  __syncthreads();
  if (threadIdx.x < 16) st->pose[threadIdx.x] = st->prev_pose[threadIdx.x];
  if (threadIdx.x == 0) st->frame_failed = 0;
}

// Stability check and result record of a level (icp_optimizer.cpp:108-169),
// by a whole workgroup (the Jacobi sweeps take its first wave), then, when
// check_rms > 0, the learned warm start's check of this level.
// t: the level's trial fields (the state itself, or a copy of them in LDS).
template <typename State>
__device__ void finish_level_block(IcpState* st, const State* t, const DeviceIcpParams& p, int level, float check_rms) {
  __shared__ double ev[6];
  __shared__ int skip, check;
  if (threadIdx.x == 0) {
    skip = st->frame_failed;
    check = skip == 0 && (t->status == 0 || t->status == 1) && t->eq_count >= p.min_corr ? 1 : 0;
  }
  __syncthreads();
  if (skip == 0) {
    if (check != 0 && threadIdx.x < 64) sym_eig6_wave(t->eq, ev);  // the first wave
    if (threadIdx.x == 0) {
      kf_icp_result& r = st->results[level];
      int status = t->status;
      r.min_eigenvalue = 0.0;
      r.condition_number = 0.0;
      if (status == 0 || status == 1) {
        const bool stable = check != 0 && stable_from_eigenvalues(ev, p, &r.min_eigenvalue, &r.condition_number);
        if (!stable && p.damping_mode == 0) status = 5;
      }
      r.status = status;
      r.trials = t->trials;
      r.rejected = t->rejected;
      r.correspondences = t->eq_count;
      if (t->eq_count > 0) {
        r.mean_distance = t->eq[27] / static_cast<double>(t->eq_count);
        r.mean_squared_residual = t->eq[28] / static_cast<double>(t->eq_count);
      }
      r.update_translation = t->update_t;
      r.update_rotation = t->update_r;
      r.lambda = t->lambda;
      st->status = status;
      if (status >= 2) {
        // failure: the outcome keeps the level's initial pose
        for (int i = 0; i < 16; ++i) st->pose[i] = st->level_pose0[i];
        st->frame_failed = 1;
        st->failed_level = level;
      }
    }
  }
  if (check_rms > 0.0F && threadIdx.x == 0) learned_check(st, level, check_rms, p.learned_max_t, p.learned_max_r);
}

// A level with no trial: its finish alone.
__global__ void __launch_bounds__(64) icp_finish_level_kernel(IcpState* st, DeviceIcpParams p, int level,
                                                               float check_rms) {
  finish_level_block(st, st, p, level, check_rms);
}

Maps make_maps(const float4* lv_v, const float4* lv_n, int lw, int lh, const float4* md_v,
               const float4* md_n, int mw, int mh, Intr k) {
  return Maps{lv_v, lv_n, md_v, md_n, lw, lh, mw, mh, k};
}

int blocks_for(int n) { return std::max(1, std::min(kMaxBlocks, (n + 255) / 256)); }

}  // namespace

DeviceIcpParams to_device_params(const kf_icp_options& o) {
  DeviceIcpParams p{};
  p.min_corr = o.min_correspondences;
  p.max_dist = o.max_point_distance;
  p.min_dot = o.min_normal_dot;
  p.min_t = o.min_update_translation;
  p.min_r = o.min_update_rotation;
  p.max_t = o.max_update_translation;
  p.max_r = o.max_update_rotation;
  p.min_eig = o.min_system_eigenvalue;
  p.max_cond = o.max_condition_number;
  p.damping_mode = o.damping_mode;
  p.lambda0 = o.damping_lambda;
  p.adaptive = o.adaptive_damping;
  p.inc = o.lambda_increase;
  p.dec = o.lambda_decrease;
  p.lmin = o.min_lambda;
  p.lmax = o.max_lambda;
  return p;
}

namespace {

// f(the pixels of a pass): as many as a thread has, to five.
template <typename F>
void for_batch(const Maps& m, int nb, const F& f) {
  const int64_t threads = static_cast<int64_t>(nb) * 256, pixels = static_cast<int64_t>(m.lw) * m.lh;
  if (pixels <= threads) f(std::integral_constant<int, 1>{});
  else if (pixels <= 2 * threads) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, 5>{});
}

void launch_single_level(const Maps& m, int nb, kf_context* ctx, const DeviceIcpParams& p, int iterations, int level) {
  for_batch(m, nb, [&](auto batch) {
    static int resident = -1;  // workgroups of this kernel resident at once on this device
    if (resident < 0) {
      int per_cu = 0, dev = 0;
      KF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, icp_level_kernel<batch.value>, 256, 0));
      KF_HIP(hipGetDevice(&dev));
      hipDeviceProp_t prop{};
      KF_HIP(hipGetDeviceProperties(&prop, dev));
      resident = per_cu * prop.multiProcessorCount;
    }
    if (nb > resident) fail(KF_ERR_DEVICE, "icp level: the grid does not fit on the device at once");
    hipLaunchKernelGGL(icp_level_kernel<batch.value>, dim3(nb), dim3(256), 0, ctx->stream, m, p, ctx->icp,
                       ctx->partials, ctx->sync_timeout_ticks, iterations, level);
    KF_HIP(hipGetLastError());
  });
}

}  // namespace

void launch_icp_begin_maps(kf_context* ctx, const double* model_pose, const double* pose) {
  Pose64 model, start;
  std::memcpy(model.m, model_pose, sizeof(model.m));
  std::memcpy(start.m, pose, sizeof(start.m));
  hipLaunchKernelGGL(icp_begin_maps_kernel, dim3(1), dim3(64), 0, ctx->stream, ctx->icp, model, start);
  KF_HIP(hipGetLastError());
}

void launch_icp_publish(kf_context* ctx, bool restore) {
  hipLaunchKernelGGL(icp_publish_kernel, dim3(1), dim3(256), 0, ctx->stream, ctx->icp, ctx->icp_mapped,
                     restore ? 1 : 0);
  KF_HIP(hipGetLastError());
}

void launch_icp_level(kf_context* ctx, const float4* lv_v, const float4* lv_n, int lw, int lh,
                      const float4* md_v, const float4* md_n, int mw, int mh, Intr k, int iterations,
                      const DeviceIcpParams& p, int level, bool single_launch, float check_max_rms) {
  const Maps m = make_maps(lv_v, lv_n, lw, lh, md_v, md_n, mw, mh, k);
  const int nb = blocks_for(lw * lh);
  if (iterations <= 0) {
    hipLaunchKernelGGL(icp_finish_level_kernel, dim3(1), dim3(64), 0, ctx->stream, ctx->icp, p, level,
                       check_max_rms);
    KF_HIP(hipGetLastError());
    return;
  }
  if (single_launch) {
    if (check_max_rms > 0.0F) fail(KF_ERR_INVALID_ARGUMENT, "icp level: the learned check needs a launch per trial");
    launch_single_level(m, nb, ctx, p, iterations, level);
    return;
  }
  // one launch per trial, and one that ends the level (and runs the learned check)
  for_batch(m, nb, [&](auto batch) {
    for (int it = 0; it < iterations; ++it)
      hipLaunchKernelGGL(icp_step_kernel<batch.value>, dim3(nb), dim3(256), 0, ctx->stream, m, p, ctx->icp,
                         ctx->partials, it);
  });
  hipLaunchKernelGGL(icp_finish_steps_kernel, dim3(1), dim3(256), 0, ctx->stream, p, ctx->icp, ctx->partials, nb,
                     iterations, level, check_max_rms);
  KF_HIP(hipGetLastError());
}

void launch_icp_reduce_once(kf_context* ctx, const float4* lv_v, const float4* lv_n, int lw, int lh,
                            const float4* md_v, const float4* md_n, int mw, int mh, Intr k,
                            const float* camera12, const float* model12, float max_dist,
                            float min_dot) {
  const Maps m = make_maps(lv_v, lv_n, lw, lh, md_v, md_n, mw, mh, k);
  const int nb = blocks_for(lw * lh);
  for_batch(m, nb, [&](auto batch) {
    hipLaunchKernelGGL(icp_sweep_kernel<batch.value>, dim3(nb), dim3(256), 0, ctx->stream, m,
                       rigid_from12(camera12), rigid_from12(model12), max_dist, min_dot, ctx->partials);
  });
  hipLaunchKernelGGL(icp_combine_kernel, dim3(1), dim3(256), 0, ctx->stream, ctx->icp, ctx->partials, nb,
                     ctx->icp_mapped);
  KF_HIP(hipGetLastError());
}

static_assert(sizeof(scratch) == sizeof(float) * kMaxBlocks * kPartialStride,
              "the static partial rows hold one row per sweep workgroup");

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept.
float* static_scratch_rows() {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static float* rows[kMaxDevices] = {};
  int dev = 0;
  KF_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) fail(KF_ERR_UNSUPPORTED, "kf_icp_reduce_static: device index out of range");
  const std::lock_guard<std::mutex> lock(mu);
  if (rows[dev] == nullptr) {
    void* p = nullptr;
    KF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (p == nullptr) fail(KF_ERR_DEVICE, "kf_icp_reduce_static: no device address for the partial rows");
    rows[dev] = static_cast<float*>(p);
  }
  return rows[dev];
}

void launch_icp_reduce_static(hipStream_t stream, const float4* lv_v, const float4* lv_n, int lw, int lh,
                              const float4* md_v, const float4* md_n, int mw, int mh, Intr k,
                              const float* camera12, const float* model12, float max_dist, float min_dot,
                              double* sums, int64_t* count) {
  float* rows = static_scratch_rows();
  const Maps m = make_maps(lv_v, lv_n, lw, lh, md_v, md_n, mw, mh, k);
  const int nb = blocks_for(lw * lh);  // <= kMaxBlocks rows, every one written by the sweep
  for_batch(m, nb, [&](auto batch) {
    hipLaunchKernelGGL(icp_sweep_kernel<batch.value>, dim3(nb), dim3(256), 0, stream, m, rigid_from12(camera12),
                       rigid_from12(model12), max_dist, min_dot, rows);
  });
  hipLaunchKernelGGL(icp_combine_out_kernel, dim3(1), dim3(256), 0, stream, rows, nb, sums, count);
  KF_HIP(hipGetLastError());
}

}  // namespace kf
