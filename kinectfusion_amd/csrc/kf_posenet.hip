// Pose-proposal network for the learned ICP warm start: BF16 MFMA training
// and inference on gfx950.  The reference has no counterpart; its hook is
// the tracker's initial pose (src/app/reconstruction.cpp:218-250), and the
// fallback reads IcpNormalEquations::mean_squared_residual
// (icp_correspondence.hpp:133-139).
//
// Network: input 2 x 120 x 160 (previous and current coarsest-level depth,
// NHWC, bf16) -> five 3x3 stride-2 pad-1 convolutions with ReLU
// (16, 32, 64, 64, 128 channels; 60x80, 30x40, 15x20, 8x10, 4x5) -> flatten
// (4 * 5 * 128 = 2560, NHWC order) -> 256 with ReLU -> 6.  Input depths are
// metres minus 1.5 m (0 where invalid), which keeps bf16's 8-bit mantissa
// fine around the working range.  The output times (0.1, 0.1, 0.1, 0.03,
// 0.03, 0.03) is the twist (omega rad, t m) of the motion from the previous
// camera to the current one: T_cur = T_prev * [R(omega) | t].
//
// Every layer is one GEMM on the matrix cores (v_mfma_f32_16x16x32_bf16,
// FP32 accumulation): convolutions as im2col (K = 9 * Cin, k = (ky * 3 + kx)
// * Cin + ci) times W^T, their weight gradients as split-K GEMMs over the
// batch-pixel axis with fixed-order partial sums, input gradients as GEMMs
// followed by a gather col2im.  Master weights and Adam moments are FP32;
// the GEMM operands are bf16 copies.  Every reduction has a fixed order, so
// training is deterministic.
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "kf_internal.hpp"

namespace {

using kf::fail;

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kInH = 120, kInW = 160;
constexpr int kConv = 5;
constexpr int kCh[kConv + 1] = {2, 16, 32, 64, 64, 128};
constexpr int kHidden = 256, kOut = 6;
constexpr int kLayers = kConv + 2;
constexpr float kDepthCentre = 1.5F;  // metres
__host__ __device__ inline float out_scale(int component) { return component < 3 ? 0.1F : 0.03F; }

__host__ __device__ inline uint16_t to_bf16(float f) {  // round to nearest even
  const uint32_t b = __builtin_bit_cast(uint32_t, f);
  return static_cast<uint16_t>((b + 0x7FFFU + ((b >> 16U) & 1U)) >> 16U);
}
__host__ __device__ inline float from_bf16(uint16_t h) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(h) << 16U);
}

struct Shape {
  bool conv;
  int cin, cout, hin, win, hout, wout;
  int fan_in;         // K of the layer's GEMM
  size_t w_off, b_off;  // into the packed parameter vector
};

std::vector<Shape> network_shapes(size_t* total) {
  std::vector<Shape> s;
  int h = kInH, w = kInW;
  size_t off = 0;
  for (int l = 0; l < kConv; ++l) {
    Shape x{true, kCh[l], kCh[l + 1], h, w, (h + 1) / 2, (w + 1) / 2, 9 * kCh[l], 0, 0};
    x.w_off = off;
    off += static_cast<size_t>(x.cout) * x.fan_in;
    x.b_off = off;
    off += x.cout;
    s.push_back(x);
    h = x.hout;
    w = x.wout;
  }
  const int flat = h * w * kCh[kConv];
  Shape f1{false, flat, kHidden, 1, 1, 1, 1, flat, 0, 0};
  f1.w_off = off;
  off += static_cast<size_t>(kHidden) * flat;
  f1.b_off = off;
  off += kHidden;
  s.push_back(f1);
  Shape f2{false, kHidden, kOut, 1, 1, 1, 1, kHidden, 0, 0};
  f2.w_off = off;
  off += static_cast<size_t>(kOut) * kHidden;
  f2.b_off = off;
  off += kOut;
  s.push_back(f2);
  if (total != nullptr) *total = off;
  return s;
}

// ---------------------------------------------------------------------------
// GEMM: C(m, n) = sum_k A(m, k) B(k, n), bf16 operands with arbitrary
// strides, FP32 accumulation.  64x64 tile per 256-thread workgroup, each of
// the four waves a 32x32 quadrant of 2x2 16x16x32 MFMA blocks, K staged 32
// at a time through LDS.  gridDim.z splits K: every split writes its FP32
// partial tile and a second kernel adds the partials in split order 0, 1,
// ... and applies the epilogue, so the sum does not depend on timing.
// A 3x3 stride-2 pad-1 convolution read as its im2col matrix, element
// (m, k) = x[b][2 yo - 1 + ky][2 xo - 1 + kx][c] with m = (b Ho + yo) Wo + xo,
// k = (ky 3 + kx) C + c (0 outside the image).  With `raw_prev` set the input
// is the depth pair itself (u16, channel 0 previous, 1 current), converted as
// the input layer does.
struct ConvView {
  const uint16_t* x;
  const uint16_t* raw_prev;  // pair b at raw_prev + b * raw_stride
  const uint16_t* raw_cur;
  long long raw_stride;
  float inv_scale;
  int H, W, C, Ho, Wo;
};

struct Gemm {
  const uint16_t* a;  // null: A is the im2col matrix of `conv`
  ConvView conv;
  long long sam, sak;
  const uint16_t* b;
  long long sbk, sbn;
  int M, N, K, kchunk;
  float* partial;  // [splits][M][N] when gridDim.z > 1
  // epilogue: v (+ bias[n]) (ReLU) -> outf and/or outh
  const float* bias;
  int relu;
  float* outf;
  long long ofm, ofn;
  uint16_t* outh;
  long long ohm, ohn;
  int scale_out;  // outf receives v * out_scale(n) (the twist)
};

constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;  // 80-byte rows: 16-byte fragment reads stay aligned
static_assert(BM == 64 && BN == 64 && BK == 32, "the staging modes map 256 threads to 64 x 32 values");
constexpr int kMaxTiles = 256;                   // at most this many tiles split K

__device__ inline uint16_t raw_to_input(uint16_t r, float inv_scale) {
  return to_bf16(r == 0 ? 0.0F : static_cast<float>(r) * inv_scale - kDepthCentre);
}

__device__ inline void gemm_store(const Gemm& g, int m, int n, float v) {
  if (g.bias != nullptr) v += g.bias[n];
  if (g.relu != 0) v = fmaxf(v, 0.0F);
  if (g.outf != nullptr) g.outf[m * g.ofm + n * g.ofn] = g.scale_out != 0 ? v * out_scale(n) : v;
  if (g.outh != nullptr) g.outh[m * g.ohm + n * g.ohn] = to_bf16(v);
}

// How a workgroup stages an operand's 64 rows (m or n) x 32 k of one K step
// (eight values a thread), by what lies next to each other in memory:
//  kStageRows8   eight k of a row per 16-byte read (k contiguous, rows 16-byte aligned)
//  kStageRows2   two k per 4-byte read (k contiguous, even row length)
//  kStageCols    two rows of two k each: rows contiguous, so a read holds two rows of
//           one k, and two reads are transposed in registers (weight and input
//           gradients, whose operands are stored k-major; lanes run along the
//           rows, so a wave's reads are whole lines)
//  kStageScalar  one value at a time
//  kStageConv8   the im2col matrix of a convolution, eight channels of a tap per
//           16-byte read
//  kStageConv    the same one value at a time (the raw depth pair)
// Every address past an edge is clamped and its value zeroed: a guarded read
// would wait for the one before it.  The values and their places are the same
// in every mode, so the sums are too.
// What bounds a tile is the read round per K step.  One value at a time, lanes
// along k, the gradients of 64 pairs took 390 us in these GEMMs (56 us for the
// second layer's weight gradient, whose reads were strided); the modes take
// 155 us (18 us).
enum StageMode { kStageScalar = 0, kStageRows8, kStageRows2, kStageCols, kStageConv8, kStageConv };

template <int Mode>
struct Stage {
  uint32_t v[4];  // eight bf16 values
  // rows of thread t: kStageRows8 / kStageConv8: t / 4, k 8 (t % 4); kStageRows2: t / 16 + 16 i, k 2 (t % 16);
  // kStageCols: 2 (t % 32), 2 (t % 32) + 1, k 2 (t / 32) + 16 i; kStageScalar / kStageConv: t / 32 + 8 i, k t % 32
  __device__ inline void read(const uint16_t* p, long long srow, long long sk, int row0, int rows, int k0, int ke,
                              const ConvView& cv, const int* org) {
    const int t = static_cast<int>(threadIdx.x);
    if constexpr (Mode == kStageRows8) {
      const int r = row0 + (t >> 2), k = k0 + (t & 3) * 8;
      // ke is a multiple of 8 (the host's check), so the eight lie inside or outside together
      const uint4 q = *reinterpret_cast<const uint4*>(p + min(r, rows - 1) * srow + min(k, ke - 8));
      const bool in = r < rows && k < ke;
      v[0] = in ? q.x : 0U;
      v[1] = in ? q.y : 0U;
      v[2] = in ? q.z : 0U;
      v[3] = in ? q.w : 0U;
    } else if constexpr (Mode == kStageRows2) {
      const int k = k0 + (t & 15) * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = *reinterpret_cast<const uint32_t*>(p + min(row0 + (t >> 4) + 16 * i, rows - 1) * srow + min(k, ke - 2));
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = row0 + (t >> 4) + 16 * i < rows && k < ke ? v[i] : 0U;
    } else if constexpr (Mode == kStageCols) {
      const int r = row0 + (t & 31) * 2;
      const uint16_t* base = p + min(r, rows - 2);  // rows is even
      uint32_t q[4];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          q[2 * i + j] = *reinterpret_cast<const uint32_t*>(base + min(k0 + (t >> 5) * 2 + 16 * i + j, ke - 1) * sk);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int k = k0 + (t >> 5) * 2 + 16 * i;
        const uint32_t a = r < rows && k < ke ? q[2 * i] : 0U, b = r < rows && k + 1 < ke ? q[2 * i + 1] : 0U;
        v[2 * i] = (a & 0xFFFFU) | (b << 16);      // row r, k and k + 1
        v[2 * i + 1] = (a >> 16) | (b & 0xFFFF0000U);  // row r + 1
      }
    } else if constexpr (Mode == kStageConv8) {
      // org: the receptive-field origin (oy, ox, pair) of this thread's row
      const int k = k0 + (t & 3) * 8, kc = min(k, ke - 8);
      const int tap = kc / cv.C, ch = kc - tap * cv.C, ky = tap / 3, kx = tap - ky * 3;
      const int yi = org[0] + ky, xi = org[1] + kx;
      const int yc = min(max(yi, 0), cv.H - 1), xc = min(max(xi, 0), cv.W - 1);
      const uint4 q = *reinterpret_cast<const uint4*>(
          cv.x + ((static_cast<long long>(org[2]) * cv.H + yc) * cv.W + xc) * cv.C + ch);
      const bool in = k < ke && yi == yc && xi == xc;
      v[0] = in ? q.x : 0U;
      v[1] = in ? q.y : 0U;
      v[2] = in ? q.z : 0U;
      v[3] = in ? q.w : 0U;
    } else {
      const int k = k0 + (t & 31), kc = min(k, ke - 1);
      uint16_t h[8];
      int ky = 0, kx = 0, ch = 0;
      if constexpr (Mode == kStageConv) {
        const int tap = kc / cv.C;
        ch = kc - tap * cv.C;
        ky = tap / 3;
        kx = tap - ky * 3;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (Mode == kStageConv) {
          const int yc = min(max(org[3 * i] + ky, 0), cv.H - 1), xc = min(max(org[3 * i + 1] + kx, 0), cv.W - 1);
          if (cv.raw_prev != nullptr)
            h[i] = (ch == 0 ? cv.raw_prev : cv.raw_cur)[org[3 * i + 2] * cv.raw_stride + yc * cv.W + xc];
          else
            h[i] = cv.x[((static_cast<long long>(org[3 * i + 2]) * cv.H + yc) * cv.W + xc) * cv.C + ch];
        } else {
          h[i] = p[min(row0 + (t >> 5) + 8 * i, rows - 1) * srow + kc * sk];
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        bool in = k < ke && row0 + (t >> 5) + 8 * i < rows;
        if constexpr (Mode == kStageConv) {
          const int yi = org[3 * i] + ky, xi = org[3 * i + 1] + kx;
          in = k < ke && yi >= 0 && yi < cv.H && xi >= 0 && xi < cv.W;
          if (cv.raw_prev != nullptr) h[i] = raw_to_input(h[i], cv.inv_scale);
        }
        h[i] = in ? h[i] : static_cast<uint16_t>(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = h[2 * i] | (static_cast<uint32_t>(h[2 * i + 1]) << 16);
    }
  }
  __device__ inline void write(uint16_t (*lds)[LDK]) const {
    const int t = static_cast<int>(threadIdx.x);
    if constexpr (Mode == kStageRows8 || Mode == kStageConv8) {
      *reinterpret_cast<uint4*>(&lds[t >> 2][(t & 3) * 8]) = make_uint4(v[0], v[1], v[2], v[3]);
    } else if constexpr (Mode == kStageRows2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint32_t*>(&lds[(t >> 4) + 16 * i][(t & 15) * 2]) = v[i];
    } else if constexpr (Mode == kStageCols) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          *reinterpret_cast<uint32_t*>(&lds[(t & 31) * 2 + j][(t >> 5) * 2 + 16 * i]) = v[2 * i + j];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        lds[(t >> 5) + 8 * i][t & 31] = static_cast<uint16_t>((i & 1) != 0 ? v[i >> 1] >> 16 : v[i >> 1]);
    }
  }
};

template <int ModeA, int ModeB>
__global__ void __launch_bounds__(256) gemm_kernel(Gemm g) {
  __shared__ __align__(16) uint16_t As[BM][LDK];
  __shared__ __align__(16) uint16_t Bs[BN][LDK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int kb = blockIdx.z * g.kchunk;
  const int ke = min(g.K, kb + g.kchunk);
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int li = lane & 15, lq = lane >> 4;
  // im2col: the receptive-field origin of this thread's rows is fixed over
  // the K loop (rows past M get an origin no tap reaches)
  constexpr int kOrigins = ModeA == kStageConv ? 8 : 1;
  int org[3 * kOrigins];
  if constexpr (ModeA == kStageConv || ModeA == kStageConv8) {
#pragma unroll
    for (int i = 0; i < kOrigins; ++i) {
      const int m = m0 + (ModeA == kStageConv ? (tid >> 5) + 8 * i : tid >> 2);
      org[3 * i] = org[3 * i + 1] = -4;
      org[3 * i + 2] = 0;
      if (m < g.M) {
        const int xo = m % g.conv.Wo, t = m / g.conv.Wo;
        org[3 * i] = 2 * (t % g.conv.Ho) - 1;
        org[3 * i + 1] = 2 * xo - 1;
        org[3 * i + 2] = t / g.conv.Ho;
      }
    }
  }
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0F, 0.0F, 0.0F, 0.0F};
  Stage<ModeA> sa;
  Stage<ModeB> sb;
  sa.read(g.a, g.sam, g.sak, m0, g.M, kb, ke, g.conv, org);
  sb.read(g.b, g.sbn, g.sbk, n0, g.N, kb, ke, g.conv, org);
  for (int k0 = kb; k0 < ke; k0 += BK) {
    sa.write(As);
    sb.write(Bs);
    __syncthreads();
    if (k0 + BK < ke) {  // the next step's reads run behind this step's MFMAs
      sa.read(g.a, g.sam, g.sak, m0, g.M, k0 + BK, ke, g.conv, org);
      sb.read(g.b, g.sbn, g.sbk, n0, g.N, k0 + BK, ke, g.conv, org);
    }
    {  // the staged 32 k as one 16x16x32 step
      s16x8 af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[i] = *reinterpret_cast<const s16x8*>(&As[wm + i * 16 + li][lq * 8]);
        bf[i] = *reinterpret_cast<const s16x8*>(&Bs[wn + i * 16 + li][lq * 8]);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[i]),
                                                              __builtin_bit_cast(bf16x8, bf[j]), acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // lane holds D[4 * lq + r][li] of each 16x16 block
  const bool split = gridDim.z > 1;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + lq * 4 + r, n = n0 + wn + j * 16 + li;
        if (m >= g.M || n >= g.N) continue;
        if (split) {
          g.partial[(static_cast<size_t>(blockIdx.z) * g.M + m) * g.N + n] = acc[i][j][r];
        } else {
          gemm_store(g, m, n, acc[i][j][r]);
        }
      }
}

// Sum of the split partials in split order 0, 1, ... (sixteen reads in
// flight per thread), then the epilogue.
__global__ void gemm_finish_kernel(Gemm g, int splits) {
  const long long total = static_cast<long long>(g.M) * g.N;
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const float* p = g.partial + i;
  float s = 0.0F;
  constexpr int kRun = 16;
  for (int z = 0; z < splits; z += kRun) {
    float v[kRun];
#pragma unroll
    for (int j = 0; j < kRun; ++j) v[j] = p[min(z + j, splits - 1) * total];
#pragma unroll
    for (int j = 0; j < kRun; ++j) s += z + j < splits ? v[j] : 0.0F;  // + 0 past the end leaves the sum as it is
  }
  gemm_store(g, static_cast<int>(i / g.N), static_cast<int>(i % g.N), s);
}

// Sums down the columns of x[rows][n], the rows in order 0, 1, ...: the order
// is serial per column, so the reads must not be.  A workgroup stages its 32
// columns 256 rows at a time in LDS (32 reads per thread in flight, the next
// piece's reads issued before this one is added) and one thread per column
// adds them.  A thread per column reading its rows itself took 175 us for
// 1200 rows of 16 columns; this takes 12 us.
constexpr int kSumCols = 32, kSumRows = 256;
struct RowSum {
  const float* x;
  int rows, n;
};
template <typename Store>
__device__ inline void row_sum(const RowSum& r, int c0, Store&& store) {
  __shared__ float piece[kSumRows][kSumCols + 1];
  constexpr int kReads = kSumRows * kSumCols / 256;
  const int col = threadIdx.x & (kSumCols - 1), row = threadIdx.x / kSumCols;
  const bool in = c0 + col < r.n;
  float v[kReads];
  auto read = [&](int r0) {
#pragma unroll
    for (int j = 0; j < kReads; ++j) {
      // clamped, not skipped: a guarded read would wait for the one before
      v[j] = r.x[static_cast<long long>(min(r0 + row + j * (256 / kSumCols), r.rows - 1)) * r.n + min(c0 + col, r.n - 1)];
    }
  };
  float s = 0.0F;
  read(0);
  for (int r0 = 0; r0 < r.rows; r0 += kSumRows) {
#pragma unroll
    for (int j = 0; j < kReads; ++j) piece[row + j * (256 / kSumCols)][col] = v[j];
    __syncthreads();
    if (r0 + kSumRows < r.rows) read(r0 + kSumRows);
    if (threadIdx.x < kSumCols) {
      const int n = min(kSumRows, r.rows - r0);
#pragma unroll 16
      for (int i = 0; i < n; ++i) s += piece[i][threadIdx.x];
    }
    __syncthreads();
  }
  if (threadIdx.x < kSumCols && in) store(c0 + col, s);
}

// The split partials of a long reduction (more splits than one piece's worth
// of reads in flight per thread), then the epilogue.
__global__ void __launch_bounds__(256) gemm_finish_rows_kernel(Gemm g, int splits) {
  row_sum(RowSum{g.partial, splits, g.M * g.N}, static_cast<int>(blockIdx.x) * kSumCols,
          [&](int i, float s) { gemm_store(g, i / g.N, i % g.N, s); });
}

// ---------------------------------------------------------------------------
// Small GEMM (few output tiles, K up to a few thousand: the layers of a pose
// proposal, and the forward layers of small batches).  One workgroup per
// 16 x 16 output tile; its Waves waves (8, or 16 for long reductions) split
// the K steps (32 wide: v_mfma_f32_16x16x32_bf16, gfx950's bf16 shape)
// between them and load their operand fragments straight from global memory
// into registers, kSmallChunk steps at a time, so that a layer costs one or
// two memory round trips instead of one per K step.  Lane l holds
// A[l % 16][8 (l / 16) + j] and B[8 (l / 16) + j][l % 16] (j = 0..7) of a
// step and D[4 (l / 16) + r][l % 16] of the tile.  The per-wave tiles are
// added in wave order through LDS, so the result does not depend on timing.
constexpr int kSmallChunk = 5;

// A(m, k) of the im2col matrix for a row whose receptive-field origin is
// (oy, ox) of pair ob (oy < -2 marks a row past M).
__device__ inline uint16_t conv_a(const ConvView& v, int oy, int ox, int ob, int k) {
  const int tap = k / v.C, ch = k - tap * v.C;
  const int ky = tap / 3, kx = tap - ky * 3;
  const int yi = oy + ky, xi = ox + kx;
  if (yi < 0 || yi >= v.H || xi < 0 || xi >= v.W) return 0;
  if (v.raw_prev != nullptr) {
    const uint16_t* src = ch == 0 ? v.raw_prev : v.raw_cur;
    return raw_to_input(src[ob * v.raw_stride + yi * v.W + xi], v.inv_scale);
  }
  return v.x[((static_cast<long long>(ob) * v.H + yi) * v.W + xi) * v.C + ch];
}

__device__ inline short as_short(uint16_t h) { return static_cast<short>(h); }

template <int Waves>
__global__ void __launch_bounds__(Waves * 64) gemm_small_kernel(Gemm g, int vec_a, int vec_b) {
  __shared__ float red[Waves][16][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lq = lane >> 4;
  const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  const int m = m0 + li, n = n0 + li;  // this lane's A row and B column
  const bool mok = m < g.M, nok = n < g.N;
  const bool implicit = g.a == nullptr;
  int oy = -4, ox = -4, ob = 0;
  if (implicit && mok) {
    const int xo = m % g.conv.Wo, t = m / g.conv.Wo;
    oy = 2 * (t % g.conv.Ho) - 1;
    ox = 2 * xo - 1;
    ob = t / g.conv.Ho;
  }
  const int steps = (g.K + 31) / 32;
  const int per = (steps + Waves - 1) / Waves;
  const int s_begin = wave * per, s_end = min(steps, s_begin + per);
  f32x4 acc = f32x4{0.0F, 0.0F, 0.0F, 0.0F};
  for (int c0 = s_begin; c0 < s_end; c0 += kSmallChunk) {
    s16x8 af[kSmallChunk], bfr[kSmallChunk];
#pragma unroll
    for (int c = 0; c < kSmallChunk; ++c) {
      af[c] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      bfr[c] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      const int k = (c0 + c) * 32 + lq * 8;
      if (c0 + c >= s_end || k >= g.K) continue;
      const bool full = k + 7 < g.K;
      if (mok) {
        if (implicit) {
          if (vec_a != 0 && full) {
            // C % 8 == 0: the eight k are channels ch..ch+7 of one tap
            const int tap = k / g.conv.C, ch = k - tap * g.conv.C;
            const int ky = tap / 3, kx = tap - ky * 3;
            const int yi = oy + ky, xi = ox + kx;
            if (yi >= 0 && yi < g.conv.H && xi >= 0 && xi < g.conv.W) {
              af[c] = *reinterpret_cast<const s16x8*>(
                  g.conv.x + ((static_cast<long long>(ob) * g.conv.H + yi) * g.conv.W + xi) * g.conv.C + ch);
            }
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (k + j < g.K) af[c][j] = as_short(conv_a(g.conv, oy, ox, ob, k + j));
          }
        } else if (vec_a != 0 && full) {
          af[c] = *reinterpret_cast<const s16x8*>(g.a + m * g.sam + k);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {  // clamped and zeroed: guarded reads would wait for one another
            const short v = as_short(g.a[m * g.sam + min(k + j, g.K - 1) * g.sak]);
            af[c][j] = k + j < g.K ? v : short{0};
          }
        }
      }
      if (nok) {
        if (vec_b != 0 && full) {
          bfr[c] = *reinterpret_cast<const s16x8*>(g.b + n * g.sbn + k);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const short v = as_short(g.b[min(k + j, g.K - 1) * g.sbk + n * g.sbn]);
            bfr[c][j] = k + j < g.K ? v : short{0};
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kSmallChunk; ++c)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[c]), __builtin_bit_cast(bf16x8, bfr[c]),
                                                    acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lq * 4 + r][li] = acc[r];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const int om = m0 + row, on = n0 + col;
    if (om < g.M && on < g.N) {
      float s = 0.0F;
#pragma unroll
      for (int w = 0; w < Waves; ++w) s += red[w][row][col];
      gemm_store(g, om, on, s);
    }
  }
}

// ---------------------------------------------------------------------------
// Depth pair -> NHWC bf16 centred metres.  pair b: prev = prev0 + b * stride,
// cur = cur0 + b * stride (u16 raw, 160 x 120 each).
__global__ void input_kernel(const uint16_t* prev0, const uint16_t* cur0, long long stride, int batch,
                             float inv_scale, uint16_t* x0) {
  const int px = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (px >= kInH * kInW || b >= batch) return;
  const uint16_t rp = prev0[b * stride + px], rc = cur0[b * stride + px];
  const float p = rp == 0 ? 0.0F : static_cast<float>(rp) * inv_scale - kDepthCentre;
  const float c = rc == 0 ? 0.0F : static_cast<float>(rc) * inv_scale - kDepthCentre;
  const size_t o = (static_cast<size_t>(b) * kInH * kInW + px) * 2;
  x0[o] = to_bf16(p);
  x0[o + 1] = to_bf16(c);
}

// col[m][k]: m = (b * Ho + yo) * Wo + xo, k = (ky * 3 + kx) * C + c.  Run
// consecutive channels of one tap per thread as one word (2 channels: 4 bytes,
// otherwise 8: 16 bytes), so a thread's index divisions are paid once per word.
template <int Run>
using Channels = std::conditional_t<Run == 8, uint4, uint32_t>;
template <int Run>
__global__ void __launch_bounds__(256) im2col_kernel(const uint16_t* x, uint16_t* col, int batch, int H, int W, int C,
                                                     int Ho, int Wo) {
  const unsigned per = static_cast<unsigned>(9 * C / Run), groups = static_cast<unsigned>(C / Run);
  const unsigned total = static_cast<unsigned>(batch * Ho * Wo) * per;  // < 2^32: at most 4096 x 4800 x 18
  for (unsigned e = blockIdx.x * 256U + threadIdx.x; e < total; e += gridDim.x * 256U) {
    const unsigned m = e / per, r = e - m * per;
    const int tap = static_cast<int>(r / groups), c = static_cast<int>(r - tap * groups) * Run;
    const int ky = tap / 3, kx = tap - ky * 3;
    const unsigned t = m / static_cast<unsigned>(Wo);
    const int xo = static_cast<int>(m - t * Wo), b = static_cast<int>(t / static_cast<unsigned>(Ho));
    const int yo = static_cast<int>(t) - b * Ho;
    const int yi = 2 * yo - 1 + ky, xi = 2 * xo - 1 + kx;
    const int yc = min(max(yi, 0), H - 1), xc = min(max(xi, 0), W - 1);
    Channels<Run> v = *reinterpret_cast<const Channels<Run>*>(x + ((static_cast<size_t>(b) * H + yc) * W + xc) * C + c);
    if (yi != yc || xi != xc) v = Channels<Run>{};
    reinterpret_cast<Channels<Run>*>(col)[e] = v;
  }
}

// dx[b][yi][xi][c] = sum over the taps that read it of dcol, in (ky, kx)
// order, times the ReLU mask of the layer input; bf16 out.  Four channels per
// thread (C is a multiple of 16); at most four taps read a pixel, and their
// reads are issued together.
__global__ void __launch_bounds__(256) col2im_kernel(const float* dcol, const uint16_t* xin, uint16_t* dx, int batch,
                                                     int H, int W, int C, int Ho, int Wo) {
  const unsigned groups = static_cast<unsigned>(C / 4);
  const unsigned total = static_cast<unsigned>(batch * H * W) * groups;
  for (unsigned e = blockIdx.x * 256U + threadIdx.x; e < total; e += gridDim.x * 256U) {
    const unsigned p = e / groups;
    const int c = static_cast<int>(e - p * groups) * 4;
    const unsigned t = p / static_cast<unsigned>(W);
    const int xi = static_cast<int>(p - t * W), b = static_cast<int>(t / static_cast<unsigned>(H));
    const int yi = static_cast<int>(t) - b * H;
    // taps with (yi + 1 - ky) even: ky = 1, or 0 and 2; along x alike
    const int ky0 = (yi & 1) != 0 ? 0 : 1, kx0 = (xi & 1) != 0 ? 0 : 1;
    float4 v[2][2];
    bool in[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int ky = ky0 + 2 * i, kx = kx0 + 2 * j, ty = yi + 1 - ky, tx = xi + 1 - kx;
        in[i][j] = ky < 3 && kx < 3 && ty >= 0 && (ty >> 1) < Ho && tx >= 0 && (tx >> 1) < Wo;
        const size_t m = in[i][j] ? (static_cast<size_t>(b) * Ho + (ty >> 1)) * Wo + (tx >> 1) : 0;
        const int tap = in[i][j] ? ky * 3 + kx : 0;
        v[i][j] = *reinterpret_cast<const float4*>(dcol + (m * 9 + tap) * C + c);
      }
    const uint2 act = reinterpret_cast<const uint2*>(xin)[e];
    float s[4] = {0.0F, 0.0F, 0.0F, 0.0F};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (!in[i][j]) continue;
        s[0] += v[i][j].x;
        s[1] += v[i][j].y;
        s[2] += v[i][j].z;
        s[3] += v[i][j].w;
      }
    auto masked = [](uint32_t a, float v) -> uint32_t {
      return to_bf16(from_bf16(static_cast<uint16_t>(a)) > 0.0F ? v : 0.0F);
    };
    reinterpret_cast<uint2*>(dx)[e] = make_uint2(masked(act.x, s[0]) | (masked(act.x >> 16, s[1]) << 16),
                                                 masked(act.y, s[2]) | (masked(act.y >> 16, s[3]) << 16));
  }
}

// out = act > 0 ? bf16(g) : 0
__global__ void relu_mask_kernel(const float* g, const uint16_t* act, uint16_t* out, long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = from_bf16(act[i]) > 0.0F ? to_bf16(g[i]) : static_cast<uint16_t>(0);
}

// Mean squared error against the targets divided by the output scale; its
// gradient as bf16.
// One workgroup, fixed-order tree.
__global__ void __launch_bounds__(256) loss_kernel(const float* out, const float* target, int batch,
                                                   uint16_t* dout, float* loss) {
  __shared__ float red[256];
  const int n = batch * kOut;
  const float inv = 1.0F / static_cast<float>(n);
  float s = 0.0F;
  for (int i = threadIdx.x; i < n; i += 256) {
    const float d = out[i] - target[i] / out_scale(i % kOut);
    s += d * d;
    dout[i] = to_bf16(2.0F * d * inv);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = red[0] * inv;
}

// Column sums of a bf16 [M][N] matrix (bias gradients), two passes with a
// fixed order: chunks of 256 rows, then the chunks.
constexpr int kColRows = 256;
__global__ void __launch_bounds__(256) colsum_chunk_kernel(const uint16_t* x, int M, int N, float* part) {
  __shared__ float red[256];
  const int r0 = blockIdx.x * kColRows, r1 = min(M, r0 + kColRows);
  for (int nb = 0; nb < N; nb += 256) {
    const int cols = min(256, N - nb);
    const int groups = 256 / cols;  // row lanes per column
    const int col = threadIdx.x % cols, grp = threadIdx.x / cols;
    float s = 0.0F;
    if (grp < groups) {
      // sixteen rows in flight, added in row order
      constexpr int kRun = 16;
      for (int r = r0 + grp; r < r1; r += kRun * groups) {
        uint16_t v[kRun];
#pragma unroll
        for (int j = 0; j < kRun; ++j) {
          // clamped, not skipped: a guarded read would wait for the one before
          v[j] = x[static_cast<long long>(min(r + j * groups, r1 - 1)) * N + nb + col];
        }
#pragma unroll
        for (int j = 0; j < kRun; ++j) s += r + j * groups < r1 ? from_bf16(v[j]) : 0.0F;  // + 0 past the end
      }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < cols) {
      float t = 0.0F;
      for (int q = 0; q < groups; ++q) t += red[q * cols + threadIdx.x];
      part[static_cast<long long>(blockIdx.x) * N + nb + threadIdx.x] = t;
    }
    __syncthreads();
  }
}
// The chunks of every layer's bias sum in one launch (blockIdx.y: the layer):
// seven launches of a few microseconds' latency each took 27 us of a batch's
// 540.
constexpr int kLayerSums = kConv + 2;
struct LayerSum {
  RowSum chunks;
  float* out;
};
struct LayerSums {
  LayerSum sum[kLayerSums];
  int count;
  size_t used;  // floats of the chunks' buffer
};
__global__ void __launch_bounds__(256) colsum_final_kernel(LayerSums all) {
  const LayerSum& l = all.sum[blockIdx.y];
  const int c0 = static_cast<int>(blockIdx.x) * kSumCols;
  if (c0 >= l.chunks.n) return;
  row_sum(l.chunks, c0, [&](int c, float s) { l.out[c] = s; });
}

__global__ void adam_kernel(float* w, const float* g, float* m, float* v, uint16_t* wh, long long n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0F - b1) * gi;
  const float vi = b2 * v[i] + (1.0F - b2) * (gi * gi);
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  w[i] = wi;
  wh[i] = to_bf16(wi);
}

__global__ void to_bf16_kernel(const float* w, uint16_t* wh, long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) wh[i] = to_bf16(w[i]);
}


int blocks_for(long long n, int per = 256) { return static_cast<int>((n + per - 1) / per); }

}  // namespace

// ---------------------------------------------------------------------------
struct kf_posenet {
  kf_posenet_config cfg{};
  std::string error;
  kf::HostStage stage;
  hipStream_t stream = nullptr;
  std::vector<Shape> shapes;
  size_t n_params = 0;
  float* w = nullptr;      // FP32 master
  float* grad = nullptr;
  float* m = nullptr;
  float* v = nullptr;
  uint16_t* wh = nullptr;  // bf16 copy used by the GEMMs
  uint16_t* act[kLayers] = {};  // act[0] input, act[l + 1] output of layer l (bf16); fc2 output is `out`
  uint16_t* col[kConv] = {};
  float* out = nullptr;    // [capacity][6] network output (normalised twist)
  float* tmp = nullptr;    // FP32 GEMM outputs of the backward pass
  uint16_t* dz[2] = {};    // bf16 gradients of layer outputs
  float* partial = nullptr;
  size_t partial_floats = 0;
  float* colpart = nullptr;
  float* loss = nullptr;   // device scalar
  float* loss_host = nullptr;  // pinned
  long long step = 0;
};

namespace {

template <typename T>
T* nalloc(size_t count) {
  void* p = nullptr;
  KF_HIP(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)));
  return static_cast<T*>(p);
}

// The staging mode of an operand with row stride srow and k stride sk over
// `rows` rows and K (a kchunk is a multiple of 32, so K decides the k edges): the widest
// read that the order, strides and alignment allow.
int stage_mode(const uint16_t* p, long long srow, long long sk, int rows, int K) {
  const auto at = reinterpret_cast<uintptr_t>(p);
  if (sk == 1 && srow % 8 == 0 && K % 8 == 0 && (at & 15U) == 0U) return kStageRows8;
  if (sk == 1 && srow % 2 == 0 && K % 2 == 0 && (at & 3U) == 0U) return kStageRows2;
  if (srow == 1 && sk % 2 == 0 && rows % 2 == 0 && (at & 3U) == 0U) return kStageCols;
  return kStageScalar;
}

template <int ModeA>
void launch_gemm_b(const Gemm& g, int mode_b, dim3 grid, hipStream_t s) {
  switch (mode_b) {
    case kStageRows8:
      hipLaunchKernelGGL((gemm_kernel<ModeA, kStageRows8>), grid, dim3(256), 0, s, g);
      break;
    case kStageRows2:
      hipLaunchKernelGGL((gemm_kernel<ModeA, kStageRows2>), grid, dim3(256), 0, s, g);
      break;
    case kStageCols:
      hipLaunchKernelGGL((gemm_kernel<ModeA, kStageCols>), grid, dim3(256), 0, s, g);
      break;
    default:
      hipLaunchKernelGGL((gemm_kernel<ModeA, kStageScalar>), grid, dim3(256), 0, s, g);
      break;
  }
}

void launch_gemm(const Gemm& g, dim3 grid, hipStream_t s) {
  const int mode_b = stage_mode(g.b, g.sbn, g.sbk, g.N, g.K);
  if (g.a == nullptr) {
    const bool vec = g.conv.raw_prev == nullptr && g.conv.C % 8 == 0 && (reinterpret_cast<uintptr_t>(g.conv.x) & 15U) == 0U;
    if (vec) launch_gemm_b<kStageConv8>(g, mode_b, grid, s);
    else launch_gemm_b<kStageConv>(g, mode_b, grid, s);
    return;
  }
  switch (stage_mode(g.a, g.sam, g.sak, g.M, g.K)) {
    case kStageRows8:
      launch_gemm_b<kStageRows8>(g, mode_b, grid, s);
      break;
    case kStageRows2:
      launch_gemm_b<kStageRows2>(g, mode_b, grid, s);
      break;
    case kStageCols:
      launch_gemm_b<kStageCols>(g, mode_b, grid, s);
      break;
    default:
      launch_gemm_b<kStageScalar>(g, mode_b, grid, s);
      break;
  }
}

void gemm(kf_posenet* net, hipStream_t s, Gemm g) {
  const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
  const int tiles = tm * tn;
  if (tiles <= 128 && g.K <= 4096) {
    // vector fragment loads need eight consecutive k in memory, 16-byte aligned
    auto aligned16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15U) == 0U; };
    int vec_a = 0;
    if (g.a == nullptr) {
      vec_a = g.conv.raw_prev == nullptr && g.conv.C % 8 == 0 && aligned16(g.conv.x) ? 1 : 0;
    } else {
      vec_a = g.sak == 1 && g.sam % 8 == 0 && aligned16(g.a) ? 1 : 0;
    }
    const int vec_b = g.sbk == 1 && g.sbn % 8 == 0 && aligned16(g.b) ? 1 : 0;
    g.partial = nullptr;
    // a reduction longer than 8 waves x kSmallChunk steps (fc1: K = 2560) takes 16 waves: one read round
    const dim3 grid((g.M + 15) / 16, (g.N + 15) / 16);
    if ((g.K + 31) / 32 > 8 * kSmallChunk) {
      hipLaunchKernelGGL(gemm_small_kernel<16>, grid, dim3(16 * 64), 0, s, g, vec_a, vec_b);
    } else {
      hipLaunchKernelGGL(gemm_small_kernel<8>, grid, dim3(8 * 64), 0, s, g, vec_a, vec_b);
    }
    KF_HIP(hipGetLastError());
    return;
  }
  // Few tiles and a long reduction: split K until about 512 workgroups run,
  // each over as little as one K step (the loop is latency bound at these
  // sizes: one pose proposal is a handful of tiles per layer).
  int splits = 1;
  if (tiles <= kMaxTiles && g.K > 2 * BK) {
    splits = std::min((g.K + BK - 1) / BK, (512 + tiles - 1) / tiles);
    const size_t cap = net->partial_floats / (static_cast<size_t>(g.M) * g.N);
    splits = static_cast<int>(std::min<size_t>(static_cast<size_t>(splits), std::max<size_t>(cap, 1)));
  }
  g.kchunk = ((g.K + splits - 1) / splits + BK - 1) / BK * BK;
  splits = (g.K + g.kchunk - 1) / g.kchunk;
  g.partial = splits > 1 ? net->partial : nullptr;
  launch_gemm(g, dim3(tm, tn, splits), s);
  if (splits > 1) {
    const long long total = static_cast<long long>(g.M) * g.N;
    // few outputs with many splits (a lone tile has up to 512): staged, 288
    // outputs 6.5 us for 21.4, 4608 4.6 for 8.7, 18432 4.1 for 7.0; otherwise a
    // thread per output, 268800 outputs 4.4 us for 19.0.  Gradients of 64 pairs
    // take 498 us so, 521 to 538 with a thread per output always, 505 with the
    // line at 16 splits.
    if (splits > 64)
      hipLaunchKernelGGL(gemm_finish_rows_kernel, dim3(blocks_for(total, kSumCols)), dim3(256), 0, s, g, splits);
    else
      hipLaunchKernelGGL(gemm_finish_kernel, dim3(blocks_for(total)), dim3(256), 0, s, g, splits);
  }
  KF_HIP(hipGetLastError());
}

Gemm make_gemm(const uint16_t* a, long long sam, long long sak, const uint16_t* b, long long sbk, long long sbn,
               int M, int N, int K) {
  Gemm g{};
  g.a = a;
  g.sam = sam;
  g.sak = sak;
  g.b = b;
  g.sbk = sbk;
  g.sbn = sbn;
  g.M = M;
  g.N = N;
  g.K = K;
  return g;
}

int col_chunks(long long rows) { return static_cast<int>((rows + kColRows - 1) / kColRows); }

// The chunks of a layer's bias sum; colsum_end adds those of all layers.
void colsum(kf_posenet* net, hipStream_t s, const uint16_t* x, int M, int N, float* out, LayerSums& sums) {
  const int chunks = col_chunks(M);
  float* part = net->colpart + sums.used;
  hipLaunchKernelGGL(colsum_chunk_kernel, dim3(chunks), dim3(256), 0, s, x, M, N, part);
  KF_HIP(hipGetLastError());
  sums.sum[sums.count++] = LayerSum{RowSum{part, chunks, N}, out};
  sums.used += static_cast<size_t>(chunks) * N;
}

void colsum_end(hipStream_t s, const LayerSums& sums) {
  int widest = 0;
  for (int i = 0; i < sums.count; ++i) widest = std::max(widest, sums.sum[i].chunks.n);
  hipLaunchKernelGGL(colsum_final_kernel, dim3(blocks_for(widest, kSumCols), sums.count), dim3(256), 0, s, sums);
  KF_HIP(hipGetLastError());
}

int pixels(const Shape& sh) { return sh.hout * sh.wout; }

// Forward pass over act[0] (already filled) for `batch` pairs.
void forward(kf_posenet* net, hipStream_t s, int batch) {
  for (int l = 0; l < kConv; ++l) {
    const Shape& sh = net->shapes[l];
    const int M = batch * pixels(sh), K = sh.fan_in;
    const long long total = static_cast<long long>(M) * K;
    if (sh.cin % 8 == 0)
      hipLaunchKernelGGL(im2col_kernel<8>, dim3(std::min(blocks_for(total / 8), 8192)), dim3(256), 0, s, net->act[l],
                         net->col[l], batch, sh.hin, sh.win, sh.cin, sh.hout, sh.wout);
    else
      hipLaunchKernelGGL(im2col_kernel<2>, dim3(std::min(blocks_for(total / 2), 8192)), dim3(256), 0, s, net->act[l],
                         net->col[l], batch, sh.hin, sh.win, sh.cin, sh.hout, sh.wout);
    Gemm g = make_gemm(net->col[l], K, 1, net->wh + sh.w_off, 1, K, M, sh.cout, K);
    g.bias = net->w + sh.b_off;
    g.relu = 1;
    g.outh = net->act[l + 1];
    g.ohm = sh.cout;
    g.ohn = 1;
    gemm(net, s, g);
  }
  const Shape& f1 = net->shapes[kConv];
  Gemm g1 = make_gemm(net->act[kConv], f1.fan_in, 1, net->wh + f1.w_off, 1, f1.fan_in, batch, f1.cout, f1.fan_in);
  g1.bias = net->w + f1.b_off;
  g1.relu = 1;
  g1.outh = net->act[kConv + 1];
  g1.ohm = f1.cout;
  g1.ohn = 1;
  gemm(net, s, g1);
  const Shape& f2 = net->shapes[kConv + 1];
  Gemm g2 = make_gemm(net->act[kConv + 1], f2.fan_in, 1, net->wh + f2.w_off, 1, f2.fan_in, batch, f2.cout,
                      f2.fan_in);
  g2.bias = net->w + f2.b_off;
  g2.outf = net->out;
  g2.ofm = kOut;
  g2.ofn = 1;
  gemm(net, s, g2);
}

// Loss and gradients of every parameter into net->grad.
void backward(kf_posenet* net, hipStream_t s, const float* targets, int batch) {
  hipLaunchKernelGGL(loss_kernel, dim3(1), dim3(256), 0, s, net->out, targets, batch, net->dz[0], net->loss);
  KF_HIP(hipGetLastError());
  LayerSums sums{};
  // fc2: dW = dout^T h, db = colsum(dout), dh = dout W masked by h > 0
  const Shape& f2 = net->shapes[kConv + 1];
  const uint16_t* h = net->act[kConv + 1];
  {
    Gemm g = make_gemm(net->dz[0], 1, kOut, h, f2.fan_in, 1, kOut, f2.fan_in, batch);
    g.outf = net->grad + f2.w_off;
    g.ofm = f2.fan_in;
    g.ofn = 1;
    gemm(net, s, g);
    colsum(net, s, net->dz[0], batch, kOut, net->grad + f2.b_off, sums);
    Gemm d = make_gemm(net->dz[0], kOut, 1, net->wh + f2.w_off, f2.fan_in, 1, batch, f2.fan_in, kOut);
    d.outf = net->tmp;
    d.ofm = f2.fan_in;
    d.ofn = 1;
    gemm(net, s, d);
    const long long n = static_cast<long long>(batch) * f2.fan_in;
    hipLaunchKernelGGL(relu_mask_kernel, dim3(blocks_for(n)), dim3(256), 0, s, net->tmp, h, net->dz[1], n);
  }
  // fc1
  const Shape& f1 = net->shapes[kConv];
  const uint16_t* x5 = net->act[kConv];
  {
    Gemm g = make_gemm(net->dz[1], 1, f1.cout, x5, f1.fan_in, 1, f1.cout, f1.fan_in, batch);
    g.outf = net->grad + f1.w_off;
    g.ofm = f1.fan_in;
    g.ofn = 1;
    gemm(net, s, g);
    colsum(net, s, net->dz[1], batch, f1.cout, net->grad + f1.b_off, sums);
    Gemm d = make_gemm(net->dz[1], f1.cout, 1, net->wh + f1.w_off, f1.fan_in, 1, batch, f1.fan_in, f1.cout);
    d.outf = net->tmp;
    d.ofm = f1.fan_in;
    d.ofn = 1;
    gemm(net, s, d);
    const long long n = static_cast<long long>(batch) * f1.fan_in;
    hipLaunchKernelGGL(relu_mask_kernel, dim3(blocks_for(n)), dim3(256), 0, s, net->tmp, x5, net->dz[0], n);
  }
  // convolutions, last to first; dz[cur] holds the gradient of layer l's output
  int cur = 0;
  for (int l = kConv - 1; l >= 0; --l) {
    const Shape& sh = net->shapes[l];
    const int M = batch * pixels(sh), N = sh.cout, K = sh.fan_in;
    Gemm g = make_gemm(net->dz[cur], 1, N, net->col[l], K, 1, N, K, M);
    g.outf = net->grad + sh.w_off;
    g.ofm = K;
    g.ofn = 1;
    gemm(net, s, g);
    colsum(net, s, net->dz[cur], M, N, net->grad + sh.b_off, sums);
    if (l == 0) break;
    Gemm d = make_gemm(net->dz[cur], N, 1, net->wh + sh.w_off, K, 1, M, K, N);
    d.outf = net->tmp;
    d.ofm = K;
    d.ofn = 1;
    gemm(net, s, d);
    const long long total = static_cast<long long>(batch) * sh.hin * sh.win * sh.cin;
    hipLaunchKernelGGL(col2im_kernel, dim3(std::min(blocks_for(total / 4), 8192)), dim3(256), 0, s, net->tmp,
                       net->act[l], net->dz[1 - cur], batch, sh.hin, sh.win, sh.cin, sh.hout, sh.wout);
    KF_HIP(hipGetLastError());
    cur = 1 - cur;
  }
  colsum_end(s, sums);
}

void check_batch(const kf_posenet* net, int batch) {
  if (batch < 1 || batch > net->cfg.batch_capacity) {
    fail(KF_ERR_INVALID_ARGUMENT, "posenet: batch must be in [1, batch_capacity]");
  }
}

void prepare_pairs(kf_posenet* net, hipStream_t s, const uint16_t* pairs, int batch) {
  const long long hw = static_cast<long long>(kInH) * kInW;
  hipLaunchKernelGGL(input_kernel, dim3(blocks_for(hw), batch), dim3(256), 0, s, pairs, pairs + hw, 2 * hw, batch,
                     1.0F / net->cfg.depth_scale, net->act[0]);
  KF_HIP(hipGetLastError());
}

template <typename F>
kf_status net_guard(kf_posenet* net, F&& body) {
  try {
    body();
    return KF_OK;
  } catch (const kf::Failure& f) {
    if (net != nullptr) net->error = f.message;
    return f.status;
  } catch (const std::exception& e) {
    if (net != nullptr) net->error = e.what();
    return KF_ERR_DEVICE;
  }
}

// Seeded He-uniform initialisation (SplitMix64), biases zero, the output
// layer scaled by 0.1.
void init_weights(const std::vector<Shape>& shapes, uint64_t seed, std::vector<float>& w) {
  uint64_t state = seed * 0x9E3779B97F4A7C15ULL + 0x2545F4914F6CDD1DULL;
  auto next = [&]() {
    uint64_t z = (state += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    z ^= z >> 31;
    return static_cast<double>(z >> 11) * (1.0 / 9007199254740992.0);
  };
  for (size_t l = 0; l < shapes.size(); ++l) {
    const Shape& sh = shapes[l];
    const double bound = std::sqrt(6.0 / sh.fan_in) * (l + 1 == shapes.size() ? 0.1 : 1.0);
    for (size_t i = 0; i < static_cast<size_t>(sh.cout) * sh.fan_in; ++i) {
      w[sh.w_off + i] = static_cast<float>((2.0 * next() - 1.0) * bound);
    }
    for (int i = 0; i < sh.cout; ++i) w[sh.b_off + i] = 0.0F;
  }
}

// Inference forward pass for `batch` depth pairs (pair b: previous at
// prev + b * stride, current at cur + b * stride, 160 x 120 u16 each) ->
// twist[batch][6] (omega rad, t m).  Eight launches: the convolutions read
// their input as an implicit im2col matrix (the first one straight from the
// depth pairs) and the last layer writes the scaled twist.
void infer(kf_posenet* net, hipStream_t s, const uint16_t* prev, const uint16_t* cur, long long stride, int batch,
           float* twist) {
  for (int l = 0; l < kConv; ++l) {
    const Shape& sh = net->shapes[l];
    const int M = batch * pixels(sh), K = sh.fan_in;
    Gemm g = make_gemm(nullptr, 0, 0, net->wh + sh.w_off, 1, K, M, sh.cout, K);
    g.conv = ConvView{net->act[l],   l == 0 ? prev : nullptr, l == 0 ? cur : nullptr, stride,
                      1.0F / net->cfg.depth_scale, sh.hin, sh.win, sh.cin, sh.hout, sh.wout};
    g.bias = net->w + sh.b_off;
    g.relu = 1;
    g.outh = net->act[l + 1];
    g.ohm = sh.cout;
    g.ohn = 1;
    gemm(net, s, g);
  }
  const Shape& f1 = net->shapes[kConv];
  Gemm g1 = make_gemm(net->act[kConv], f1.fan_in, 1, net->wh + f1.w_off, 1, f1.fan_in, batch, f1.cout, f1.fan_in);
  g1.bias = net->w + f1.b_off;
  g1.relu = 1;
  g1.outh = net->act[kConv + 1];
  g1.ohm = f1.cout;
  g1.ohn = 1;
  gemm(net, s, g1);
  const Shape& f2 = net->shapes[kConv + 1];
  Gemm g2 = make_gemm(net->act[kConv + 1], f2.fan_in, 1, net->wh + f2.w_off, 1, f2.fan_in, batch, f2.cout,
                      f2.fan_in);
  g2.bias = net->w + f2.b_off;
  g2.outf = twist;
  g2.ofm = kOut;
  g2.ofn = 1;
  g2.scale_out = 1;
  gemm(net, s, g2);
}

}  // namespace

namespace kf {

// The pose proposal on the pipeline's stream for one pair.
void posenet_propose(kf_posenet* net, hipStream_t s, const uint16_t* prev, const uint16_t* cur, float* twist) {
  infer(net, s, prev, cur, 0LL, 1, twist);
}

bool posenet_input_matches(int width, int height) { return width == kInW && height == kInH; }

void posenet_prepare_attach(kf_posenet* net, float depth_scale) {
  if (net->cfg.depth_scale != depth_scale)
    fail(KF_ERR_INVALID_ARGUMENT, "kf_attach_posenet: the network's depth scale differs from the context's");
  KF_HIP(hipStreamSynchronize(net->stream));
}

}  // namespace kf

extern "C" {

void kf_posenet_config_defaults(kf_posenet_config* cfg) {
  if (cfg == nullptr) return;
  std::memset(cfg, 0, sizeof(*cfg));
  cfg->batch_capacity = 64;
  cfg->seed = 0;
  cfg->learning_rate = 1.0e-3F;
  cfg->beta1 = 0.9F;
  cfg->beta2 = 0.999F;
  cfg->epsilon = 1.0e-8F;
  cfg->depth_scale = 1000.0F;
}

int64_t kf_posenet_parameter_count(void) {
  size_t total = 0;
  network_shapes(&total);
  return static_cast<int64_t>(total);
}

kf_status kf_posenet_create(const kf_posenet_config* cfg, kf_posenet** out) {
  if (cfg == nullptr || out == nullptr) return KF_ERR_INVALID_ARGUMENT;
  *out = nullptr;
  auto* net = new kf_posenet();
  const kf_status st = net_guard(net, [&] {
    if (cfg->batch_capacity < 1 || cfg->batch_capacity > 4096) fail(KF_ERR_INVALID_ARGUMENT, "batch_capacity");
    if (!(cfg->depth_scale > 0.0F)) fail(KF_ERR_INVALID_ARGUMENT, "depth_scale must be > 0");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1) fail(KF_ERR_UNSUPPORTED, "no HIP device");
    net->cfg = *cfg;
    net->shapes = network_shapes(&net->n_params);
    KF_HIP(hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking));
    const size_t P = net->n_params;
    net->w = nalloc<float>(P);
    net->grad = nalloc<float>(P);
    net->m = nalloc<float>(P);
    net->v = nalloc<float>(P);
    net->wh = nalloc<uint16_t>(P);
    const int B = cfg->batch_capacity;
    size_t max_tmp = 0, max_dz = 0;
    net->act[0] = nalloc<uint16_t>(static_cast<size_t>(B) * kInH * kInW * 2);
    for (int l = 0; l < kLayers - 1; ++l) {
      const Shape& sh = net->shapes[l];
      const size_t M = static_cast<size_t>(B) * pixels(sh);
      net->act[l + 1] = nalloc<uint16_t>(M * sh.cout);
      if (l < kConv) net->col[l] = nalloc<uint16_t>(M * sh.fan_in);
      max_tmp = std::max(max_tmp, M * sh.fan_in);  // dcol / dx of any layer
      max_dz = std::max(max_dz, M * sh.cout);
    }
    max_dz = std::max(max_dz, static_cast<size_t>(B) * kOut);
    net->out = nalloc<float>(static_cast<size_t>(B) * kOut);
    net->tmp = nalloc<float>(max_tmp);
    net->dz[0] = nalloc<uint16_t>(max_dz);
    net->dz[1] = nalloc<uint16_t>(max_dz);
    net->partial_floats = static_cast<size_t>(8) << 20;
    net->partial = nalloc<float>(net->partial_floats);
    size_t chunk_floats = 0;  // of every layer's bias sum (a dense layer's shape has one pixel)
    for (const Shape& sh : net->shapes)
      chunk_floats += static_cast<size_t>(col_chunks(static_cast<long long>(B) * pixels(sh))) * sh.cout;
    net->colpart = nalloc<float>(chunk_floats);
    net->loss = nalloc<float>(1);
    KF_HIP(hipHostMalloc(reinterpret_cast<void**>(&net->loss_host), sizeof(float), hipHostMallocDefault));
    std::vector<float> w(P);
    init_weights(net->shapes, cfg->seed, w);
    KF_HIP(hipMemcpyAsync(net->w, w.data(), P * sizeof(float), hipMemcpyHostToDevice, net->stream));
    KF_HIP(hipMemsetAsync(net->m, 0, P * sizeof(float), net->stream));
    KF_HIP(hipMemsetAsync(net->v, 0, P * sizeof(float), net->stream));
    KF_HIP(hipMemsetAsync(net->grad, 0, P * sizeof(float), net->stream));
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(P)), dim3(256), 0, net->stream, net->w, net->wh,
                       static_cast<long long>(P));
    KF_HIP(hipGetLastError());
    KF_HIP(hipStreamSynchronize(net->stream));
  });
  if (st != KF_OK) {
    kf_posenet_destroy(net);
    return st;
  }
  *out = net;
  return KF_OK;
}

void kf_posenet_destroy(kf_posenet* net) {
  if (net == nullptr) return;
  if (net->stream != nullptr) (void)hipStreamSynchronize(net->stream);
  for (void* p : {static_cast<void*>(net->w), static_cast<void*>(net->grad), static_cast<void*>(net->m),
                  static_cast<void*>(net->v), static_cast<void*>(net->wh), static_cast<void*>(net->out),
                  static_cast<void*>(net->tmp), static_cast<void*>(net->dz[0]), static_cast<void*>(net->dz[1]),
                  static_cast<void*>(net->partial), static_cast<void*>(net->colpart),
                  static_cast<void*>(net->loss)}) {
    if (p != nullptr) (void)hipFree(p);
  }
  for (auto* p : net->act)
    if (p != nullptr) (void)hipFree(p);
  for (auto* p : net->col)
    if (p != nullptr) (void)hipFree(p);
  if (net->loss_host != nullptr) (void)hipHostFree(net->loss_host);
  if (net->stream != nullptr) (void)hipStreamDestroy(net->stream);
  delete net;
}

const char* kf_posenet_last_error(const kf_posenet* net) {
  return net == nullptr ? "null posenet" : net->error.c_str();
}

kf_status kf_posenet_get_parameters(kf_posenet* net, float* params) {
  return net_guard(net, [&] {
    if (net == nullptr || params == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null argument");
    const kf::HostStage::Piece out{params, net->w, net->n_params * sizeof(float)};
    KF_HIP(net->stage.copy(&out, 1, net->stream));
  });
}

kf_status kf_posenet_set_parameters(kf_posenet* net, const float* params) {
  return net_guard(net, [&] {
    if (net == nullptr || params == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null argument");
    KF_HIP(hipMemcpyAsync(net->w, params, net->n_params * sizeof(float), hipMemcpyHostToDevice, net->stream));
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(net->n_params)), dim3(256), 0, net->stream, net->w, net->wh,
                       static_cast<long long>(net->n_params));
    KF_HIP(hipGetLastError());
    KF_HIP(hipMemsetAsync(net->m, 0, net->n_params * sizeof(float), net->stream));
    KF_HIP(hipMemsetAsync(net->v, 0, net->n_params * sizeof(float), net->stream));
    net->step = 0;
    KF_HIP(hipStreamSynchronize(net->stream));
  });
}

kf_status kf_posenet_forward(kf_posenet* net, const uint16_t* pairs, int32_t batch, float* twists) {
  return net_guard(net, [&] {
    if (net == nullptr || pairs == nullptr || twists == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null argument");
    check_batch(net, batch);
    const long long hw = static_cast<long long>(kInH) * kInW;
    infer(net, net->stream, pairs, pairs + hw, 2 * hw, batch, twists);
    KF_HIP(hipGetLastError());
    KF_HIP(hipStreamSynchronize(net->stream));
  });
}

kf_status kf_posenet_gradients(kf_posenet* net, const uint16_t* pairs, const float* targets, int32_t batch,
                               float* loss, float* grads) {
  return net_guard(net, [&] {
    if (net == nullptr || pairs == nullptr || targets == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null argument");
    check_batch(net, batch);
    prepare_pairs(net, net->stream, pairs, batch);
    forward(net, net->stream, batch);
    backward(net, net->stream, targets, batch);
    KF_HIP(hipMemcpyAsync(net->loss_host, net->loss, sizeof(float), hipMemcpyDeviceToHost, net->stream));
    const kf::HostStage::Piece out{grads, net->grad, net->n_params * sizeof(float)};
    KF_HIP(net->stage.copy(&out, 1, net->stream));
    if (loss != nullptr) *loss = *net->loss_host;
  });
}

kf_status kf_posenet_train_step(kf_posenet* net, const uint16_t* pairs, const float* targets, int32_t batch,
                                float* loss) {
  return net_guard(net, [&] {
    if (net == nullptr || pairs == nullptr || targets == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null argument");
    check_batch(net, batch);
    prepare_pairs(net, net->stream, pairs, batch);
    forward(net, net->stream, batch);
    backward(net, net->stream, targets, batch);
    net->step += 1;
    const double t = static_cast<double>(net->step);
    const float c1 = static_cast<float>(1.0 / (1.0 - std::pow(static_cast<double>(net->cfg.beta1), t)));
    const float c2 = static_cast<float>(1.0 / (1.0 - std::pow(static_cast<double>(net->cfg.beta2), t)));
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(net->n_params)), dim3(256), 0, net->stream, net->w, net->grad,
                       net->m, net->v, net->wh, static_cast<long long>(net->n_params), net->cfg.learning_rate,
                       net->cfg.beta1, net->cfg.beta2, net->cfg.epsilon, c1, c2);
    KF_HIP(hipGetLastError());
    if (loss != nullptr) {
      KF_HIP(hipMemcpyAsync(net->loss_host, net->loss, sizeof(float), hipMemcpyDeviceToHost, net->stream));
      KF_HIP(hipStreamSynchronize(net->stream));
      *loss = *net->loss_host;
    }
  });
}

kf_status kf_posenet_set_learning_rate(kf_posenet* net, float learning_rate) {
  return net_guard(net, [&] {
    if (net == nullptr || !(learning_rate > 0.0F)) fail(KF_ERR_INVALID_ARGUMENT, "learning rate must be > 0");
    net->cfg.learning_rate = learning_rate;
  });
}

kf_status kf_posenet_synchronize(kf_posenet* net) {
  return net_guard(net, [&] {
    if (net == nullptr) fail(KF_ERR_INVALID_ARGUMENT, "null posenet");
    KF_HIP(hipStreamSynchronize(net->stream));
  });
}

}  // extern "C"
