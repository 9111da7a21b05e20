// Marching cubes on the device with the reference's exact output order
// (MarchingCubes::extract + MeshBuilder, src/kinectfusion/marching_cubes.cpp:
// 315-507; the reference runs it on the host only).
//
// The reference walks cells x-fastest (a sparse volume: its allocated blocks
// in key order, each block's cells x-fastest), emits each case's triangles as
// (e0, e2, e1) and numbers a welded vertex the first time its edge is met.
// The first cell to meet an edge is the lowest-ranked *active* cell sharing
// it (a crossed edge is used by every valid cell around it).  Few cells are
// active (0.2 % of a 512^3 room), so the passes over the volume work on bits
// and everything after them on the list of active cells:
//   1. voxel bits  -- two bits per voxel, usable (observed, finite, at least
//                     min_weight) and usable with tsdf < 0, by wave ballots:
//                     the only pass that reads the volume, one streaming read;
//   2. active      -- one bit per cell, 64 cells at a time: the eight corners
//                     are eight shifted words;
//   3. list        -- the active cells in traversal order, and for every word
//                     of cells the list position of its first active cell
//                     (a cell's position is that plus a bit count);
//   4. info        -- per active cell: cube index and the edges it owns (those
//                     for which it is the lowest-ranked active cell);
//   5. offsets     -- prefix sums: first triangle and first vertex of each
//                     active cell, and the edge of every vertex;
//   6. triangles   -- one thread per active cell, foreign vertices numbered by
//                     the owner's offset plus their rank in its emit order (a
//                     bit count over its owned edges);
//   7. vertices    -- one thread per vertex: position, central-difference
//                     normal, trilinear colour;
//   8. fill        -- vertices without a gradient normal get the normalised
//                     sum of their triangles' face normals, summed in triangle
//                     order (MeshBuilder::fill_missing_normals).
// Triangle order, vertex numbering, positions, normals and colours are
// identical to the CPU mesher's.
//
// Walking all cells with a thread each instead (one byte and two offsets per
// cell, a wave waiting for its one active cell's serial vertex work) took
// 4.6 ms of kernel time for a 512^3 bf16 room with colour and 31 ms for a
// 2048^3 hashed hall of 44 k blocks; the passes above take 0.28 ms and
// 0.34 ms.  The first pass is bound by the volume read (0.15 ms of the dense
// mesh, 3.6 TB/s), the others by latency.
#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "kf_sampler.hpp"

namespace kf {
namespace {

#include "mc_cases.inc"

// corner offsets (marching_cubes.cpp:315-324) and edges {near, far, axis}
// (:330-348)
constexpr int kCorner[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0},
                               {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};
constexpr int kEdge[12][3] = {{0, 1, 0}, {1, 2, 1}, {3, 2, 0}, {0, 3, 1}, {4, 5, 0}, {5, 6, 1},
                              {7, 6, 0}, {4, 7, 1}, {0, 4, 2}, {1, 5, 2}, {2, 6, 2}, {3, 7, 2}};

// Neighbour offsets (dx, dy, dz) in {-1, 0, 1}^3 are numbered
// (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1); 13 is the cell itself.
constexpr int kSelf = 13;
constexpr int offset_index(int dx, int dy, int dz) { return (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1); }

struct CaseTables {
  uint8_t ntri[256];
  uint16_t used[256];         // edges the cube crosses
  uint8_t emit[256][16];      // edges in emit order: entries (0, 2, 1) of each table triangle
  uint16_t before[256][12];   // edges whose first appearance in emit order precedes this edge's
};

constexpr CaseTables make_tables() {
  CaseTables t{};
  for (int k = 0; k < 256; ++k) {
    int n = 0;
    while (kTriCases[k][n] != '\0') ++n;
    t.ntri[k] = static_cast<uint8_t>(n / 3);
    uint16_t seen = 0;
    for (int i = 0; i < n; ++i) {
      const int s = i % 3;
      const char c = kTriCases[k][i - s + (s == 0 ? 0 : (s == 1 ? 2 : 1))];
      const int e = c <= '9' ? c - '0' : c - 'a' + 10;
      t.emit[k][i] = static_cast<uint8_t>(e);
      if (((seen >> e) & 1) == 0) {
        t.before[k][e] = seen;
        seen = static_cast<uint16_t>(seen | (1 << e));
      }
    }
    t.used[k] = seen;
  }
  return t;
}
__constant__ constexpr CaseTables c_tab = make_tables();

// The three other cells around each edge of a cell, as neighbour offsets, and
// the edge's number in each of them.
struct Around {
  int cell[12][3];
  int edge[12][3];
};
constexpr Around make_around() {
  Around a{};
  for (int e = 0; e < 12; ++e) {
    const int ox = kCorner[kEdge[e][0]][0], oy = kCorner[kEdge[e][0]][1], oz = kCorner[kEdge[e][0]][2];
    const int axis = kEdge[e][2];
    int n = 0;
    for (int k = 0; k < 2; ++k)
      for (int j = 0; j < 2; ++j) {
        // the edge's voxel is the near corner; a sharing cell sits 0 or 1
        // below it on each of the two other axes
        const int dx = axis == 0 ? 0 : ox - j;
        const int dy = axis == 0 ? oy - j : (axis == 1 ? 0 : oy - k);
        const int dz = axis == 2 ? 0 : oz - k;
        if (dx == 0 && dy == 0 && dz == 0) continue;
        a.cell[e][n] = offset_index(dx, dy, dz);
        for (int f = 0; f < 12; ++f)
          if (kEdge[f][2] == axis && kCorner[kEdge[f][0]][0] == ox - dx && kCorner[kEdge[f][0]][1] == oy - dy &&
              kCorner[kEdge[f][0]][2] == oz - dz)
            a.edge[e][n] = f;
        ++n;
      }
  }
  return a;
}
constexpr Around kAround = make_around();
// Neighbours that share an edge with the cell (all but the eight corners).
constexpr bool shares_edge(int d) {
  const int x = d % 3, y = (d / 3) % 3, z = d / 9;
  return d != kSelf && (x == 1 || y == 1 || z == 1);
}

using Word = unsigned long long;

// A cell: its word of 64 cells, its bit there, its voxel coordinates and (block
// layout) its block's position in key order.
struct Cell {
  uint32_t word;
  int bit;
  int x, y, z;
  int block;
};

// Layouts: how voxels and cells (a cell is named by its lowest corner) map to
// words of 64 bits, in traversal order.
//
// Dense: each row of voxels (fixed y, z) takes whole words.
struct DenseLayout {
  int nx, ny, nz;
  int wpr;  // words per row
  uint32_t nwords;
  __device__ inline Cell cell(uint32_t word, int bit) const {
    const uint32_t row = word / static_cast<uint32_t>(wpr);
    Cell c;
    c.word = word;
    c.bit = bit;
    c.x = static_cast<int>(word - row * wpr) * 64 + bit;
    c.z = static_cast<int>(row / static_cast<uint32_t>(ny));
    c.y = static_cast<int>(row - static_cast<uint32_t>(c.z) * ny);
    c.block = 0;
    return c;
  }
  // word and bit of voxel / cell (x, y, z); false outside the volume
  __device__ inline bool locate(int x, int y, int z, uint32_t& word, int& bit) const {
    if (x < 0 || y < 0 || z < 0 || x >= nx || y >= ny || z >= nz) return false;
    word = (static_cast<uint32_t>(z) * ny + y) * wpr + (x >> 6);
    bit = x & 63;
    return true;
  }
  __device__ inline bool at(const Cell& c, int dx, int dy, int dz, uint32_t& word, int& bit) const {
    return locate(c.x + dx, c.y + dy, c.z + dz, word, bit);
  }
  // position of a neighbour in traversal order, relative to the others'
  __device__ inline int order(const Cell&, int dx, int dy, int dz) const { return offset_index(dx, dy, dz); }
  // active cells of a word
  __device__ inline Word active(const Word* __restrict__ usable, const Word* __restrict__ inside, uint32_t w) const {
    const uint32_t row = w / static_cast<uint32_t>(wpr);
    const int z = static_cast<int>(row / static_cast<uint32_t>(ny)), y = static_cast<int>(row - static_cast<uint32_t>(z) * ny);
    if (y + 1 >= ny || z + 1 >= nz) return 0;
    const bool next = static_cast<int>(w - row * wpr) + 1 < wpr;
    const uint32_t rows[4] = {w, w + wpr, w + static_cast<uint32_t>(ny) * wpr, w + static_cast<uint32_t>(ny + 1) * wpr};
    Word v = ~0ULL, any = 0, all = ~0ULL;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Word u0 = usable[rows[i]], n0 = inside[rows[i]];
      const Word u1 = next ? usable[rows[i] + 1] : 0, n1 = next ? inside[rows[i] + 1] : 0;
      const Word us = (u0 >> 1) | (u1 << 63), ns = (n0 >> 1) | (n1 << 63);
      v &= u0 & us;
      any |= n0 | ns;
      all &= n0 & ns;
    }
    return v & any & ~all;
  }
};

// Sparse: the allocated blocks in key order, eight words per block (one per
// z-slice, bit y * 8 + x).  nbr: per block the positions of its 27 neighbours
// in that order (-1: not allocated).
struct BlockLayout {
  uint32_t nwords;
  const uint32_t* __restrict__ keys;
  const int* __restrict__ nbr;
  int bx, by, bz;  // blocks per axis
  const uint32_t* __restrict__ occ;   // one bit per block of the grid: allocated
  const uint32_t* __restrict__ rank;  // allocated blocks before each 32-bit word of occ
  __device__ inline int position(int x, int y, int z) const {
    if (x < 0 || y < 0 || z < 0 || x >= bx || y >= by || z >= bz) return -1;
    const uint32_t key = (static_cast<uint32_t>(z) * by + y) * bx + x;
    const uint32_t w = occ[key >> 5], b = key & 31U;
    return ((w >> b) & 1U) != 0U ? static_cast<int>(rank[key >> 5] + __popc(w & ((1U << b) - 1U))) : -1;
  }
  __device__ inline Cell cell(uint32_t word, int bit) const {
    Cell c;
    c.word = word;
    c.bit = bit;
    c.block = static_cast<int>(word >> 3);
    const uint32_t key = keys[c.block];
    const uint32_t row = key / static_cast<uint32_t>(bx);
    c.x = static_cast<int>(key - row * bx) * 8 + (bit & 7);
    c.y = static_cast<int>(row % static_cast<uint32_t>(by)) * 8 + (bit >> 3);
    c.z = static_cast<int>(row / static_cast<uint32_t>(by)) * 8 + static_cast<int>(word & 7U);
    return c;
  }
  __device__ inline bool locate(int x, int y, int z, uint32_t& word, int& bit) const {
    if (x < 0 || y < 0 || z < 0) return false;
    const int p = position(x >> 3, y >> 3, z >> 3);
    if (p < 0) return false;
    word = static_cast<uint32_t>(p) * 8U + (z & 7);
    bit = (y & 7) * 8 + (x & 7);
    return true;
  }
  __device__ inline bool at(const Cell& c, int dx, int dy, int dz, uint32_t& word, int& bit) const {
    const int lx = (c.x & 7) + dx, ly = (c.y & 7) + dy, lz = (c.z & 7) + dz;
    const int ox = lx >> 3, oy = ly >> 3, oz = lz >> 3;
    int p = c.block;
    if ((ox | oy | oz) != 0) p = nbr[static_cast<size_t>(p) * 27 + offset_index(ox, oy, oz)];
    if (p < 0) return false;
    word = static_cast<uint32_t>(p) * 8U + (lz & 7);
    bit = (ly & 7) * 8 + (lx & 7);
    return true;
  }
  __device__ inline int order(const Cell& c, int dx, int dy, int dz) const {
    const int ox = ((c.x & 7) + dx) >> 3, oy = ((c.y & 7) + dy) >> 3, oz = ((c.z & 7) + dz) >> 3;
    return offset_index(ox, oy, oz) * 27 + offset_index(dx, dy, dz);
  }
  __device__ inline Word active(const Word* __restrict__ usable, const Word* __restrict__ inside, uint32_t w) const {
    const uint32_t b = w >> 3;
    const int lz = static_cast<int>(w & 7U);
    const int* __restrict__ nb = nbr + static_cast<size_t>(b) * 27;
    constexpr Word kCol0 = 0x0101010101010101ULL, kCols = 0x7F7F7F7F7F7F7F7FULL;
    Word v = ~0ULL, any = 0, all = ~0ULL;
#pragma unroll
    for (int dz = 0; dz < 2; ++dz) {
      const int oz = (lz + dz) >> 3;
      const uint32_t sl = static_cast<uint32_t>((lz + dz) & 7);
      const int q00 = oz != 0 ? nb[offset_index(0, 0, 1)] : static_cast<int>(b);
      const int q10 = nb[offset_index(1, 0, oz)], q01 = nb[offset_index(0, 1, oz)], q11 = nb[offset_index(1, 1, oz)];
      const Word* maps[2] = {usable, inside};
      Word sum[2], prod[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        auto slice = [&](int q) { return q >= 0 ? maps[m][static_cast<uint32_t>(q) * 8U + sl] : 0ULL; };
        const Word s = slice(q00), sx = slice(q10), sy = slice(q01), sxy = slice(q11);
        const Word t = (s >> 8) | (sy << 56), tx = (sx >> 8) | (sxy << 56);  // one voxel along y
        const Word s1 = ((s >> 1) & kCols) | ((sx & kCol0) << 7), t1 = ((t >> 1) & kCols) | ((tx & kCol0) << 7);
        sum[m] = s | s1 | t | t1;
        prod[m] = s & s1 & t & t1;
      }
      v &= prod[0];
      any |= sum[1];
      all &= prod[1];
    }
    return v & any & ~all;
  }
};

// ---- 1. voxel bits -----------------------------------------------------------
// The usable and inside words of eight groups of 64 voxels held by a wave, one
// voxel per lane and group; lane j keeps group j's words.
template <int Kind>
__device__ inline void pack_words(const typename VoxelIO<Kind>::Raw (&r)[8], float min_weight, int lane, Word& usable,
                                  Word& inside) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float t, w;
    bool obs, fin;
    VoxelIO<Kind>::unpack(r[j], t, w, obs, fin);
    const bool ok = obs && fin && !(w < min_weight);
    const Word mu = __ballot(ok), mi = __ballot(ok && t < 0.0F);
    if (lane == j) {
      usable = mu;
      inside = mi;
    }
  }
}

// A wave takes eight consecutive words, its reads (256 or 512 contiguous bytes
// each) all in flight.
template <int Kind>
__global__ void __launch_bounds__(256) dense_bits_kernel(const typename VoxelIO<Kind>::Raw* __restrict__ vox,
                                                          DenseLayout o, float min_weight, Word* __restrict__ usable,
                                                          Word* __restrict__ inside) {
  const int lane = threadIdx.x & 63;
  const uint32_t w0 = (blockIdx.x * 4U + (threadIdx.x >> 6)) * 8U;
  typename VoxelIO<Kind>::Raw r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t w = w0 + j, row = w / static_cast<uint32_t>(o.wpr);
    const int x = static_cast<int>(w - row * o.wpr) * 64 + lane;
    r[j] = (w < o.nwords && x < o.nx) ? vox[static_cast<size_t>(row) * o.nx + x] : VoxelIO<Kind>::fresh();
  }
  Word u = 0, n = 0;
  pack_words<Kind>(r, min_weight, lane, u, n);
  if (lane < 8 && w0 + lane < o.nwords) {
    usable[w0 + lane] = u;
    inside[w0 + lane] = n;
  }
}

// A wave takes one block.  A voxel beyond the grid is never observed.
template <int Kind>
__global__ void __launch_bounds__(256) block_bits_kernel(const typename VoxelIO<Kind>::Raw* __restrict__ pool,
                                                          const uint32_t* __restrict__ slots, uint32_t nblocks,
                                                          float min_weight, Word* __restrict__ usable,
                                                          Word* __restrict__ inside) {
  const int lane = threadIdx.x & 63;
  const uint32_t b = blockIdx.x * 4U + (threadIdx.x >> 6);
  if (b >= nblocks) return;
  const typename VoxelIO<Kind>::Raw* v = pool + static_cast<size_t>(slots[b]) * kBlockVoxels + lane;
  typename VoxelIO<Kind>::Raw r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = v[j * 64];
  Word u = 0, n = 0;
  pack_words<Kind>(r, min_weight, lane, u, n);
  if (lane < 8) {
    usable[b * 8U + lane] = u;
    inside[b * 8U + lane] = n;
  }
}

// ---- prefix sums -------------------------------------------------------------
// Exclusive scan of two counters across the 256 threads of a workgroup.
__device__ inline void block_scan2(unsigned a, unsigned b, unsigned& ea, unsigned& eb, unsigned& ta, unsigned& tb) {
  __shared__ unsigned sa[4], sb[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned ia = a, ib = b;
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned va = __shfl_up(ia, off), vb = __shfl_up(ib, off);
    if (lane >= off) {
      ia += va;
      ib += vb;
    }
  }
  if (lane == 63) {
    sa[wave] = ia;
    sb[wave] = ib;
  }
  __syncthreads();
  unsigned pa = 0, pb = 0;
  for (int w = 0; w < wave; ++w) {
    pa += sa[w];
    pb += sb[w];
  }
  ea = pa + ia - a;
  eb = pb + ib - b;
  ta = sa[0] + sa[1] + sa[2] + sa[3];
  tb = sb[0] + sb[1] + sb[2] + sb[3];
  __syncthreads();
}

// Single workgroup: exclusive scan in place of n pairs of chunk counts; the
// totals in 64 bits.  Eight counts per thread and pass, coalesced through the
// thread's consecutive reads, so the pass count, not a serial walk, sets it.
__global__ void __launch_bounds__(256) chunk_scan_kernel(uint2* __restrict__ chunks, uint32_t n,
                                                          unsigned long long* __restrict__ totals) {
  constexpr int kRun = 8;
  __shared__ unsigned long long carry[2];
  if (threadIdx.x < 2) carry[threadIdx.x] = 0ULL;
  __syncthreads();
  for (uint32_t base = 0; base < n; base += 256U * kRun) {
    const uint32_t i0 = base + threadIdx.x * kRun;
    uint2 v[kRun];
    unsigned sa = 0, sb = 0;
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
      v[j] = i0 + j < n ? chunks[i0 + j] : make_uint2(0U, 0U);
      sa += v[j].x;
      sb += v[j].y;
    }
    unsigned ea, eb, ta, tb;
    block_scan2(sa, sb, ea, eb, ta, tb);
    const unsigned long long ca = carry[0], cb = carry[1];
    ea += static_cast<unsigned>(ca);
    eb += static_cast<unsigned>(cb);
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
      if (i0 + j < n) chunks[i0 + j] = make_uint2(ea, eb);
      ea += v[j].x;
      eb += v[j].y;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      carry[0] = ca + ta;
      carry[1] = cb + tb;
    }
    __syncthreads();
  }
  if (threadIdx.x < 2) totals[threadIdx.x] = carry[threadIdx.x];
}

// ---- block order of a hashed volume -------------------------------------------
// Allocated blocks sorted by key without a sort: keys are unique, so a bitmap
// of them with word-prefix counts gives every block its position.
__global__ void __launch_bounds__(256) occ_mark_kernel(const uint32_t* __restrict__ block_of_slot, uint32_t n,
                                                        uint32_t* __restrict__ occ) {
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  if (i < n) atomicOr(&occ[block_of_slot[i] >> 5], 1U << (block_of_slot[i] & 31U));
}
constexpr uint32_t kOccRun = 8;  // words per thread, consecutive
__global__ void __launch_bounds__(256) occ_count_kernel(const uint32_t* __restrict__ occ, uint32_t words,
                                                         uint2* __restrict__ chunks) {
  const uint32_t i0 = (blockIdx.x * 256U + threadIdx.x) * kOccRun;
  unsigned s = 0;
#pragma unroll
  for (uint32_t j = 0; j < kOccRun; ++j) s += i0 + j < words ? __popc(occ[i0 + j]) : 0U;
  unsigned ea, eb, ta, tb;
  block_scan2(s, 0U, ea, eb, ta, tb);
  if (threadIdx.x == 0) chunks[blockIdx.x] = make_uint2(ta, 0U);
}
__global__ void __launch_bounds__(256) occ_rank_kernel(const uint32_t* __restrict__ occ, uint32_t words,
                                                        const uint2* __restrict__ chunks, uint32_t* __restrict__ rank) {
  const uint32_t i0 = (blockIdx.x * 256U + threadIdx.x) * kOccRun;
  unsigned c[kOccRun], s = 0;
#pragma unroll
  for (uint32_t j = 0; j < kOccRun; ++j) {
    c[j] = i0 + j < words ? __popc(occ[i0 + j]) : 0U;
    s += c[j];
  }
  unsigned ea, eb, ta, tb;
  block_scan2(s, 0U, ea, eb, ta, tb);
  ea += chunks[blockIdx.x].x;
#pragma unroll
  for (uint32_t j = 0; j < kOccRun; ++j) {
    if (i0 + j < words) rank[i0 + j] = ea;
    ea += c[j];
  }
}
// Key and pool slot of every block in key order.
__global__ void __launch_bounds__(256) block_order_kernel(const uint32_t* __restrict__ block_of_slot, uint32_t n,
                                                           BlockLayout o, uint32_t* __restrict__ keys,
                                                           uint32_t* __restrict__ slots) {
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  if (i >= n) return;
  const uint32_t key = block_of_slot[i], w = o.occ[key >> 5];
  const uint32_t p = o.rank[key >> 5] + static_cast<uint32_t>(__popc(w & ((1U << (key & 31U)) - 1U)));
  keys[p] = key;
  slots[p] = i;
}
// Positions of every block's 27 neighbours.
__global__ void __launch_bounds__(256) block_neighbours_kernel(BlockLayout o, uint32_t n, int* __restrict__ nbr) {
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  const uint32_t b = i / 27U;
  if (b >= n) return;
  const int d = static_cast<int>(i - b * 27U);
  const uint32_t key = o.keys[b], row = key / static_cast<uint32_t>(o.bx);
  nbr[i] = o.position(static_cast<int>(key - row * o.bx) + d % 3 - 1,
                      static_cast<int>(row % static_cast<uint32_t>(o.by)) + (d / 3) % 3 - 1,
                      static_cast<int>(row / static_cast<uint32_t>(o.by)) + d / 9 - 1);
}

// ---- 2., 3. active cells and their list ---------------------------------------
constexpr uint32_t kWordRun = 4;  // words per thread (strided by 256: coalesced)

template <typename Layout>
__global__ void __launch_bounds__(256) active_kernel(Layout o, const Word* __restrict__ usable,
                                                      const Word* __restrict__ inside, Word* __restrict__ active,
                                                      uint2* __restrict__ chunks) {
  const uint32_t w0 = blockIdx.x * (256U * kWordRun) + threadIdx.x;
  unsigned s = 0;
#pragma unroll
  for (uint32_t j = 0; j < kWordRun; ++j) {
    const uint32_t w = w0 + j * 256U;
    if (w >= o.nwords) continue;
    const Word a = o.active(usable, inside, w);
    active[w] = a;
    s += static_cast<unsigned>(__popcll(a));
  }
  unsigned ea, eb, ta, tb;
  block_scan2(s, 0U, ea, eb, ta, tb);
  if (threadIdx.x == 0) chunks[blockIdx.x] = make_uint2(ta, 0U);
}

// list[i] = word << 6 | bit of the i-th active cell; first[w]: list position of
// word w's first active cell (written where there is one).
__global__ void __launch_bounds__(256) list_kernel(uint32_t nwords, const Word* __restrict__ active,
                                                    const uint2* __restrict__ chunks, uint32_t* __restrict__ first,
                                                    Word* __restrict__ list) {
  const uint32_t w0 = blockIdx.x * (256U * kWordRun) + threadIdx.x;
  unsigned at = chunks[blockIdx.x].x;
  Word a[kWordRun];
#pragma unroll
  for (uint32_t j = 0; j < kWordRun; ++j) a[j] = w0 + j * 256U < nwords ? active[w0 + j * 256U] : 0ULL;
#pragma unroll
  for (uint32_t j = 0; j < kWordRun; ++j) {
    const unsigned c = static_cast<unsigned>(__popcll(a[j]));
    unsigned ea, eb, ta, tb;
    block_scan2(c, 0U, ea, eb, ta, tb);
    if (c != 0U) {
      const uint32_t w = w0 + j * 256U;
      unsigned p = at + ea;
      first[w] = p;
      for (Word m = a[j]; m != 0ULL; m &= m - 1ULL) list[p++] = (static_cast<Word>(w) << 6) | static_cast<unsigned>(__ffsll(m) - 1);
    }
    at += ta;
  }
}

// ---- 4. - 6. the active cells -------------------------------------------------
struct ActiveSet {
  const Word* __restrict__ active;
  const uint32_t* __restrict__ first;
  const Word* __restrict__ list;
  uint32_t n;
  // list position of the active cell at (word, bit)
  __device__ inline uint32_t position(uint32_t word, int bit) const {
    return first[word] + static_cast<uint32_t>(__popcll(active[word] & ((1ULL << bit) - 1ULL)));
  }
};

// Bit d: the neighbour at offset d shares an edge with the cell and is active.
template <typename Layout>
__device__ inline uint32_t active_around(const Layout& o, const Cell& c, const Word* __restrict__ active) {
  uint32_t m = 0;
#pragma unroll
  for (int d = 0; d < 27; ++d) {
    if (!shares_edge(d)) continue;
    uint32_t w;
    int b;
    if (o.at(c, d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1, w, b) && ((active[w] >> b) & 1ULL) != 0ULL) m |= 1U << d;
  }
  return m;
}

// info[i] = cube | owned edges << 8.
template <typename Layout>
__global__ void __launch_bounds__(256) info_kernel(Layout o, ActiveSet set, const Word* __restrict__ inside,
                                                    uint32_t* __restrict__ info, uint2* __restrict__ chunks) {
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  unsigned nt = 0, nv = 0;
  if (i < set.n) {
    const Word id = set.list[i];
    const Cell c = o.cell(static_cast<uint32_t>(id >> 6), static_cast<int>(id & 63ULL));
    unsigned cube = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint32_t w;
      int b;
      if (o.at(c, kCorner[k][0], kCorner[k][1], kCorner[k][2], w, b) && ((inside[w] >> b) & 1ULL) != 0ULL) cube |= 1U << k;
    }
    const uint32_t around = active_around(o, c, set.active);
    // the neighbours that come before this cell
    uint32_t earlier = 0;
    const int self = o.order(c, 0, 0, 0);
#pragma unroll
    for (int d = 0; d < 27; ++d)
      if (shares_edge(d) && o.order(c, d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1) < self) earlier |= 1U << d;
    earlier &= around;
    const uint32_t used = c_tab.used[cube];
    uint32_t owned = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e) {
      const uint32_t others = (1U << kAround.cell[e][0]) | (1U << kAround.cell[e][1]) | (1U << kAround.cell[e][2]);
      if ((earlier & others) == 0U) owned |= 1U << e;
    }
    owned &= used;
    info[i] = cube | (owned << 8);
    nt = c_tab.ntri[cube];
    nv = static_cast<unsigned>(__popc(owned));
  }
  unsigned ea, eb, ta, tb;
  block_scan2(nt, nv, ea, eb, ta, tb);
  if (threadIdx.x == 0) chunks[blockIdx.x] = make_uint2(ta, tb);
}

// off[i] = first triangle, first vertex; vkey[v]: voxel x | y << 16 | z << 32
// of vertex v's edge and its axis << 48.
template <typename Layout>
__global__ void __launch_bounds__(256) offset_kernel(Layout o, ActiveSet set, const uint32_t* __restrict__ info,
                                                      const uint2* __restrict__ chunks, uint2* __restrict__ off,
                                                      Word* __restrict__ vkey) {
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  const uint32_t inf = i < set.n ? info[i] : 0U;
  const uint32_t cube = inf & 255U, owned = inf >> 8;
  unsigned ea, eb, ta, tb;
  block_scan2(c_tab.ntri[cube], static_cast<unsigned>(__popc(owned)), ea, eb, ta, tb);
  if (i >= set.n) return;
  const uint2 base = make_uint2(chunks[blockIdx.x].x + ea, chunks[blockIdx.x].y + eb);
  off[i] = base;
  if (owned == 0U) return;
  const Word id = set.list[i];
  const Cell c = o.cell(static_cast<uint32_t>(id >> 6), static_cast<int>(id & 63ULL));
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    if (((owned >> e) & 1U) == 0U) continue;
    const uint32_t v = base.y + static_cast<uint32_t>(__popc(owned & c_tab.before[cube][e]));
    const int* k = kCorner[kEdge[e][0]];
    vkey[v] = static_cast<Word>(c.x + k[0]) | (static_cast<Word>(c.y + k[1]) << 16) |
              (static_cast<Word>(c.z + k[2]) << 32) | (static_cast<Word>(kEdge[e][2]) << 48);
  }
}

template <typename Layout>
__global__ void __launch_bounds__(256) triangle_kernel(Layout o, ActiveSet set, const uint32_t* __restrict__ info,
                                                        const uint2* __restrict__ off, uint32_t* __restrict__ tris) {
  __shared__ uint32_t ids[12][256];
  const uint32_t i = blockIdx.x * 256U + threadIdx.x;
  if (i >= set.n) return;
  const uint32_t inf = info[i], cube = inf & 255U, owned = inf >> 8, used = c_tab.used[cube];
  const uint2 base = off[i];
  const Word id = set.list[i];
  const Cell c = o.cell(static_cast<uint32_t>(id >> 6), static_cast<int>(id & 63ULL));
  const uint32_t around = active_around(o, c, set.active);
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    if (((used >> e) & 1U) == 0U) continue;
    uint32_t v;
    if (((owned >> e) & 1U) != 0U) {
      v = base.y + static_cast<uint32_t>(__popc(owned & c_tab.before[cube][e]));
    } else {
      // the first active cell around the edge
      int best = 0x7FFFFFFF, edge = 0;
      uint32_t word = 0;
      int bit = 0;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int d = kAround.cell[e][q];
        const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
        const int ord = o.order(c, dx, dy, dz);
        if (((around >> d) & 1U) != 0U && ord < best) {
          best = ord;
          edge = kAround.edge[e][q];
          o.at(c, dx, dy, dz, word, bit);
        }
      }
      const uint32_t p = set.position(word, bit), other = info[p];
      v = off[p].y + static_cast<uint32_t>(__popc((other >> 8) & c_tab.before[other & 255U][edge]));
    }
    ids[e][threadIdx.x] = v;  // read back by this thread only
  }
  const int n = 3 * c_tab.ntri[cube];
  for (int k = 0; k < n; ++k) tris[3 * static_cast<size_t>(base.x) + k] = ids[c_tab.emit[cube][k]][threadIdx.x];
}

// ---- 7. vertices ---------------------------------------------------------------
template <int Kind, typename Store>
__global__ void __launch_bounds__(256) vertex_kernel(Sampler<Kind, Store> vol, const Word* __restrict__ vkey,
                                                      float* __restrict__ pos, float* __restrict__ nrm,
                                                      float* __restrict__ col, unsigned* __restrict__ fix_list,
                                                      unsigned* __restrict__ fix_count, unsigned nvert) {
  using IO = VoxelIO<Kind>;
  const unsigned v = blockIdx.x * 256U + threadIdx.x;
  if (v >= nvert) return;
  const Word key = vkey[v];
  const int vx = static_cast<int>(key & 0xFFFFULL), vy = static_cast<int>((key >> 16) & 0xFFFFULL),
            vz = static_cast<int>((key >> 32) & 0xFFFFULL), axis = static_cast<int>(key >> 48);
  const int fx = vx + (axis == 0 ? 1 : 0), fy = vy + (axis == 1 ? 1 : 0), fz = vz + (axis == 2 ? 1 : 0);
  float nv, fv, w;
  bool obs, fin;
  SlotCache cache;
  IO::unpack(vol.s.voxel_cached(vol.g, vx, vy, vz, cache), nv, w, obs, fin);
  IO::unpack(vol.s.voxel_cached(vol.g, fx, fy, fz, cache), fv, w, obs, fin);
  const V3 np = vol.g.center(vx, vy, vz);
  const V3 fp = vol.g.center(fx, fy, fz);
  const float frac = -nv / (fv - nv);
  const V3 p = add3(np, scale3(sub3(fp, np), frac));
  V3 nn;
  if (!vol.normal(p, false, nn)) nn = mk3(0.0F, 0.0F, 0.0F);
  V3 cc;
  if (!vol.color(p, cc)) cc = mk3(255.0F, 255.0F, 255.0F);
  const size_t at = 3 * static_cast<size_t>(v);
  pos[at] = p.x;
  pos[at + 1] = p.y;
  pos[at + 2] = p.z;
  nrm[at] = nn.x;
  nrm[at + 1] = nn.y;
  nrm[at + 2] = nn.z;
  col[at] = cc.x;
  col[at + 1] = cc.y;
  col[at + 2] = cc.z;
  if (nn.x == 0.0F && nn.y == 0.0F && nn.z == 0.0F) fix_list[atomicAdd(fix_count, 1U)] = v;
}

// ---- 8. fill -------------------------------------------------------------------
template <typename Layout>
__global__ void __launch_bounds__(256) fill_normals_kernel(Layout o, ActiveSet set, const uint32_t* __restrict__ info,
                                                            const uint2* __restrict__ off,
                                                            const uint32_t* __restrict__ tris,
                                                            const float* __restrict__ pos,
                                                            const Word* __restrict__ vkey,
                                                            const unsigned* __restrict__ fix_list,
                                                            const unsigned* __restrict__ fix_count,
                                                            float* __restrict__ nrm) {
  const unsigned n = *fix_count;
  for (unsigned i = blockIdx.x * 256U + threadIdx.x; i < n; i += gridDim.x * 256U) {
    const unsigned vid = fix_list[i];
    const Word key = vkey[vid];
    const int vx = static_cast<int>(key & 0xFFFFULL), vy = static_cast<int>((key >> 16) & 0xFFFFULL),
              vz = static_cast<int>((key >> 32) & 0xFFFFULL), axis = static_cast<int>(key >> 48);
    // the active cells around the edge in traversal order, as list positions
    uint32_t r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = q & 1, k = q >> 1;
      uint32_t w = 0;
      int b = 0;
      r[q] = 0xFFFFFFFFU;
      if (o.locate(axis == 0 ? vx : vx - j, axis == 0 ? vy - j : (axis == 1 ? vy : vy - k), axis == 2 ? vz : vz - k, w, b) &&
          ((set.active[w] >> b) & 1ULL) != 0ULL)
        r[q] = set.position(w, b);
    }
    auto order2 = [](uint32_t& a, uint32_t& b) {
      const uint32_t lo = min(a, b), hi = max(a, b);
      a = lo;
      b = hi;
    };
    order2(r[0], r[1]);
    order2(r[2], r[3]);
    order2(r[0], r[2]);
    order2(r[1], r[3]);
    order2(r[1], r[2]);
    V3 sum = mk3(0.0F, 0.0F, 0.0F);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (r[q] == 0xFFFFFFFFU) continue;
      const int nt = c_tab.ntri[info[r[q]] & 255U];
      const uint32_t* tr = tris + 3 * static_cast<size_t>(off[r[q]].x);
      for (int t = 0; t < nt; ++t, tr += 3) {
        const size_t a = tr[0], b = tr[1], c = tr[2];
        if (a != vid && b != vid && c != vid) continue;
        const V3 p0 = mk3(pos[3 * a], pos[3 * a + 1], pos[3 * a + 2]);
        const V3 p1 = mk3(pos[3 * b], pos[3 * b + 1], pos[3 * b + 2]);
        const V3 p2 = mk3(pos[3 * c], pos[3 * c + 1], pos[3 * c + 2]);
        sum = add3(sum, cross3(sub3(p1, p0), sub3(p2, p0)));
      }
    }
    const V3 nn = normalize3(sum);
    nrm[3 * static_cast<size_t>(vid)] = nn.x;
    nrm[3 * static_cast<size_t>(vid) + 1] = nn.y;
    nrm[3 * static_cast<size_t>(vid) + 2] = nn.z;
  }
}

__global__ void zero_words_kernel(uint32_t* p, size_t n) {
  for (size_t i = blockIdx.x * 256ULL + threadIdx.x; i < n; i += gridDim.x * 256ULL) p[i] = 0U;
}

unsigned groups(unsigned long long n, unsigned per) { return static_cast<unsigned>((n + per - 1) / per); }

// One of the context's device scratch blocks for extraction, at least `bytes`
// long and kept for the next call; parts are handed out in turn.
class Scratch {
 public:
  Scratch(kf_context* ctx, int which, size_t bytes) : block_(ctx->mesh_scratch[which]) {
    if (block_.bytes < bytes) {
      // nothing on the stream reads the old block: extraction calls end synchronised
      if (block_.p != nullptr) (void)hipFree(block_.p);
      block_ = DeviceBlock{};
      KF_HIP(hipMalloc(&block_.p, bytes));
      block_.bytes = bytes;
    }
  }
  template <typename T>
  T* take(size_t count) {
    T* p = reinterpret_cast<T*>(static_cast<char*>(block_.p) + used_);
    used_ += padded(count * sizeof(T));
    return p;
  }
  static size_t padded(size_t bytes) { return (bytes + 255) / 256 * 256; }

 private:
  DeviceBlock& block_;
  size_t used_ = 0;
};

}  // namespace
}  // namespace kf

// A mesh on the device: positions, normals, colours (3 floats a vertex each)
// and triangles, in one block that the mesh owns.
struct kf_mesh {
  kf::DeviceBlock block;
  size_t vertices = 0, triangles = 0;
  std::shared_ptr<kf::MeshShare> share;
  hipStream_t copies = nullptr;  // the share's
  float* positions() const { return static_cast<float*>(block.p); }
  float* normals() const { return positions() + 3 * vertices; }
  float* colors() const { return normals() + 3 * vertices; }
  uint32_t* faces() const { return reinterpret_cast<uint32_t*>(colors() + 3 * vertices); }
  kf_mesh() = default;
  kf_mesh(const kf_mesh&) = delete;
  kf_mesh& operator=(const kf_mesh&) = delete;
  ~kf_mesh() {
    if (block.p != nullptr) share->give(block);
  }
};

namespace kf {

MeshShare::~MeshShare() {
  release();
  if (stream_ != nullptr) (void)hipStreamDestroy(stream_);
}

hipStream_t MeshShare::stream() {
  const std::lock_guard<std::mutex> lock(mu_);
  if (stream_ == nullptr) KF_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  return stream_;
}

DeviceBlock MeshShare::take(size_t bytes) {
  {
    const std::lock_guard<std::mutex> lock(mu_);
    for (int i = 0; i < n_; ++i)
      if (kept_[i].bytes >= bytes && kept_[i].bytes <= 2 * bytes) {
        const DeviceBlock b = kept_[i];
        kept_[i] = kept_[--n_];
        return b;
      }
  }
  release();
  DeviceBlock b{nullptr, bytes};
  KF_HIP(hipMalloc(&b.p, bytes));
  return b;
}

void MeshShare::give(DeviceBlock block) {
  {
    const std::lock_guard<std::mutex> lock(mu_);
    size_t all = block.bytes;
    for (int i = 0; i < n_; ++i) all += kept_[i].bytes;
    if (all <= kKeepBytes && n_ < kBlocks) {
      kept_[n_++] = block;
      return;
    }
  }
  (void)hipFree(block.p);
}

void MeshShare::release() {
  DeviceBlock blocks[kBlocks];
  int n = 0;
  {
    const std::lock_guard<std::mutex> lock(mu_);
    while (n_ > 0) blocks[n++] = kept_[--n_];
  }
  while (n > 0) (void)hipFree(blocks[--n].p);  // waits for the device: not with the lock held
}

namespace {

// The scratch blocks kept between calls are at most this long in all: beyond it
// the longest are returned when their call ends.
constexpr size_t kKeepBytes = size_t{256} << 20;

void read_totals(kf_context* ctx) { KF_HIP(hipStreamSynchronize(ctx->stream)); }

// Steps 2 to 8 over the voxel bits.
template <int Kind, typename Store, typename Layout>
void run_mc(kf_context* ctx, const Sampler<Kind, Store>& vol, const Layout& o, const Word* usable, const Word* inside,
            Word* active, uint32_t* first, uint2* chunks, kf_mesh* mesh) {
  hipStream_t s = ctx->stream;
  unsigned long long* totals = ctx->mesh_totals;  // pinned: the device writes them, the host reads after a wait
  const unsigned wg = groups(o.nwords, 256U * kWordRun);
  hipLaunchKernelGGL(active_kernel<Layout>, dim3(wg), dim3(256), 0, s, o, usable, inside, active, chunks);
  hipLaunchKernelGGL(chunk_scan_kernel, dim3(1), dim3(256), 0, s, chunks, wg, totals);
  KF_HIP(hipGetLastError());
  mesh->copies = mesh->share->stream();  // made, by the first extraction, while the device reads the volume
  read_totals(ctx);
  const unsigned long long n = totals[0];
  if (n >= (1ULL << 31)) fail(KF_ERR_OUT_OF_MEMORY, "mesh exceeds 2^31 elements");
  if (n == 0) return;
  const unsigned cg = groups(n, 256);
  Scratch cells(ctx, 1,
                Scratch::padded(n * sizeof(Word)) + Scratch::padded(n * 4) + Scratch::padded(n * sizeof(uint2)) +
                    Scratch::padded(cg * sizeof(uint2)));
  Word* list = cells.take<Word>(n);
  uint32_t* info = cells.take<uint32_t>(n);
  uint2* off = cells.take<uint2>(n);
  uint2* cell_chunks = cells.take<uint2>(cg);
  const ActiveSet set{active, first, list, static_cast<uint32_t>(n)};
  hipLaunchKernelGGL(list_kernel, dim3(wg), dim3(256), 0, s, o.nwords, active, chunks, first, list);
  hipLaunchKernelGGL(info_kernel<Layout>, dim3(cg), dim3(256), 0, s, o, set, inside, info, cell_chunks);
  hipLaunchKernelGGL(chunk_scan_kernel, dim3(1), dim3(256), 0, s, cell_chunks, cg, totals);
  KF_HIP(hipGetLastError());
  read_totals(ctx);
  const unsigned long long ntri = totals[0], nvert = totals[1];
  if (ntri >= (1ULL << 31) || nvert >= (1ULL << 31)) fail(KF_ERR_OUT_OF_MEMORY, "mesh exceeds 2^31 elements");
  mesh->block = mesh->share->take(36 * nvert + 12 * ntri);
  mesh->vertices = nvert;
  mesh->triangles = ntri;
  Scratch verts(ctx, 2, Scratch::padded(nvert * sizeof(Word)) + Scratch::padded(nvert * 4) + Scratch::padded(16));
  Word* vkey = verts.take<Word>(nvert);
  unsigned* fix = verts.take<unsigned>(nvert);
  unsigned* fix_count = verts.take<unsigned>(4);
  hipLaunchKernelGGL(offset_kernel<Layout>, dim3(cg), dim3(256), 0, s, o, set, info, cell_chunks, off, vkey);
  hipLaunchKernelGGL(triangle_kernel<Layout>, dim3(cg), dim3(256), 0, s, o, set, info, off, mesh->faces());
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(256), 0, s, fix_count, size_t{4});
  hipLaunchKernelGGL((vertex_kernel<Kind, Store>), dim3(groups(nvert, 256)), dim3(256), 0, s, vol, vkey,
                     mesh->positions(), mesh->normals(), mesh->colors(), fix, fix_count, static_cast<unsigned>(nvert));
  hipLaunchKernelGGL(fill_normals_kernel<Layout>, dim3(256), dim3(256), 0, s, o, set, info, off, mesh->faces(),
                     mesh->positions(), vkey, fix, fix_count, mesh->normals());
  KF_HIP(hipGetLastError());
}

template <int Kind>
void extract_dense(kf_context* ctx, float min_weight, kf_mesh* mesh) {
  using Raw = typename VoxelIO<Kind>::Raw;
  const Grid& g = ctx->grid;
  DenseLayout o{g.nx, g.ny, g.nz, (g.nx + 63) / 64, 0};
  o.nwords = static_cast<uint32_t>(o.wpr) * static_cast<uint32_t>(g.ny) * static_cast<uint32_t>(g.nz);  // <= 2^30
  const size_t w = o.nwords, wg = groups(w, 256U * kWordRun);
  Scratch bits(ctx, 0, 3 * Scratch::padded(w * sizeof(Word)) + Scratch::padded(w * 4) + Scratch::padded(wg * sizeof(uint2)));
  Word* usable = bits.take<Word>(w);
  Word* inside = bits.take<Word>(w);
  Word* active = bits.take<Word>(w);
  uint32_t* first = bits.take<uint32_t>(w);
  uint2* chunks = bits.take<uint2>(wg);
  const Raw* vox = static_cast<const Raw*>(ctx->voxels);
  hipLaunchKernelGGL(dense_bits_kernel<Kind>, dim3(groups(w, 32)), dim3(256), 0, ctx->stream, vox, o, min_weight, usable,
                     inside);
  Sampler<Kind> vol{DenseStore<Kind>{vox, ctx->colors}, g, 1.0F / g.voxel};
  run_mc(ctx, vol, o, usable, inside, active, first, chunks, mesh);
}

template <int Kind>
void extract_hashed(kf_context* ctx, float min_weight, kf_mesh* mesh) {
  using Raw = typename VoxelIO<Kind>::Raw;
  hipStream_t s = ctx->stream;
  const Grid& g = ctx->grid;
  uint32_t requested = 0;  // slots 0 .. requested - 1 (at most the capacity) hold the allocated blocks
  KF_HIP(hipMemcpyAsync(&requested, ctx->sparse, sizeof(requested), hipMemcpyDeviceToHost, s));
  KF_HIP(hipStreamSynchronize(s));
  const uint32_t n = static_cast<uint32_t>(std::min<size_t>(requested, ctx->capacity));
  if (n == 0) return;
  const BlockMap bm = block_map(g);
  const size_t occ_words = (static_cast<size_t>(bm.bx) * bm.by * bm.bz + 31) / 32, w = size_t{8} * n;
  const size_t wg = std::max<size_t>(groups(w, 256U * kWordRun), groups(occ_words, 256U * kOccRun));
  Scratch bits(ctx, 0, 3 * Scratch::padded(w * sizeof(Word)) + Scratch::padded(w * 4) + Scratch::padded(wg * sizeof(uint2)) +
                           2 * Scratch::padded(occ_words * 4) + 2 * Scratch::padded(size_t{4} * n) +
                           Scratch::padded(size_t{108} * n));
  Word* usable = bits.take<Word>(w);
  Word* inside = bits.take<Word>(w);
  Word* active = bits.take<Word>(w);
  uint32_t* first = bits.take<uint32_t>(w);
  uint2* chunks = bits.take<uint2>(wg);
  uint32_t* occ = bits.take<uint32_t>(occ_words);
  uint32_t* rank = bits.take<uint32_t>(occ_words);
  uint32_t* keys = bits.take<uint32_t>(n);
  uint32_t* slots = bits.take<uint32_t>(n);
  int* nbr = bits.take<int>(size_t{27} * n);
  const BlockLayout o{8U * n, keys, nbr, bm.bx, bm.by, bm.bz, occ, rank};
  const unsigned og = groups(occ_words, 256U * kOccRun);
  hipLaunchKernelGGL(zero_words_kernel, dim3(std::min(1024U, groups(occ_words, 256))), dim3(256), 0, s, occ, occ_words);
  hipLaunchKernelGGL(occ_mark_kernel, dim3(groups(n, 256)), dim3(256), 0, s, ctx->block_of_slot, n, occ);
  hipLaunchKernelGGL(occ_count_kernel, dim3(og), dim3(256), 0, s, occ, static_cast<uint32_t>(occ_words), chunks);
  hipLaunchKernelGGL(chunk_scan_kernel, dim3(1), dim3(256), 0, s, chunks, og, ctx->mesh_totals);
  hipLaunchKernelGGL(occ_rank_kernel, dim3(og), dim3(256), 0, s, occ, static_cast<uint32_t>(occ_words), chunks, rank);
  hipLaunchKernelGGL(block_order_kernel, dim3(groups(n, 256)), dim3(256), 0, s, ctx->block_of_slot, n, o, keys, slots);
  hipLaunchKernelGGL(block_neighbours_kernel, dim3(groups(27ULL * n, 256)), dim3(256), 0, s, o, n, nbr);
  const Raw* pool = static_cast<const Raw*>(ctx->voxels);
  hipLaunchKernelGGL(block_bits_kernel<Kind>, dim3(groups(n, 4)), dim3(256), 0, s, pool, slots, n, min_weight, usable,
                     inside);
  Sampler<Kind, HashedStore<Kind>> vol{HashedStore<Kind>{hash_view(ctx), pool, ctx->colors}, g, 1.0F / g.voxel};
  run_mc(ctx, vol, o, usable, inside, active, first, chunks, mesh);
}

template <int Kind>
void extract_t(kf_context* ctx, float min_weight, kf_mesh* mesh) {
  if (ctx->mesh_totals == nullptr)
    KF_HIP(hipHostMalloc(reinterpret_cast<void**>(&ctx->mesh_totals), 2 * sizeof(unsigned long long), hipHostMallocDefault));
  if (hashed(ctx)) extract_hashed<Kind>(ctx, min_weight, mesh);
  else extract_dense<Kind>(ctx, min_weight, mesh);
}

// The end of a call: the stream idle (the mesh complete, the scratch unused),
// and scratch beyond the bound returned.
void end_extract(kf_context* ctx) {
  const hipError_t err = hipStreamSynchronize(ctx->stream);
  for (;;) {
    size_t all = 0;
    DeviceBlock* longest = ctx->mesh_scratch;
    for (auto& b : ctx->mesh_scratch) {
      all += b.bytes;
      if (b.bytes > longest->bytes) longest = &b;
    }
    if (all <= kKeepBytes) break;
    (void)hipFree(longest->p);
    *longest = DeviceBlock{};
  }
  KF_HIP(err);
}

}  // namespace
}  // namespace kf

using namespace kf;

extern "C" {

kf_status kf_mesh_extract(kf_context* ctx, float min_weight, kf_mesh** out) {
  if (ctx == nullptr || out == nullptr) return KF_ERR_INVALID_ARGUMENT;
  *out = nullptr;
  auto* mesh = new (std::nothrow) kf_mesh();
  if (mesh == nullptr) return KF_ERR_OUT_OF_MEMORY;
  mesh->share = ctx->share;
  kf_status status = KF_OK;
  auto attempt = [&](auto&& body) {
    try {
      body();
    } catch (const Failure& f) {
      if (status != KF_OK) return;
      ctx->error = f.message;
      status = f.status;
    } catch (...) {
      if (status != KF_OK) return;
      ctx->error = "mesh extraction failed";
      status = KF_ERR_DEVICE;
    }
  };
  attempt([&] {
    switch (ctx->cfg.voxel_store) {
      case KF_VOXEL_QUANTIZED:
        extract_t<KF_VOXEL_QUANTIZED>(ctx, min_weight, mesh);
        break;
      case KF_VOXEL_BF16:
        extract_t<KF_VOXEL_BF16>(ctx, min_weight, mesh);
        break;
      default:
        extract_t<KF_VOXEL_FLOAT>(ctx, min_weight, mesh);
        break;
    }
  });
  attempt([&] { end_extract(ctx); });
  if (status != KF_OK) {
    delete mesh;
    return status;
  }
  *out = mesh;
  return KF_OK;
}

kf_status kf_mesh_size(const kf_mesh* mesh, int64_t* vertices, int64_t* triangles) {
  if (mesh == nullptr) return KF_ERR_INVALID_ARGUMENT;
  if (vertices != nullptr) *vertices = static_cast<int64_t>(mesh->vertices);
  if (triangles != nullptr) *triangles = static_cast<int64_t>(mesh->triangles);
  return KF_OK;
}

kf_status kf_mesh_copy(const kf_mesh* mesh, float* positions, float* normals, float* colors, uint32_t* triangles) {
  if (mesh == nullptr) return KF_ERR_INVALID_ARGUMENT;
  const size_t v = 12 * mesh->vertices;
  const HostStage::Piece out[4] = {{positions, mesh->positions(), v},
                                   {normals, mesh->normals(), v},
                                   {colors, mesh->colors(), v},
                                   {triangles, mesh->faces(), 12 * mesh->triangles}};
  if (mesh->vertices == 0) return KF_OK;
  const BesideCaptures allowed;
  const hipError_t err = mesh->share->stage.copy(out, 4, mesh->copies);
  return err == hipSuccess ? KF_OK : detached_error(err, "kf_mesh_copy");
}

void kf_mesh_free(kf_mesh* mesh) {
  const BesideCaptures allowed;
  delete mesh;
}

}  // extern "C"
