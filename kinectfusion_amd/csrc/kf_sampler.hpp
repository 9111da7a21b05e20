// Trilinear TSDF sampler over the dense voxel array or the hashed block pool
// (reference: TrilinearSampler + DenseCornerAccess / SparseCornerAccess, include/kinectfusion/
// volume_sampler.hpp:36-255; blend_tsdf / blend_color / cell_gradient /
// central_normal, trilinear.hpp:85-269).  Shared by the raycaster and the
// mesher so both read the volume with the same float operations as the CPU
// sampler: the 2^3 stencil is visited z -> y -> x and each corner weight is
// ((wx * wy) * wz).
#pragma once

#include "kf_internal.hpp"

namespace kf {

// Corner access (DenseCornerAccess / SparseCornerAccess,
// volume_sampler.hpp:36-109 and block_rep.hpp:113-160).  A voxel of an
// unallocated block reads as a fresh voxel and a colour voxel as zero: the
// blends treat both exactly like the reference's missing (null) corners.
// The last block that voxel_cached looked up in a hashed store (key, pool
// slot).
struct SlotCache {
  uint32_t key = kNoSlot;
  uint32_t slot = kNoSlot;
};

// Two x-neighbouring voxels as one vector load (x-fastest layout: they are
// adjacent in memory; the pair is only as aligned as one voxel).
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

template <typename Raw>
__device__ inline void load_pair(const Raw* p, Raw& a, Raw& b);
template <>
__device__ inline void load_pair<uint32_t>(const uint32_t* p, uint32_t& a, uint32_t& b) {
  const u32x2_a4 v = *reinterpret_cast<const u32x2_a4*>(p);
  a = v.x;
  b = v.y;
}
template <>
__device__ inline void load_pair<float2>(const float2* p, float2& a, float2& b) {
  const f32x4_a8 v = *reinterpret_cast<const f32x4_a8*>(p);
  a = make_float2(v.x, v.y);
  b = make_float2(v.z, v.w);
}

template <int Kind>
struct DenseStore {
  using Raw = typename VoxelIO<Kind>::Raw;
  static constexpr bool kDirect = true;  // a voxel is one load
  const Raw* __restrict__ vox;
  const float4* __restrict__ colors;
  __device__ inline Raw voxel(const Grid& g, int x, int y, int z) const { return vox[g.flat(x, y, z)]; }
  // The eight corners of the cell at (x, y, z) (z -> y -> x order), all
  // inside the grid: one 64-bit index, then four x-pair loads at fixed
  // row and slice offsets.
  __device__ inline void cell(const Grid& g, int x, int y, int z, Raw (&raw)[8]) const {
    const Raw* p = vox + g.flat(x, y, z);
    const size_t row = static_cast<size_t>(g.nx), slice = static_cast<size_t>(g.nx) * static_cast<size_t>(g.ny);
    load_pair<Raw>(p, raw[0], raw[1]);
    load_pair<Raw>(p + row, raw[2], raw[3]);
    load_pair<Raw>(p + slice, raw[4], raw[5]);
    load_pair<Raw>(p + slice + row, raw[6], raw[7]);
  }
  __device__ inline Raw voxel_cached(const Grid& g, int x, int y, int z, SlotCache&) const { return voxel(g, x, y, z); }
  // The colour voxels of the corners of the 2^3 stencil with base corner
  // (x, y, z), four of them (z fixed): a corner outside the grid reads a
  // clamped one, which the caller drops.
  __device__ inline void colors4(const Grid& g, int x, int y, int z, float4 (&c)[4]) const {
    const int x0 = min(max(x, 0), g.nx - 1), x1 = min(x + 1, g.nx - 1), y0 = min(max(y, 0), g.ny - 1),
              y1 = min(y + 1, g.ny - 1), zc = min(max(z, 0), g.nz - 1);
    c[0] = colors[g.flat(x0, y0, zc)];
    c[1] = colors[g.flat(x1, y0, zc)];
    c[2] = colors[g.flat(x0, y1, zc)];
    c[3] = colors[g.flat(x1, y1, zc)];
  }
  __device__ inline bool has_colors() const { return colors != nullptr; }
};

template <int Kind>
struct HashedStore {
  using Raw = typename VoxelIO<Kind>::Raw;
  static constexpr bool kDirect = false;  // a voxel needs its block's slot first
  HashView hv;
  const Raw* __restrict__ pool;
  const float4* __restrict__ cpool;
  __device__ inline uint32_t slot_of(int x, int y, int z, SlotCache& cache) const {
    const uint32_t key = hv.key_of(x, y, z);
    if (key != cache.key) {
      cache.key = key;
      cache.slot = hv.slots[key];
    }
    return cache.slot;
  }
  // A corner's voxel: an unallocated block's read goes to slot 0 and is
  // replaced, since a guarded read would wait for the one before it.
  __device__ inline size_t at(uint32_t slot, int x, int y, int z) const {
    return static_cast<size_t>(slot == kNoSlot ? 0U : slot) * kBlockVoxels + intra_of(x, y, z);
  }
  __device__ inline Raw voxel_cached(const Grid&, int x, int y, int z, SlotCache& cache) const {
    const uint32_t slot = slot_of(x, y, z, cache);
    const Raw v = pool[at(slot, x, y, z)];
    return slot == kNoSlot ? VoxelIO<Kind>::fresh() : v;
  }
  __device__ inline bool has_colors() const { return cpool != nullptr; }
  // The pool slots of the corners of the 2^3 stencil with base corner (x, y, z)
  // in the z-layer z, x fastest: two x-neighbouring index entries per read
  // (the index has one entry to spare).  Corners outside the grid read a
  // clamped block's slot, which the caller drops.
  __device__ inline void slots4(const Grid& g, int x, int y, int z, uint32_t (&slot)[4]) const {
    const int x0 = max(x, 0) >> 3, x1 = min(x + 1, g.nx - 1) >> 3, y0 = max(y, 0) >> 3, y1 = min(y + 1, g.ny - 1) >> 3,
              zc = min(max(z, 0), g.nz - 1) >> 3;
    const uint32_t* p = hv.slots + (static_cast<size_t>(zc) * hv.by + y0) * hv.bx + x0;
    const u32x2_a4 a = *reinterpret_cast<const u32x2_a4*>(p);
    const u32x2_a4 b = *reinterpret_cast<const u32x2_a4*>(p + (y1 != y0 ? hv.bx : 0));
    slot[0] = a.x;
    slot[1] = x1 != x0 ? a.y : a.x;
    slot[2] = b.x;
    slot[3] = x1 != x0 ? b.y : b.x;
  }
  __device__ inline void colors4(const Grid& g, int x, int y, int z, float4 (&c)[4]) const {
    uint32_t slot[4];
    slots4(g, x, y, z, slot);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = cpool[at(slot[i], x + (i & 1), y + (i >> 1), z)];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (slot[i] == kNoSlot) c[i] = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
  }
};

template <int Kind, typename Store = DenseStore<Kind>>
struct Sampler {
  using IO = VoxelIO<Kind>;
  Store s;
  Grid g;
  float inv_voxel;

  __device__ inline bool contains(V3 p) const {
    // one condition, not six branches
    return (static_cast<int>(p.x >= 0.0F) & static_cast<int>(p.y >= 0.0F) & static_cast<int>(p.z >= 0.0F) &
            static_cast<int>(p.x < static_cast<float>(g.nx)) & static_cast<int>(p.y < static_cast<float>(g.ny)) &
            static_cast<int>(p.z < static_cast<float>(g.nz))) != 0;
  }
  __device__ inline V3 grid_coords(V3 p) const {
    return scale3(sub3(p, mk3(g.ox, g.oy, g.oz)), inv_voxel);
  }
  __device__ static inline float axis_w(float f, int o) { return o == 0 ? 1.0F - f : f; }

  // The 2^3 stencil of a point: base corner, fractions, in-volume flag.
  struct Stencil {
    int bx, by, bz;
    V3 fr;
    bool ok;        // the point lies inside the grid
    bool interior;  // all eight corners lie inside the grid
  };
  __device__ inline Stencil stencil(V3 p) const { return stencil_gc(grid_coords(p)); }
  // the same from grid coordinates already computed
  __device__ inline Stencil stencil_gc(V3 gc) const {
    Stencil st;
    st.ok = contains(gc);
    const V3 gg = sub3(gc, mk3(0.5F, 0.5F, 0.5F));
    const V3 fl = mk3(floorf(gg.x), floorf(gg.y), floorf(gg.z));
    st.bx = static_cast<int>(fl.x);
    st.by = static_cast<int>(fl.y);
    st.bz = static_cast<int>(fl.z);
    st.fr = sub3(gg, fl);
    st.interior = (static_cast<int>(st.bx >= 0) & static_cast<int>(st.by >= 0) & static_cast<int>(st.bz >= 0) &
                   static_cast<int>(st.bx + 1 < g.nx) & static_cast<int>(st.by + 1 < g.ny) &
                   static_cast<int>(st.bz + 1 < g.nz)) != 0;
    return st;
  }
  // Bit c (x fastest): corner c of the stencil lies inside the grid.
  __device__ inline unsigned corners_inside(const Stencil& st) const {
    const unsigned mx = (st.bx >= 0 ? 0x55U : 0U) | (st.bx + 1 < g.nx ? 0xAAU : 0U);
    const unsigned my = (st.by >= 0 ? 0x33U : 0U) | (st.by + 1 < g.ny ? 0xCCU : 0U);
    const unsigned mz = (st.bz >= 0 ? 0x0FU : 0U) | (st.bz + 1 < g.nz ? 0xF0U : 0U);
    return mx & my & mz;
  }
  // Loads of the eight corners (z -> y -> x order); bit c of `inb` marks a
  // corner inside the grid.
  __device__ inline void load8(const Stencil& st, typename IO::Raw (&raw)[8], unsigned& inb) const {
    if constexpr (Store::kDirect) {
      if (st.ok && st.interior) {  // four x-pairs
        s.cell(g, st.bx, st.by, st.bz, raw);
        inb = 0xFFU;
        return;
      }
      inb = 0U;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int x = st.bx + (c & 1), y = st.by + ((c >> 1) & 1), z = st.bz + (c >> 2);
        raw[c] = IO::fresh();
        if (!st.ok) continue;
        if (!st.interior && (x < 0 || y < 0 || z < 0 || x >= g.nx || y >= g.ny || z >= g.nz)) continue;
        raw[c] = s.voxel(g, x, y, z);
        inb |= 1U << c;
      }
    } else {
      // the eight slots in one round of reads, then the eight voxels
      inb = corners_inside(st);
      if (!st.ok) return;
      uint32_t lo[4], hi[4];
      s.slots4(g, st.bx, st.by, st.bz, lo);
      s.slots4(g, st.bx, st.by, st.bz + 1, hi);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        raw[c] = s.pool[s.at(c < 4 ? lo[c & 3] : hi[c & 3], st.bx + (c & 1), st.by + ((c >> 1) & 1), st.bz + (c >> 2))];
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if ((c < 4 ? lo[c & 3] : hi[c & 3]) == kNoSlot) raw[c] = IO::fresh();
    }
  }
  // blend_tsdf over loaded corners, without branches: a corner outside the
  // grid (its bit of inb clear), unobserved or not finite adds +0 to both sums,
  // which leaves them unchanged (neither sum is ever -0: they start at +0 and
  // a round-to-nearest sum is -0 only when both terms are).  All: every corner
  // lies inside the grid (inb is not looked at; a separate instance, so that
  // the march's common case carries no corner mask).
  template <bool All = false>
  __device__ inline bool blend(const Stencil& st, const typename IO::Raw (&raw)[8], unsigned inb, bool require_all,
                               float& out) const {
    float acc = 0.0F, wsum = 0.0F;
    int valid = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      float t, w;
      bool obs, fin;
      IO::unpack(raw[c], t, w, obs, fin);
      const unsigned in = All ? 1U : inb >> c;
      const bool use = (static_cast<unsigned>(obs) & static_cast<unsigned>(fin) & in) != 0U;
      const float cw = axis_w(st.fr.x, c & 1) * axis_w(st.fr.y, (c >> 1) & 1) * axis_w(st.fr.z, c >> 2);
      acc += use ? cw * t : 0.0F;
      wsum += use ? cw : 0.0F;
      valid += use ? 1 : 0;
    }
    if (!st.ok || (require_all && valid < 8)) return false;
    if (wsum <= 1.0e-6F) return false;
    const float d = acc / wsum;
    if (!isfinite(d)) return false;
    out = d;
    return true;
  }

  // The same of a cell at the grid's edge, corner by corner.
  __device__ inline bool blend_edge(const Stencil& st, const typename IO::Raw (&raw)[8], unsigned inb, bool require_all,
                               float& out) const {
    if (!st.ok) return false;
    float acc = 0.0F, wsum = 0.0F;
    int valid = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (((inb >> c) & 1U) == 0U) continue;
      float t, w;
      bool obs, fin;
      IO::unpack(raw[c], t, w, obs, fin);
      if (!obs || !fin) continue;
      const float cw = axis_w(st.fr.x, c & 1) * axis_w(st.fr.y, (c >> 1) & 1) * axis_w(st.fr.z, c >> 2);
      acc += cw * t;
      wsum += cw;
      ++valid;
    }
    if (require_all && valid < 8) return false;
    if (wsum <= 1.0e-6F) return false;
    const float d = acc / wsum;
    if (!isfinite(d)) return false;
    out = d;
    return true;
  }
  // TrilinearSampler::tsdf + blend_tsdf.
  __device__ bool tsdf(V3 p, bool require_all, float& out) const {
    const Stencil st = stencil(p);
    if (!st.ok) return false;
    typename IO::Raw raw[8];
    if constexpr (Store::kDirect) {
      // the eight corners as four x-pair loads
      if (st.interior) {
        s.cell(g, st.bx, st.by, st.bz, raw);
        return blend<true>(st, raw, 0xFFU, require_all, out);
      }
    }
    unsigned inb;
    load8(st, raw, inb);
    // the two blends of a direct store must not share code: merged, the march's
    // interior cells wait for this path's registers (60 -> 68 us at 160x120)
    if constexpr (Store::kDirect) return blend_edge(st, raw, inb, require_all, out);
    else return blend(st, raw, inb, require_all, out);
  }

  // blend_color.
  __device__ bool color(V3 p, V3& out) const {
    if (!s.has_colors()) return false;
    const V3 gc = grid_coords(p);
    if (!contains(gc)) return false;
    const V3 gg = sub3(gc, mk3(0.5F, 0.5F, 0.5F));
    const V3 fl = mk3(floorf(gg.x), floorf(gg.y), floorf(gg.z));
    const int bx = static_cast<int>(fl.x), by = static_cast<int>(fl.y), bz = static_cast<int>(fl.z);
    const V3 fr = sub3(gg, fl);
    V3 acc = mk3(0.0F, 0.0F, 0.0F);
    float wsum = 0.0F;
    float4 c[2][4];
    s.colors4(g, bx, by, bz, c[0]);
    s.colors4(g, bx, by, bz + 1, c[1]);
#pragma unroll
    for (int oz = 0; oz <= 1; ++oz)
#pragma unroll
      for (int oy = 0; oy <= 1; ++oy)
#pragma unroll
        for (int ox = 0; ox <= 1; ++ox) {
          const int x = bx + ox, y = by + oy, z = bz + oz;
          const float4 v = c[oz][oy * 2 + ox];
          if (x < 0 || y < 0 || z < 0 || x >= g.nx || y >= g.ny || z >= g.nz || v.w <= 0.0F) continue;
          const float cw = axis_w(fr.x, ox) * axis_w(fr.y, oy) * axis_w(fr.z, oz);
          acc = add3(acc, scale3(mk3(v.x, v.y, v.z), cw));
          wsum += cw;
        }
    if (wsum <= 1.0e-6F) return false;
    out = div3(acc, wsum);
    return true;
  }

  // central_normal (trilinear.hpp:246-269).  The corner loads of the two
  // samples of an axis are issued together; the blends run in the
  // reference's order.  Two samples at a time (not all six) bound the
  // register use of the raycaster, where the normal's peak would otherwise
  // set the register allocation, and so the occupancy, of the whole march.
  __device__ __forceinline__ bool normal(V3 p, bool require_all, V3& out) const {
    V3 dir = mk3(0.0F, 0.0F, 0.0F);
    if constexpr (Store::kDirect) {
      float v[6];
#pragma unroll
      for (int a0 = 0; a0 < 6; a0 += 2) {
        Stencil st[2];
        typename IO::Raw raw[2][8];
        unsigned inb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int axis = (a0 + i) >> 1;
          const V3 off = scale3(mk3(axis == 0 ? 1.0F : 0.0F, axis == 1 ? 1.0F : 0.0F, axis == 2 ? 1.0F : 0.0F), g.voxel);
          st[i] = stencil(((a0 + i) & 1) == 0 ? add3(p, off) : sub3(p, off));
          load8(st[i], raw[i], inb[i]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (!blend(st[i], raw[i], inb[i], require_all, v[a0 + i])) return false;
      }
      dir = mk3(v[0] - v[1], v[2] - v[3], v[4] - v[5]);
    } else {
      // one sample at a time in a loop that is not unrolled: unrolled, the six
      // (when a slot took a probe of the table and a walk) were 54 KB of code, a
      // call out of the march that kept the sampler in scratch memory for all of
      // it
      float plus = 0.0F;
#pragma unroll 1
      for (int k = 0; k < 6; ++k) {
        const int axis = k >> 1;
        const V3 off = scale3(mk3(axis == 0 ? 1.0F : 0.0F, axis == 1 ? 1.0F : 0.0F, axis == 2 ? 1.0F : 0.0F), g.voxel);
        const Stencil st = stencil((k & 1) == 0 ? add3(p, off) : sub3(p, off));
        typename IO::Raw raw[8];
        unsigned inb;
        load8(st, raw, inb);
        float v;
        if (!blend(st, raw, inb, require_all, v)) return false;
        const float d = plus - v;
        if ((k & 1) == 0) plus = v;
        else if (axis == 0) dir.x = d;
        else if (axis == 1) dir.y = d;
        else dir.z = d;
      }
    }
    const float len = norm3(dir);
    if (len <= 0.0F) return false;
    out = div3(dir, len);
    return true;
  }

  // cell_normal + cell_gradient (volume_sampler.hpp:189-239).
  __device__ bool cell_normal(V3 p, V3& out) const {
    const V3 gc = grid_coords(p);
    if (!contains(gc)) return false;
    const V3 gg = sub3(gc, mk3(0.5F, 0.5F, 0.5F));
    const V3 fl = mk3(floorf(gg.x), floorf(gg.y), floorf(gg.z));
    const int bx = static_cast<int>(fl.x), by = static_cast<int>(fl.y), bz = static_cast<int>(fl.z);
    const V3 f = sub3(gg, fl);
    float c[2][2][2];
    bool complete = true;
    SlotCache cache;
#pragma unroll
    for (int oz = 0; oz <= 1; ++oz)
#pragma unroll
      for (int oy = 0; oy <= 1; ++oy)
#pragma unroll
        for (int ox = 0; ox <= 1; ++ox) {
          const int x = bx + ox, y = by + oy, z = bz + oz;
          c[oz][oy][ox] = 0.0F;
          if (x < 0 || y < 0 || z < 0 || x >= g.nx || y >= g.ny || z >= g.nz) {
            complete = false;
            continue;
          }
          float t, w;
          bool obs, fin;
          IO::unpack(s.voxel_cached(g, x, y, z, cache), t, w, obs, fin);
          if (!obs || !fin) complete = false;
          c[oz][oy][ox] = t;
        }
    if (!complete) return normal(p, false, out);
    auto lerp2 = [](float lo, float hi, float m) { return lo + (m * (hi - lo)); };
    const float gx = lerp2(lerp2(c[0][0][1] - c[0][0][0], c[0][1][1] - c[0][1][0], f.y),
                           lerp2(c[1][0][1] - c[1][0][0], c[1][1][1] - c[1][1][0], f.y), f.z);
    const float gy = lerp2(lerp2(c[0][1][0] - c[0][0][0], c[0][1][1] - c[0][0][1], f.x),
                           lerp2(c[1][1][0] - c[1][0][0], c[1][1][1] - c[1][0][1], f.x), f.z);
    const float gz = lerp2(lerp2(c[1][0][0] - c[0][0][0], c[1][0][1] - c[0][0][1], f.x),
                           lerp2(c[1][1][0] - c[0][1][0], c[1][1][1] - c[0][1][1], f.x), f.y);
    const V3 grad = mk3(gx, gy, gz);
    const float len = norm3(grad);
    if (len <= 0.0F) return false;
    out = div3(grad, len);
    return true;
  }
};

}  // namespace kf
