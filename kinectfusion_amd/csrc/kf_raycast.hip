// Raycaster (reference: SurfaceRaycast::render_pixel / find_zero_crossing /
// write_surface_sample, include/kinectfusion/raycasting.hpp:116-245;
// TrilinearSampler, volume_sampler.hpp:116-255; trilinear helpers,
// trilinear.hpp:85-269).
//
// One thread per pixel, a wave's rays a compact block of pixels (RayTile) so
// that they march through neighbouring voxels together.
// Corner blends visit the 2^3 stencil in z -> y -> x order with the
// reference's weight products, so every sample is bit-identical to the CPU
// sampler.
#include "kf_march.hpp"

namespace kf {
namespace {

template <int Kind, typename Store>
__global__ void __launch_bounds__(256) raycast_kernel(Sampler<Kind, Store> vol, RayParams rp, Rigid pose_arg,
                                                       IcpState* state, float4* __restrict__ pts,
                                                       float4* __restrict__ nrm, uint32_t* __restrict__ col,
                                                       const uint32_t* __restrict__ class_bits,
                                                       const uint32_t* __restrict__ nbr_obs, BlockMap bm,
                                                       const uint8_t* __restrict__ coarse, BlockMap cm,
                                                       int begin_level, RayTile shape) {
  Rigid pose = pose_arg;
  // the level's preparation touches neither frame_failed nor pose, which
  // every workgroup reads below
  if (begin_level >= 0 && state != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)
    icp_begin_level(state, begin_level);
  if (state != nullptr) {
    if (state->frame_failed) return;
    pose = rigid_from_pose64(state->pose);
  }
  // Workgroups are dealt to the 8 XCDs round-robin by their linear id, and
  // each XCD has its own L2: XCD k takes the k-th contiguous run of tiles
  // (row-major), so the rays that share volume blocks share an L2.  The map
  // is a bijection of [0, tiles) for any tile count.
  const int tiles = static_cast<int>(gridDim.x * gridDim.y);
  const int id = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
  const int q = tiles >> 3, r = tiles & 7, k = id & 7;
  const int tile = k * q + min(k, r) + (id >> 3);
  int x, y;
  if (!shape.pixel(tile, static_cast<int>(gridDim.x), static_cast<int>(threadIdx.x), x, y) || x >= rp.w || y >= rp.h)
    return;
  raycast_pixel(vol, rp, pose, x, y, pts, nrm, col, class_bits, nbr_obs, bm, coarse, cm);
}

// Rays per wave.  A dense store's waves are full: its lanes do much the same
// work at every pass, and fewer lanes only mean more waves.  512^3 bf16 room,
// 64, 32, 16 and 8 rays a wave: 325, 364, 429, 560 us at 640x480, 248, 254,
// 265, 299 at 320x240 and 173, 172, 172, 181 at 160x120 (float voxels alike;
// eight plain FP32 frames 4.07, 4.42, 5.22, 6.97 ms).
// A hashed store's rays diverge (a wave runs the sampler at nearly every pass
// for some lane), so where full waves leave the chip's wave slots empty, a
// wave takes fewer rays: at most kSlots waves, at least 8 rays each.  2048^3
// hall, 16 and 8 rays a wave instead of 64: 358 -> 334 us at 320x240, 324 ->
// 295 us at 160x120; 16 at 640x480 (19200 waves) was slower (554 -> 1017 us),
// as were 2 at 160x120 (400 -> 500 us).
RayTile ray_tile(int w, int h, bool hashed_store) {
  constexpr long long kSlots = 5120;  // 256 CUs x 4 SIMDs x 5 waves
  RayTile t{3, 3};
  if (!hashed_store) return t;
  auto waves = [&](int lanes_log2) { return (static_cast<long long>(w) * h) >> lanes_log2; };
  while (t.lw + t.lh > 3 && waves(t.lw + t.lh - 1) <= kSlots) {
    if (t.lw > t.lh || t.lh == 0) --t.lw;
    else --t.lh;
  }
  return t;
}

template <int Kind>
void launch_t(kf_context* ctx, const RayParams& rp, const Rigid& pose, IcpState* state,
              LevelBuffers& L, int begin_level) {
  using Raw = typename VoxelIO<Kind>::Raw;
  const RayTile shape = ray_tile(rp.w, rp.h, hashed(ctx));
  const dim3 grid((rp.w + shape.width() - 1) / shape.width(), (rp.h + shape.height() - 1) / shape.height());
  if (hashed(ctx)) {
    Sampler<Kind, HashedStore<Kind>> vol{
        HashedStore<Kind>{hash_view(ctx), static_cast<const Raw*>(ctx->voxels), ctx->colors}, ctx->grid,
        1.0F / ctx->grid.voxel};
    hipLaunchKernelGGL((raycast_kernel<Kind, HashedStore<Kind>>), grid, dim3(256), 0, ctx->stream, vol, rp, pose,
                       state, L.model_pts, L.model_nrm, L.model_col, ctx->class_bits, ctx->nbr_obs,
                       block_map(ctx->grid), ctx->coarse, coarse_map(ctx->grid), begin_level, shape);
    return;
  }
  Sampler<Kind> vol{DenseStore<Kind>{static_cast<const Raw*>(ctx->voxels), ctx->colors}, ctx->grid,
                    1.0F / ctx->grid.voxel};
  hipLaunchKernelGGL((raycast_kernel<Kind, DenseStore<Kind>>), grid, dim3(256), 0, ctx->stream, vol, rp, pose, state,
                     L.model_pts, L.model_nrm, L.model_col, ctx->class_bits, ctx->nbr_obs, block_map(ctx->grid),
                     ctx->coarse, coarse_map(ctx->grid), begin_level, shape);
}

}  // namespace

void launch_raycast(kf_context* ctx, int level, const double* /*unused*/, const Rigid* pose_host,
                    bool from_state, int begin_level) {
  const kf_config& c = ctx->cfg;
  LevelBuffers& L = ctx->lv[level];
  const RayParams rp = ray_params(ctx, level);
  const Rigid pose = pose_host != nullptr ? *pose_host : Rigid{};
  IcpState* state = from_state ? ctx->icp : nullptr;
  switch (c.voxel_store) {
    case KF_VOXEL_QUANTIZED:
      launch_t<KF_VOXEL_QUANTIZED>(ctx, rp, pose, state, L, begin_level);
      break;
    case KF_VOXEL_BF16:
      launch_t<KF_VOXEL_BF16>(ctx, rp, pose, state, L, begin_level);
      break;
    default:
      launch_t<KF_VOXEL_FLOAT>(ctx, rp, pose, state, L, begin_level);
      break;
  }
  KF_HIP(hipGetLastError());
}

}  // namespace kf
