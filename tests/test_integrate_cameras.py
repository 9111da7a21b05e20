"""The integration's projection test over cameras: the margin that depends on
the image and not on the voxel, on the CPU with the worst-case error of the
hardware reciprocal (relative 2^-21), and on the device whole volumes against
the CPU oracle, bit for bit, for images from one pixel to thousands wide,
principal points off centre and outside, and both kinds of distance."""
import numpy as np
import pytest

from kf_helpers import STORE_KIND, first_mismatch, same_bits, to_dev

F = np.float32


@pytest.mark.parametrize("width,cx,fx", [(640, 319.5, 525.0), (1, 0.0, 1.0), (33, -200.0, 60.0), (33, 250.0, 60.0),
                                         (4096, 2047.5, 3300.0), (9000, 100.0, 7000.0)])
@pytest.mark.parametrize("aim", ["anywhere", "half-integers", "far"])
def test_margin_of_the_image(width, cx, fx, aim):
    rng = np.random.default_rng(width)
    n = 200_000
    fx, cx = F(fx), F(cx)
    z = rng.uniform(0.05, 6, n).astype(F)
    if aim == "anywhere":
        target = rng.uniform(-2, width + 2, n)
    elif aim == "half-integers":
        target = rng.integers(-3, width + 3, n) + 0.5 + rng.uniform(-4e-3, 4e-3, n)
    else:
        target = rng.uniform(-1, 1, n) * 10.0 ** rng.uniform(1, 8, n)
    x = ((target - float(cx)) * z / float(fx)).astype(F)
    a = (fx * x).astype(F)
    exact_u = ((a / z).astype(F) + cx).astype(F).astype(np.float64)
    exact = np.where(exact_u >= 0, np.floor(exact_u + 0.5), -np.floor(-exact_u + 0.5))
    exact = np.where((exact >= 0) & (exact < width), exact, -1)
    near = 0.5 - (3e-4 + 2e-6 * (max(abs(float(cx)), abs(width - float(cx))) + 1))
    for e in (-2.0 ** -21, 0.0, 2.0 ** -21):
        u = (a.astype(np.float64) * (1 / z.astype(np.float64)).astype(F) * (1 + e) + float(cx)).astype(F)
        nu = np.rint(u)
        safe = np.abs(u - nu) < F(near)
        fast = np.where((nu >= 0) & (nu < width), nu, -1)
        assert np.array_equal(fast[safe], exact[safe])


@pytest.mark.gpu
@pytest.mark.parametrize("size,intr", [((1, 1), (20.0, 20.0, 0.0, 0.0)), ((17, 5), (30.0, 28.0, 8.0, 2.0)),
                                       ((64, 48), (60.0, 60.0, -20.0, 70.0)), ((2500, 9), (2000.0, 15.0, 1250.0, 4.0))])
@pytest.mark.parametrize("store,color,projective,scaled", [("float", "float", True, False),
                                                           ("bf16", "none", True, True),
                                                           ("quantized", "float", False, True)])
def test_volumes_over_cameras(ko, torch_gpu, size, intr, store, color, projective, scaled):
    import kinectfusion_amd as K

    w, h = size
    res, voxel, origin, trunc = (37, 30, 45), 0.03, (-0.5, -0.4, 0.2), 0.08
    cfg = K.PipelineConfig(voxel=store, tsdf_rule="classic", color=color,
                           volume=K.VolumeGeometry(res, voxel, origin, trunc),
                           integration=K.TsdfIntegrationOptions(depth_scale=1000.0, mode="full"),
                           depth=K.DepthProcessingOptions(levels=1), intrinsics=K.CameraIntrinsics(*intr), width=w,
                           height=h)
    cfg.integration.projective_distance, cfg.integration.distance_scaled_truncation = projective, scaled
    opts = ko.integration_options(1000.0, projective_distance=int(projective), distance_scaled_truncation=int(scaled))
    p = K.Pipeline(cfg)
    vol = ko.Volume.create(res, voxel, origin, trunc, STORE_KIND[store], color == "float")
    rng = np.random.default_rng(w)
    for i in range(3):
        depth = rng.integers(600, 1500, (h, w)).astype(np.uint16)
        depth[rng.random((h, w)) < 0.1] = 0
        rgba = rng.integers(0, 1 << 24, (h, w)).astype(np.uint32)
        w2c = np.eye(4)
        w2c[:3, 3] = [0.02 * i, -0.01 * i, 0.05 * i]
        n_ref = ko.integrate(vol, 0, depth, intr, w2c, opts, color=rgba)
        n_gpu = p.integrate(to_dev(torch_gpu, depth), w2c, color=to_dev(torch_gpu, rgba), count=True)
        assert tuple(n_gpu) == n_ref
    vox, col = p.host_view()
    assert np.array_equal(vox.view(np.uint8), vol.voxels.view(np.uint8)), first_mismatch(vox, vol.voxels)
    if color == "float":
        assert same_bits(col, vol.colors)
    p.close()
