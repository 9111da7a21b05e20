"""Hashed raycasts against the CPU oracle, bit for bit, over block grids whose
rows are and are not whole words, cells cut by the grid's edge, cameras from a
few waves to thousands (rays per wave change with the size), and views that
start outside the volume or look past the surfaces."""
import numpy as np
import pytest

from kf_helpers import RULE, STORE_KIND, host, pipeline_config, same_bits, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import kinectfusion_amd

    return kinectfusion_amd


def moved(pose, t, yaw=0.0):
    out = np.array(pose, np.float64)
    c, s = np.cos(yaw), np.sin(yaw)
    out[:3, :3] = out[:3, :3] @ np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]])
    out[:3, 3] += t
    return out


@pytest.mark.parametrize("res,voxel,store,color", [((256, 256, 256), 0.01, "float", "none"),
                                                   ((264, 200, 328), 0.008, "bf16", "float"),
                                                   ((72, 520, 100), 0.02, "quantized", "none")])
@pytest.mark.parametrize("size", [(640, 480), (203, 151), (33, 20)])
def test_hashed_raycast_over_grids_and_cameras(K, ko, torch_gpu, res, voxel, store, color, size):
    w, h = size
    intr = (525.0 * w / 640, 525.0 * w / 640, 0.5 * (w - 1), 0.5 * (h - 1))
    origin = (-voxel * res[0] / 2, -voxel * res[1] / 2, -0.5)
    cfg = pipeline_config(K, store=store, color=color, voxel=voxel, storage="hashed", hash_buckets=1 << 16,
                          block_capacity=16384, levels=1)
    cfg.volume = K.VolumeGeometry(res, voxel, origin, 0.05)
    cfg.intrinsics, cfg.width, cfg.height = K.CameraIntrinsics(*intr), w, h
    p = K.Pipeline(cfg)
    vol = ko.SparseVolume.create_sparse(res, voxel, origin, 0.05, STORE_KIND[store], color == "float", capacity=16384)
    scene = K.SyntheticScene("room", seed=5, width=w, height=h, fx=intr[0], fy=intr[1], cx=intr[2], cy=intr[3])
    for i in (0, 12):
        depth, rgba, pose = scene.frame(i)
        w2c = ko.rigid_inverse(pose)
        img = rgba if color == "float" else None
        ko.integrate_sparse(vol, RULE["angle-weighted"], depth, intr, w2c, ko.integration_options(1000.0), color=img)
        p.integrate(to_dev(torch_gpu, depth), w2c, color=to_dev(torch_gpu, img) if img is not None else None)
    hits = 0
    for pose in (scene.pose(6), moved(scene.pose(0), [0.3, -0.2, -1.5]), moved(scene.pose(0), [0, 0, 0.2], 1.3)):
        maps = p.raycast(pose, 0)
        pts, nrm, col, _ = ko.raycast(vol, pose, intr, w, h)
        hits += int(np.isfinite(pts).all(-1).sum())
        assert same_bits(host(maps.points)[..., :3], pts) and same_bits(host(maps.normals)[..., :3], nrm)
        assert np.array_equal(host(maps.colors).view(np.uint32), col)
    assert hits > w * h // 4
    p.close()
