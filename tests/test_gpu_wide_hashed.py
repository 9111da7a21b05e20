"""Hashed raycasts over a grid wider than 2048 voxels in x, whose rows of cells
are more than one 64-bit word, against the CPU oracle bit for bit: two walls on
either side of the words' seam (x = 2048), seen along x from both ends through
the unobserved space between them."""
import numpy as np
import pytest

from kf_helpers import RULE, STORE_KIND, host, pipeline_config, same_bits, to_dev

pytestmark = pytest.mark.gpu

VOXEL = 0.005
SIZE = 64  # pixels a side
INTR = (700.0, 700.0, 31.5, 31.5)


def looking_along_x(x, sign, yz):
    """Camera to world: the optical axis along +x or -x, at voxel x."""
    out = np.eye(4)
    out[:3, :3] = np.array([[0, 0, sign], [0, 1, 0], [-sign, 0, 0]], np.float64)
    out[:3, 3] = [x * VOXEL, yz * VOXEL, yz * VOXEL]
    return out


# the nearest wall in the next word, or in the one before, though the other is
# in the ray's own
@pytest.mark.parametrize("nx,walls", [(2312, (1700, 2070)), (2312, (2020, 2200)), (2312, (1950, 2076)),
                                      (2080, (1700, 2070)), (2080, (2020, 2060)), (4096, (2020, 2200))])
def test_rays_across_the_words_of_a_row(ko, torch_gpu, nx, walls):
    import kinectfusion_amd as K

    res = (nx, 64, 64)
    cfg = pipeline_config(K, store="bf16", color="none", voxel=VOXEL, storage="hashed", hash_buckets=1 << 14,
                          block_capacity=4096, levels=1)
    cfg.volume = K.VolumeGeometry(res, VOXEL, (0.0, 0.0, 0.0), 0.02)
    cfg.intrinsics, cfg.width, cfg.height = K.CameraIntrinsics(*INTR), SIZE, SIZE
    p = K.Pipeline(cfg)
    vol = ko.SparseVolume.create_sparse(res, VOXEL, (0.0, 0.0, 0.0), 0.02, STORE_KIND["bf16"], False, capacity=4096)
    for i, wall in enumerate(walls):
        for sign in (1, -1):  # seen from both sides, each wall over its half of the image
            pose = looking_along_x(wall - sign * 200, sign, 32.0)
            depth = np.full((SIZE, SIZE), int(round(200 * VOXEL * 1000)), np.uint16)
            depth[: SIZE // 2] *= i == 0
            depth[SIZE // 2:] *= i == 1
            w2c = ko.rigid_inverse(pose)
            ko.integrate_sparse(vol, RULE["angle-weighted"], depth, INTR, w2c, ko.integration_options(1000.0))
            p.integrate(to_dev(torch_gpu, depth), w2c)
    for x, sign in ((walls[0] - 500, 1), (walls[0] - 37, 1), (min(walls[1] + 200, nx - 1), -1), (walls[1] + 3, -1), (walls[0] + 10, 1)):
        pose = looking_along_x(x, sign, 31.0)
        maps = p.raycast(pose, 0)
        pts, nrm, _, _ = ko.raycast(vol, pose, INTR, SIZE, SIZE)
        hit = np.isfinite(pts).all(-1)
        if x == walls[0] - 500 or (sign < 0 and x == walls[1] + 200):  # both walls, so rays that cross the seam
            seen = np.round(pts[hit][:, 0] / VOXEL)
            assert all(np.any(np.abs(seen - w) < 8) for w in walls), (x, sign, np.unique(seen))
        assert same_bits(host(maps.points)[..., :3], pts) and same_bits(host(maps.normals)[..., :3], nrm)
    p.close()
