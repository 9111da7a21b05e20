"""Marching cubes at the edges of its word and block layouts, against the CPU
mesher bit for bit: rows shorter than, equal to and just past a 64-voxel word,
every cube case (random signs), unobserved, under-weight and non-finite
voxels, and hashed grids whose extents are no multiple of the block edge."""
import numpy as np
import pytest

from kf_helpers import INTR, RULE, STORE_KIND, pipeline_config, same_bits, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import kinectfusion_amd

    return kinectfusion_amd


def check(gpu, ref):
    pos, nrm, col, tri = ref
    assert np.array_equal(gpu.triangles, tri)
    assert same_bits(gpu.positions, pos) and same_bits(gpu.normals, nrm) and same_bits(gpu.colors, col)


def random_volume(ko, res, store, color, seed):
    """Voxels with random signs, one in eight unobserved, weights around the
    mesher's bar, and (float store) a few non-finite distances."""
    rng = np.random.default_rng(seed)
    vol = ko.Volume.create(res, 0.01, (-0.3, 0.1, 0.2), 0.05, STORE_KIND[store], color)
    n = int(np.prod(res))
    t = rng.uniform(-1.0, 1.0, n).astype(np.float32)
    w = rng.choice([0.0, 0.5, 1.0, 3.0], n, p=[0.125, 0.25, 0.25, 0.375]).astype(np.float32)
    if store == "float":
        t[rng.integers(0, n, max(1, n // 64))] = np.float32("nan")
        vol.voxels[:, 0], vol.voxels[:, 1] = t, w
    else:
        enc = (t * 32767.0).astype(np.int16).view(np.uint16) if store == "quantized" else (t.view(np.uint32) >> 16)
        vol.voxels[:, 0], vol.voxels[:, 1] = enc.astype(np.uint16), (w * 256.0).astype(np.uint16)
    if color:
        vol.colors[:, :3] = rng.uniform(0.0, 255.0, (n, 3))
        vol.colors[:, 3] = w
    return vol


@pytest.mark.parametrize("store,color", [("float", True), ("quantized", False), ("bf16", True)])
@pytest.mark.parametrize("res", [(2, 2, 2), (64, 9, 5), (65, 8, 7), (63, 5, 12), (129, 6, 4), (3, 70, 5)])
def test_dense_mesh_of_random_voxels(K, ko, torch_gpu, store, color, res):
    vol = random_volume(ko, res, store, color, seed=sum(res))
    cfg = K.PipelineConfig(voxel=store, color="float" if color else "none",
                           volume=K.VolumeGeometry(res, 0.01, (-0.3, 0.1, 0.2), 0.05))
    p = K.Pipeline(cfg)
    p.upload_volume(vol.voxels, vol.colors)
    for min_weight in (0.0, 1.0):
        check(p.extract_mesh(min_weight), ko.mesh(vol, min_weight))
    # a second, smaller mesh from the same context reuses its scratch
    vol.voxels[len(vol.voxels) // 2:, 1] = 0
    p.upload_volume(vol.voxels, vol.colors)
    check(p.extract_mesh(0.0), ko.mesh(vol, 0.0))
    p.close()


@pytest.mark.parametrize("store", ["float", "bf16"])
@pytest.mark.parametrize("res", [(100, 93, 117), (128, 128, 128)])
def test_hashed_mesh_of_partial_blocks(K, ko, torch_gpu, store, res):
    voxel, origin = 0.02, (-0.02 * res[0] / 2, -0.02 * res[1] / 2, -0.5)
    cfg = pipeline_config(K, store=store, voxel=voxel, storage="hashed", hash_buckets=1 << 16, block_capacity=8192)
    cfg.volume = K.VolumeGeometry(res, voxel, origin, 0.05)
    p = K.Pipeline(cfg)
    vol = ko.SparseVolume.create_sparse(res, voxel, origin, 0.05, STORE_KIND[store], True, capacity=8192)
    assert len(p.extract_mesh().triangles) == 0  # nothing allocated
    scene = K.SyntheticScene("room", seed=3)
    for i in range(2):
        depth, rgba, pose = scene.frame(8 * i)
        w2c = ko.rigid_inverse(pose)
        ko.integrate_sparse(vol, RULE["angle-weighted"], depth, INTR, w2c, ko.integration_options(1000.0), color=rgba)
        p.integrate(to_dev(torch_gpu, depth), w2c, color=to_dev(torch_gpu, rgba))
        for min_weight in (0.0, 1.5):
            ref = ko.mesh(vol, min_weight)
            assert min_weight > 0 or len(ref[3]) > 1000
            check(p.extract_mesh(min_weight), ref)
    p.close()


def test_mesh_outlives_its_context(K, ko, torch_gpu):
    """A mesh handle holds its own memory: it is copied after the context that
    made it is gone."""
    import ctypes as C

    from kinectfusion_amd import _native as N

    vol = random_volume(ko, (40, 30, 20), "bf16", False, seed=1)
    p = K.Pipeline(K.PipelineConfig(voxel="bf16", color="none",
                                    volume=K.VolumeGeometry((40, 30, 20), 0.01, (-0.3, 0.1, 0.2), 0.05)))
    p.upload_volume(vol.voxels)
    lib, h, nv, nt = N.hip(), C.c_void_p(), C.c_int64(), C.c_int64()
    N.check(lib.kf_mesh_extract(p.ctx, 0.0, C.byref(h)), p.ctx)
    p.close()
    N.check(lib.kf_mesh_size(h, C.byref(nv), C.byref(nt)))
    pos, tri = np.empty((nv.value, 3), np.float32), np.empty((nt.value, 3), np.uint32)
    N.check(lib.kf_mesh_copy(h, pos.ctypes.data_as(C.c_void_p), None, None, tri.ctypes.data_as(C.c_void_p)))
    lib.kf_mesh_free(h)
    ref = ko.mesh(vol, 0.0)
    assert same_bits(pos, ref[0]) and np.array_equal(tri, ref[3])
