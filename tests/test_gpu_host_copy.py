"""Copies from the device into the caller's memory, byte for byte: sizes around
the bar below which a copy goes the plain way, whole and partial slots, enough
of them for the second thread and to go round the ring, destinations that are
pageable, off alignment and pinned, and two threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import kinectfusion_amd

    return kinectfusion_amd


def destinations(torch, n):
    """n bytes each: pageable, off any alignment, pinned (as uint8 arrays)."""
    yield np.zeros(n, np.uint8)
    yield np.zeros(n + 64, np.uint8)[13:13 + n]
    yield torch.zeros(n, dtype=torch.uint8).pin_memory().numpy()


def random_pipeline(K, res, store):
    p = K.Pipeline(K.PipelineConfig(voxel=store, color="float", volume=K.VolumeGeometry(res, 0.01, (0, 0, 0), 0.05)))
    n = int(np.prod(res))
    rng = np.random.default_rng(n)
    width = 2 if store == "float" else 1
    vox = rng.integers(0, 1 << 30, (n, width), dtype=np.uint32)  # finite floats and any 16-bit pairs
    vox = vox.view(np.float32) if store == "float" else vox.view(np.uint16).reshape(n, 2)
    col = rng.random((n, 4), np.float32)
    p.upload_volume(vox, col)
    return p, vox, col


@pytest.mark.parametrize("store", ["float", "bf16"])
@pytest.mark.parametrize("res", [(31, 32, 32), (32, 32, 32), (64, 64, 64), (65, 63, 67), (128, 128, 80),
                                 (131, 127, 129)])
def test_volume_comes_back(K, torch_gpu, store, res):
    from kinectfusion_amd import _native as N

    p, vox, col = random_pipeline(K, res, store)
    for v, c in zip(destinations(torch_gpu, vox.nbytes), destinations(torch_gpu, col.nbytes)):
        N.check(N.hip().kf_volume_download(p.ctx, v.ctypes.data_as(C.c_void_p), c.ctypes.data_as(C.c_void_p)))
        assert np.array_equal(v, vox.reshape(-1).view(np.uint8)) and np.array_equal(c, col.reshape(-1).view(np.uint8))
    p.close()


def test_two_threads_at_once(K, torch_gpu):
    pipes = [random_pipeline(K, (128, 96, 100 + i), "float") for i in range(2)]
    got, lib = [[], []], pytest.importorskip("kinectfusion_amd._native").hip()

    def work(i):
        p, vox, _ = pipes[i]
        for _ in range(4):
            out = np.zeros(vox.nbytes, np.uint8)
            status = lib.kf_volume_download(p.ctx, out.ctypes.data_as(C.c_void_p), None)
            got[i].append(status == 0 and np.array_equal(out, vox.reshape(-1).view(np.uint8)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == [[True] * 4] * 2
    for p, _, _ in pipes:
        p.close()
