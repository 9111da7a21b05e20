"""One context's ring of pinned slots, wanted by three threads at once: two copy
meshes of the context and the third downloads its volume, so that some copies
find the ring taken and go the plain way.  Every byte is that of a copy alone."""
import ctypes as C
import threading

import numpy as np
import pytest

from kf_helpers import copy_mesh, extract_mesh, noisy_pipeline, same_mesh

pytestmark = pytest.mark.gpu


def test_three_threads_and_one_ring(torch_gpu):
    import kinectfusion_amd as K
    from kinectfusion_amd import _native as N

    lib = N.hip()
    p = noisy_pipeline(K, 96)
    meshes = [extract_mesh(p) for _ in range(2)]
    assert meshes[0][1] * 36 > 8 << 20  # longer than the ring
    ref = copy_mesh(meshes[0])[1]
    volume = np.zeros(96 ** 3 * 4, np.uint8)
    assert lib.kf_volume_download(p.ctx, volume.ctypes.data_as(C.c_void_p), None) == 0
    start, bad = threading.Barrier(3), []

    def copies(mesh):
        for _ in range(6):
            start.wait()
            status, out = copy_mesh(mesh)
            if status != 0 or not same_mesh(out, ref):
                bad.append("mesh")

    def downloads():
        for _ in range(6):
            start.wait()
            out = np.zeros_like(volume)
            if lib.kf_volume_download(p.ctx, out.ctypes.data_as(C.c_void_p), None) != 0 or not np.array_equal(out, volume):
                bad.append("volume")

    threads = [threading.Thread(target=copies, args=(m,)) for m in meshes] + [threading.Thread(target=downloads)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m in meshes:
        lib.kf_mesh_free(m[0])
    p.close()
    assert not bad, bad
