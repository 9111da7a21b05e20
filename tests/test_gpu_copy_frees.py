"""Meshes extracted, copied and freed in two threads' turns: a freed mesh's
memory serves the next one of about its size, and no other's contents change."""
import threading

import pytest

from kf_helpers import copy_mesh, extract_mesh, noisy_pipeline, same_mesh

pytestmark = pytest.mark.gpu


def test_memory_of_freed_meshes_is_used_again(torch_gpu):
    import kinectfusion_amd as K
    from kinectfusion_amd import _native as N

    lib = N.hip()
    p = noisy_pipeline(K, 40)
    ref = copy_mesh(extract_mesh(p))[1]
    live, bad = [extract_mesh(p) for _ in range(3)], []

    def copy_and_free(mesh):  # in another thread than the context's
        status, out = copy_mesh(mesh)
        if status != 0 or not same_mesh(out, ref):
            bad.append(mesh)
        lib.kf_mesh_free(mesh[0])

    torch_gpu.cuda.synchronize()
    before = torch_gpu.cuda.mem_get_info()[0]
    for _ in range(12):
        t = threading.Thread(target=copy_and_free, args=(live.pop(0),))
        t.start()
        live.append(extract_mesh(p))
        t.join()
    torch_gpu.cuda.synchronize()
    grown = before - torch_gpu.cuda.mem_get_info()[0]
    for m in live:
        status, out = copy_mesh(m)
        assert status == 0 and same_mesh(out, ref)
        lib.kf_mesh_free(m[0])
    p.close()
    assert not bad and grown <= 32 << 20  # not twelve meshes' worth
