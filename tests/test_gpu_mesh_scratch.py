"""Device memory that a context keeps after an extraction."""
import pytest

from kf_helpers import extract_mesh, noisy_pipeline

pytestmark = pytest.mark.gpu


def test_kept_scratch_is_bounded_in_all(torch_gpu):
    """At 224^3 voxels of random signs the active cells and the vertices take
    some 200 MB of scratch each: together they stay within the 256 MB that a
    context keeps."""
    import kinectfusion_amd as K
    from kinectfusion_amd import _native as N

    torch, lib = torch_gpu, N.hip()
    p = noisy_pipeline(K, 224)
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        mesh = extract_mesh(p)
        assert mesh[1] * 12 > 150 << 20  # the vertices' share of the scratch
        lib.kf_mesh_free(mesh[0])
    kept = before - torch.cuda.mem_get_info()[0]
    p.close()
    assert kept <= (256 << 20) + (32 << 20), kept >> 20
