"""kf_mesh_copy and kf_mesh_free beside other work of the program: neither
waits for another stream's, and both work while the program captures a graph,
which is unharmed."""
import pytest

from kf_helpers import copy_mesh, extract_mesh, noisy_pipeline, same_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import kinectfusion_amd

    return kinectfusion_amd


@pytest.fixture(scope="module")
def lib():
    from kinectfusion_amd import _native as N

    return N.hip()


def sleep_for(torch, seconds):
    """Occupies the current stream for about that long; the event at its end."""
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    a.record()
    torch.cuda._sleep(1_000_000)
    b.record()
    b.synchronize()
    torch.cuda._sleep(int(1_000_000 * seconds * 1e3 / a.elapsed_time(b)))
    end = torch.cuda.Event()
    end.record()
    return end


@pytest.mark.parametrize("res", [20, 96])  # shorter and longer than the ring
def test_copy_and_free_wait_for_no_other_work(K, torch_gpu, lib, res):
    """Beside a kernel on the default stream, from several contexts: the
    runtime maps streams onto four hardware queues, and one that shares the
    kernel's has to wait there."""
    pipes = [noisy_pipeline(K, res) for _ in range(4)]
    ref = copy_mesh(extract_mesh(pipes[0]))[1]
    waited = []
    for p in pipes:
        mesh = extract_mesh(p)
        end = sleep_for(torch_gpu, 0.4)
        status, out = copy_mesh(mesh)
        in_copy = end.query()
        lib.kf_mesh_free(mesh[0])
        waited.append((in_copy, end.query()))
        end.synchronize()
        assert status == 0 and same_mesh(out, ref)
    for p in pipes:
        p.close()
    assert (False, False) in waited and (False, True) not in waited, waited


@pytest.mark.parametrize("res", [20, 96])
def test_copy_and_free_during_a_capture(K, torch_gpu, lib, res):
    torch = torch_gpu
    p = noisy_pipeline(K, res)
    ref = copy_mesh(extract_mesh(p))[1]
    p2 = noisy_pipeline(K, res)  # whose first long copy this is
    mesh = extract_mesh(p2)
    x = torch.ones(1000, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        x.mul_(2.0)
        status, out = copy_mesh(mesh)
        lib.kf_mesh_free(mesh[0])
        x.add_(1.0)
    assert status == 0 and same_mesh(out, ref)
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert bool((x == 2.0 ** (i + 2) - 1).all())
        again = extract_mesh(p2)  # the freed mesh's memory may be in use again
        assert same_mesh(copy_mesh(again)[1], ref)
        lib.kf_mesh_free(again[0])
    p.close()
    p2.close()
