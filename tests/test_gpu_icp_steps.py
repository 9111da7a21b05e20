"""The correspondence sweep and the level's steps against the CPU oracle, over
map sizes that give a thread one, two or five pixels a pass (and several
passes), with a last pass and a last workgroup that are partly empty, holes in
the maps, and levels that latch early, late or not at all."""
import numpy as np
import pytest

from kf_helpers import f4, host, pipeline_config, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    import kinectfusion_amd

    return kinectfusion_amd


def surface(w, h, intr, seed):
    """Vertices and normals of a wavy surface seen from the identity, a tenth
    of them missing."""
    fx, fy, cx, cy = intr
    u, v = np.meshgrid(np.arange(w, dtype=np.float64), np.arange(h, dtype=np.float64))
    x, y = (u - cx) / fx, (v - cy) / fy
    z = 1.5 + 0.2 * np.sin(3 * x) * np.cos(4 * y) + 0.1 * x
    p = np.stack([x * z, y * z, z], -1)
    n = np.cross(np.gradient(p, axis=0) if h > 1 else np.zeros_like(p),
                 np.gradient(p, axis=1) if w > 1 else np.zeros_like(p))
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    hole = np.random.default_rng(seed).random((h, w)) < 0.1
    p[hole] = np.nan
    n[hole] = np.nan
    return p.astype(np.float32), n.astype(np.float32)


def moved(t, yaw):
    out = np.eye(4)
    c, s = np.cos(yaw), np.sin(yaw)
    out[:3, :3] = [[c, 0, s], [0, 1, 0], [-s, 0, c]]
    out[:3, 3] = t
    return out


@pytest.mark.parametrize("live,model", [((3, 2), (5, 4)), ((16, 16), (16, 16)), ((161, 119), (160, 120)),
                                        ((256, 256), (320, 240)), ((257, 256), (320, 240)), ((512, 256), (201, 303)),
                                        ((513, 257), (320, 240)), ((640, 513), (640, 480)), ((1283, 967), (640, 480))])
def test_sums_over_sizes(K, ko, torch_gpu, live, model):
    intr = lambda s: (0.8 * s[0], 0.8 * s[0], 0.5 * (s[0] - 1), 0.5 * (s[1] - 1))
    lv, ln = surface(*live, intr(live), 1)
    mv, mn = surface(*model, intr(model), 2)
    pose, inverse = moved([0.01, -0.005, 0.02], 0.01), np.eye(4)
    k = intr(model)
    s64, _, n_ref = ko.icp_sums(lv, ln, mv, mn, k, pose, inverse)
    p = K.Pipeline(pipeline_config(K, res=16))
    tracker = K.ProjectiveIcpTracker(p)
    sums, count = tracker.normal_equations(*(to_dev(torch_gpu, f4(a)) for a in (lv, ln, mv, mn)),
                                           K.CameraIntrinsics(*k), ko.pose12(pose), ko.pose12(inverse))
    assert count == n_ref
    assert np.abs(sums - s64).max() <= 1e-5 * max(np.abs(s64).max(), 1e-30)
    p.close()


@pytest.mark.parametrize("size", [(64, 48), (321, 239), (640, 480)])
@pytest.mark.parametrize("iterations", [1, 2, 12])
def test_level_over_sizes(K, ko, torch_gpu, size, iterations):
    k = (0.8 * size[0], 0.8 * size[0], 0.5 * (size[0] - 1), 0.5 * (size[1] - 1))
    lv, ln = surface(*size, k, 3)
    mv, mn = surface(*size, k, 4)
    start = moved([0.01, 0.004, -0.01], 0.006)
    ref, r = ko.icp_track_level(lv, ln, mv, mn, k, np.eye(4), start, iterations)
    p = K.Pipeline(pipeline_config(K, res=16))
    out = K.ProjectiveIcpTracker(p).estimate_pose(*(to_dev(torch_gpu, f4(a)) for a in (lv, ln, mv, mn)),
                                                  K.CameraIntrinsics(*k), np.eye(4), start, iterations)
    assert out.ok == (r.status in (0, 1))
    assert out.diagnostics.correspondences == r.correspondences
    assert np.abs(out.pose - ref).max() < 1e-6
    p.close()


def test_standalone_level_leaves_the_track_alone(K, scene_room, torch_gpu):
    k = (64.0, 64.0, 31.5, 23.5)
    maps = [to_dev(torch_gpu, f4(a)) for a in (*surface(64, 48, k, 5), *surface(64, 48, k, 6))]
    poses = []
    for between in (False, True):
        p = K.Pipeline(pipeline_config(K, res=64))
        for i in range(4):
            if between:  # one that converges, one that finds nothing
                t = K.ProjectiveIcpTracker(p)
                t.estimate_pose(*maps, K.CameraIntrinsics(*k), np.eye(4), np.eye(4), 3)
                assert not t.estimate_pose(*maps, K.CameraIntrinsics(*k), np.eye(4), moved([50, 0, 0], 0), 3).ok
            p.process_frame(to_dev(torch_gpu, scene_room.frame(i)[0]))
        poses.append(p.trajectory())
        p.close()
    assert np.array_equal(np.asarray(poses[0]), np.asarray(poses[1]))
