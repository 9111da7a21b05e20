"""The wave's 6 x 6 solve against the oracle's scalar LDL^T on chosen systems:
maps of small integers and dyadic offsets, whose 29 sums are exact in FP32, so
that both sides solve the same system bit for bit.  Among them equal diagonals,
diagonals that differ only below their upper 32 bits, zero pivots of systems of
every rank, and every damping mode.  The update's lengths are equal to the last
bit; the pose, which sin and cos enter, within 1e-12."""
import numpy as np
import pytest

from kf_helpers import f4, to_dev

pytestmark = pytest.mark.gpu

MODES = ("none", "identity", "diagonal")


def maps(normals, offsets):
    """Live points on integer pixels of the plane z = 1 and model points off
    them by multiples of 1/64: J = (p x n, n), residual n . offset."""
    h, w, _ = normals.shape
    v, u = np.mgrid[:h, :w]
    live = np.stack([u - w // 2, v - h // 2, np.ones_like(u)], -1).astype(np.float32)
    n = normals.astype(np.float32)
    intr = (1.0, 1.0, float(w // 2), float(h // 2))
    return live, n, live + (offsets / 64.0).astype(np.float32), n, intr


def uniform(h, w, n, rng):
    return np.broadcast_to(np.asarray(n), (h, w, 3)).copy(), rng.integers(-4, 5, (h, w, 3))


def systems():
    rng = np.random.default_rng(11)
    for n in ([0, 0, 1], [1, 0, 0], [0, -1, 0], [1, 1, 0], [0, 2, 1]):  # planes: rank 3, some with exact zero pivots
        yield uniform(5, 5, n, rng)
    for shape in ((1, 1), (1, 2), (2, 1), (1, 5), (2, 2)):  # rank 1 and up
        yield rng.choice([-2, -1, 1, 2], shape + (3,)), rng.integers(-4, 5, shape + (3,))
    cube = np.zeros((3, 6, 3), int)  # the axes' normals on symmetric points: equal diagonals
    cube[:, 0::3, 0] = cube[:, 1::3, 1] = cube[:, 2::3, 2] = 1
    yield cube, rng.integers(-4, 5, cube.shape)
    for extra in (0, 1, 2):  # 2^22 and 2^22 + extra: one upper half in FP64
        n = np.zeros((1, 5, 3), int)
        n[0, 0], n[0, 1], n[0, 2], n[0, 3] = [2048, 0, 0], [0, 2048, 0], [0, 1, 0], [0, 0, 1]
        n[0, 4] = [0, 1, 0] if extra == 2 else [0, 0, 1]
        if extra == 0:
            n[0, 2] = [0, 0, 1]
        yield n, np.concatenate([np.zeros((1, 3, 3), int), rng.integers(-2, 3, (1, 2, 3))], 1)
    for i in range(60):  # any
        shape = tuple(rng.integers(1, 8, 2))
        n = rng.integers(-2, 3, shape + (3,))
        n[(n == 0).all(-1)] = [0, 0, 1]
        if i % 3 == 0:
            n[..., int(rng.integers(0, 3))] = 0
            n[(n == 0).all(-1)] = [1, 1, 1]
        yield n, rng.integers(-8, 9, shape + (3,))


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_solve_of_chosen_systems(ko, torch_gpu, mode):
    import kinectfusion_amd as K
    from kf_helpers import pipeline_config

    p = K.Pipeline(pipeline_config(K, res=16))
    wide = dict(min_correspondences=1, max_point_distance=1.0, max_update_translation=1e3, max_update_rotation=1e3)
    ref_opt = ko.icp_options(damping_mode=mode, **wide)
    tracker = K.ProjectiveIcpTracker(p, K.ProjectiveIcpOptions(damping=MODES[mode], **wide))
    singular = solved = 0
    for normals, offsets in systems():
        lv, ln, mv, mn, intr = maps(normals, offsets)
        s64, _, count = ko.icp_sums(lv, ln, mv, mn, intr, np.eye(4), np.eye(4), 1.0)
        assert count == normals.shape[0] * normals.shape[1]
        assert np.array_equal(s64[:27], s64[:27].astype(np.float32).astype(np.float64))  # exact in FP32
        a = np.zeros((6, 6))
        a[np.triu_indices(6)] = s64[:21]
        singular += bool(np.linalg.matrix_rank(a + np.triu(a, 1).T) < 6)
        ref, r = ko.icp_track_level(lv, ln, mv, mn, intr, np.eye(4), np.eye(4), 1, ref_opt)
        out = tracker.estimate_pose(*(to_dev(torch_gpu, f4(m)) for m in (lv, ln, mv, mn)), K.CameraIntrinsics(*intr),
                                    np.eye(4), np.eye(4), 1)
        d = out.diagnostics
        key = (normals.tolist(), offsets.tolist())
        assert d.correspondences == r.correspondences and d.status == r.status, (key, d.status, r.status)
        assert (d.update_translation, d.update_rotation) == (r.update_translation, r.update_rotation), key
        assert np.abs(out.pose - ref).max() <= 1e-12, key
        solved += r.status in (0, 1)
    assert singular >= 10 and solved >= (30 if mode == 0 else 60)
    p.close()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("where", [0, 1, 2])
def test_a_system_that_is_not_finite_moves_nothing(ko, torch_gpu, mode, where):
    """A normal of 1e20 squares past FP32's range: infinite sums, and NaN in
    the factors, whichever pivot it lies on."""
    import kinectfusion_amd as K
    from kf_helpers import pipeline_config

    normals = np.random.default_rng(where).integers(1, 3, (4, 4, 3)).astype(np.float64)
    lv, ln, mv, mn, intr = maps(normals, np.ones((4, 4, 3)))
    mn = mn.copy()
    mn[1, 2] = 0
    mn[1, 2, where] = 1e20
    start = np.eye(4)
    start[:3, 3] = [0.0, 0.0, 1.0 / 64]
    p = K.Pipeline(pipeline_config(K, res=16))
    tracker = K.ProjectiveIcpTracker(p, K.ProjectiveIcpOptions(
        damping=MODES[mode], min_correspondences=1, max_point_distance=1.0, min_normal_dot=-1e30))
    out = tracker.estimate_pose(*(to_dev(torch_gpu, f4(m)) for m in (lv, ln, mv, mn)), K.CameraIntrinsics(*intr),
                                np.eye(4), start, 2)
    assert not out.ok and out.diagnostics.status in ((3, 5) if mode == 0 else (3,))
    assert np.array_equal(out.pose, start)
    p.close()
