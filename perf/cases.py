"""The measured workloads: what a program built on this package has it do, one
dict of plain values per case, each run through the package's entry points.

  listed()            the fixed cases
  draw(rng)           one more case from the same ranges
  prepare(case, seed) what the program holds before the call, on the GPU
  run(state)          one pass; returns its outputs
  work(case)          bytes and operations a pass cannot do without
  exact(case, seed)   the computed outputs in 64 bits, where they have such a value

Scenes are the seeded synthetic rooms and halls of the package (uint16
millimetre depth with noise and dropouts, RGBA8 colour); the seed picks the
scene.  Stage sizes are those of the benchmark and the tests: 640 x 480
frames, 3 pyramid levels, a 512^3 volume of 5 mm voxels over the room, a
2048^3 hashed volume of 5 mm voxels over the hall.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import kinectfusion_amd as K
from kinectfusion_amd import _native as N
from kinectfusion_amd import posenet as PN

SCALE = 1000.0        # raw depth units per metre
MIN_DEPTH, MAX_DEPTH = 0.4, 8.0
TRUNC = 0.05
SIGMA_S, SIGMA_R = 4.5, 0.03
JUMP = 0.1            # the pyramid's depth-jump limits (m)
MAX_DIST, MIN_DOT = 0.05, 0.9659258
BURST = 8             # frames a reconstruction enqueues before it looks at the result
WARM = 16             # frames the pipeline has already seen
SEQUENCE = 24         # resident frames, played back and forth


# ---- the cases -----------------------------------------------------------------------------------
def listed():
    return [
        # one correspondence sweep of the coarsest pyramid level: the smallest call, all latency
        {"name": "sums-160x120", "kind": "sums", "width": 160, "height": 120},
        # the depth pyramid of one camera frame (bilateral r = 3, 3 levels of vertices and normals)
        {"name": "pyramid-640x480", "kind": "pyramid", "width": 640, "height": 480, "radius": 3},
        # aligning one full-resolution frame to another: a finest-level tracking call of 10 iterations
        {"name": "icp-640x480", "kind": "icp", "width": 640, "height": 480, "iterations": 10},
        # fusing a frame with a known pose into a volume of odd extents (float voxels, classic rule, no colour)
        {"name": "integrate-ragged-float", "kind": "integrate", "nx": 251, "ny": 203, "nz": 270, "store": "float",
         "color": "none", "rule": "classic", "width": 640, "height": 480},
        # the same into the benchmark's volume (bf16 voxels, angle-weighted rule, colour)
        {"name": "integrate-512-bf16", "kind": "integrate", "nx": 512, "ny": 512, "nz": 512, "store": "bf16",
         "color": "float", "rule": "angle-weighted", "width": 640, "height": 480},
        # rendering the model from a viewpoint
        {"name": "raycast-512-bf16", "kind": "raycast", "nx": 512, "ny": 512, "nz": 512, "store": "bf16",
         "color": "float", "width": 640, "height": 480, "level": 0},
        # whole frames of the benchmark's three pipelines: a burst of frames, the last one's report, and the
        # model rendered from it; learned warm start with bf16 voxels ...
        {"name": "frames-512-bf16-learned", "kind": "frames", "scene": "room", "res": 512, "store": "bf16",
         "color": "float", "init": "learned", "width": 640, "height": 480},
        # ... the plain FP32 method ...
        {"name": "frames-512-float", "kind": "frames", "scene": "room", "res": 512, "store": "float",
         "color": "float", "init": "previous", "width": 640, "height": 480},
        # ... and the sparse hashed volume of the large hall
        {"name": "frames-2048-hashed", "kind": "frames", "scene": "hall", "res": 2048, "store": "float",
         "color": "none", "init": "previous", "width": 640, "height": 480},
        # the end of a reconstruction: the mesh of a dense and of a hashed volume, on the host
        {"name": "mesh-512-bf16", "kind": "mesh", "scene": "room", "res": 512, "store": "bf16", "color": "float"},
        {"name": "mesh-2048-hashed", "kind": "mesh", "scene": "hall", "res": 2048, "store": "float", "color": "none"},
        # training the pose network: loss and gradients of a batch
        {"name": "posenet-gradients-64", "kind": "posenet", "mode": "gradients", "batch": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sums", "pyramid", "icp", "integrate", "raycast", "frames", "mesh", "posenet"])
    store = rng.choice(["float", "quantized", "bf16"])
    color = rng.choice(["float", "none"])
    if kind in ("sums", "icp"):
        w = _log(rng, 80, 640)
        c = {"kind": kind, "width": w, "height": int(w * rng.uniform(0.6, 0.75))}
        return dict(c, iterations=rng.randint(4, 10)) if kind == "icp" else c
    if kind == "pyramid":
        w = _log(rng, 160, 1280)
        return {"kind": kind, "width": w, "height": int(w * rng.uniform(0.6, 0.75)), "radius": rng.randint(2, 5)}
    if kind in ("integrate", "raycast"):
        w = _log(rng, 200, 640)
        c = {"kind": kind, "nx": _log(rng, 64, 512), "ny": _log(rng, 64, 512), "nz": _log(rng, 64, 512),
             "store": store, "color": color, "width": w, "height": int(w * 0.75)}
        if kind == "raycast":
            return dict(c, level=rng.randint(0, 2))
        return dict(c, rule=rng.choice(["classic", "angle-weighted"]))
    if kind == "frames":
        if rng.random() < 0.3:
            return {"kind": kind, "scene": "hall", "res": 8 * rng.randint(128, 256), "store": store, "color": "none",
                    "init": "previous", "width": 640, "height": 480}
        init = rng.choice(["learned", "previous", "constant-velocity"])
        w = 640 if init == "learned" else rng.randint(400, 640)
        return {"kind": kind, "scene": "room", "res": _log(rng, 128, 512), "store": store, "color": color,
                "init": init, "width": w, "height": 480 if w == 640 else int(w * 0.75)}
    if kind == "mesh":
        scene = rng.choice(["room", "room", "hall"])
        res = _log(rng, 64, 512) if scene == "room" else 8 * rng.randint(128, 256)
        return {"kind": kind, "scene": scene, "res": res, "store": store,
                "color": color if scene == "room" else "none"}
    return {"kind": kind, "mode": rng.choice(["forward", "gradients"]), "batch": rng.randint(1, 64)}


# ---- inputs --------------------------------------------------------------------------------------
def _camera(w, h):
    """The 640 x 480 camera scaled to w x h."""
    return K.CameraIntrinsics(525.0 * w / 640.0, 525.0 * w / 640.0, 0.5 * (w - 1), 0.5 * (h - 1))


def _scene(kind, seed, w, h):
    k = _camera(w, h)
    return K.SyntheticScene(kind, seed=seed % (1 << 31), width=w, height=h, fx=k.fx, fy=k.fy, cx=k.cx, cy=k.cy)


def _frames(scene, first, count, color):
    """Resident frames (depth, colour or None, camera_to_world) of the scene's trajectory."""
    poses = [scene.pose(first + i) for i in range(count)]
    if color:
        host = [scene.frame(first + i) for i in range(count)]
        return [(torch.from_numpy(d.view(np.int16)).cuda(), torch.from_numpy(c.view(np.int32)).cuda(), p)
                for (d, c, _), p in zip(host, poses)]
    depth = scene.render_device(np.stack(poses), np.arange(first, first + count))
    return [(depth[i], None, p) for i, p in enumerate(poses)]


def _config(w, h, n, voxel, store="float", color="none", rule="angle-weighted", radius=3, **kw):
    """A pipeline over n = (nx, ny, nz) voxels, centred in x and y on the first camera, 0.5 m behind it."""
    trunc = max(TRUNC, 3.0 * voxel)
    origin = (-0.5 * n[0] * voxel, -0.5 * n[1] * voxel, -0.5)
    hashed = kw.get("storage") == "hashed"
    return K.PipelineConfig(
        voxel=store, color=color, tsdf_rule=rule, volume=K.VolumeGeometry(tuple(n), voxel, origin, trunc),
        integration=K.TsdfIntegrationOptions(depth_scale=SCALE, mode="band" if hashed else "full"),
        depth=K.DepthProcessingOptions(levels=3, bilateral_radius=radius, bilateral_spatial_sigma=SIGMA_S,
                                       bilateral_depth_sigma=SIGMA_R),
        intrinsics=_camera(w, h), width=w, height=h, icp_iterations=(10, 5, 4), **kw)


def _scene_config(case, w, h):
    """The pipeline of a scene case: a dense volume over the room, a hashed one over the hall."""
    res = case["res"]
    kw = {"store": case["store"], "color": case["color"], "init": case.get("init", "previous")}
    if case["scene"] == "hall":
        return _config(w, h, (res, res, res), 10.24 / res, storage="hashed", hash_buckets=1 << 20,
                       block_capacity=500_000, **kw)
    if kw["init"] == "learned":
        kw["learned_iterations"] = (2, 0, 0)
    return _config(w, h, (res, res, res), 2.56 / res, **kw)


def _volume_config(case):
    n = (case["nx"], case["ny"], case["nz"])
    return _config(case["width"], case["height"], n, 2.56 / max(n), store=case["store"], color=case["color"],
                   rule=case.get("rule", "angle-weighted"))


class _Array:
    """Library device memory as torch takes it.  The tensor's storage holds this object, and so the pipeline whose
    buffer it is: the buffer lives as long as any view of it."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2, "strides": None}


def _view(p, ptr, shape, typestr):
    """A tensor over device memory that the pipeline p owns."""
    return torch.as_tensor(_Array(p, ptr, shape, typestr), device="cuda")


def _volume(p):
    """The dense volume's own device buffers as tensors (kf_volume_device)."""
    vox, col = C.c_void_p(), C.c_void_p()
    N.check(N.hip().kf_volume_device(p.ctx, C.byref(vox), C.byref(col)), p.ctx)
    n = int(np.prod(p.config.volume.resolution))
    out = {"voxels": _view(p, vox.value, (n, 2), "<f4") if p.config.voxel == "float" else _view(p, vox.value, (n,), "<i4")}
    if col.value:
        out["colors"] = _view(p, col.value, (n, 4), "<f4")
    return out


def _pair_maps(case, seed):
    """Vertices and normals of two neighbouring frames, their camera and the true motion between them."""
    w, h = case["width"], case["height"]
    p = K.Pipeline(_config(w, h, (16, 16, 16), 0.01))
    src = K.PyramidSource(p)
    maps = []
    for depth, _, pose in _frames(_scene("room", seed, w, h), 10, 2, False):
        src.build(depth)
        lv = src.level(0)
        maps.append((lv["vertices"], lv["normals"], pose))
    return p, maps


def _integration_frames(case, seed):
    """Frames with their normals, as a tracked pipeline fuses them."""
    w, h = case["width"], case["height"]
    frames = _frames(_scene("room", seed, w, h), 0, 6, case["color"] == "float")
    q = K.Pipeline(_config(w, h, (16, 16, 16), 0.01))
    src = K.PyramidSource(q)
    out = []
    for depth, color, pose in frames:
        src.build(depth)
        out.append((depth, color, src.level(0)["normals"], np.linalg.inv(pose)))
    q.close()
    return out


def _pairs(case, seed):
    """Depth pairs at the network's input size and the twists between their cameras."""
    b = case["batch"]
    rng = np.random.default_rng(seed)
    base = [PN.random_view(rng) for _ in range(b)]
    motion = [PN.random_motion(rng, 0.05, 5.0) for _ in range(b)]
    frames = _scene("room", seed, 160, 120).render_device(np.stack(base + [p @ m for p, m in zip(base, motion)]),
                                                           rng.integers(0, 2**62, size=2 * b, dtype=np.uint64))
    pairs = torch.stack([frames[:b], frames[b:]], dim=1).contiguous()
    targets = torch.from_numpy(np.stack([PN.pose_to_twist(m) for m in motion]).astype(np.float32)).cuda()
    return pairs, targets


def _still_network(seed):
    """A pose network whose output layer is zero: it proposes no motion.  Frame to frame the camera moves little,
    so its proposals are kept as a trained network's are, without a training run for each state."""
    net = PN.PoseNet(PN.PoseNetConfig(batch_capacity=1, seed=seed % (1 << 31)))
    w = net.parameters()
    w[-(256 * 6 + 6):] = 0.0
    net.set_parameters(w)
    return net


def _mesh_capacity(case):
    """Vertices and triangles that the program's buffers hold: the scene's visible surface at this voxel size, with
    room to spare."""
    voxel = (10.24 if case["scene"] == "hall" else 2.56) / case["res"]
    v = int((60.0 if case["scene"] == "hall" else 20.0) / voxel**2) + 20_000
    return v, 2 * v


class _State:
    def __init__(self, case, **kw):
        self.case = case
        self.at = 0
        self.__dict__.update(kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("sums", "icp"):
        p, (model, live) = _pair_maps(case, seed)
        return _State(case, p=p, tracker=K.ProjectiveIcpTracker(p), live=live, model=model,
                      k=_camera(case["width"], case["height"]))
    if kind == "pyramid":
        w, h = case["width"], case["height"]
        p = K.Pipeline(_config(w, h, (16, 16, 16), 0.01, radius=case["radius"]))
        return _State(case, p=p, src=K.PyramidSource(p), frames=_frames(_scene("room", seed, w, h), 0, 6, False),
                      views={})
    if kind in ("integrate", "raycast"):
        p = K.Pipeline(_volume_config(case))
        frames = _integration_frames(case, seed)
        for depth, color, normals, w2c in frames:
            p.integrate(depth, w2c, color=color, normals=normals)
        p.synchronize()
        if kind == "integrate":
            return _State(case, p=p, frames=frames, outputs=_volume(p))
        scene = _scene("room", seed, case["width"], case["height"])
        return _State(case, p=p, poses=[scene.pose(6 + i) for i in range(6)])
    if kind == "frames":
        w, h = case["width"], case["height"]
        p = K.Pipeline(_scene_config(case, w, h))
        net = None
        if case["init"] == "learned":
            net = _still_network(seed)
            p.attach_posenet(net)
        frames = _frames(_scene(case["scene"], seed, w, h), 0, SEQUENCE, case["color"] == "float")
        for depth, color, _ in frames[:WARM]:
            p.process_frame(depth, color, report=False)
        p.synchronize()
        return _State(case, p=p, net=net, frames=frames, at=WARM,
                      volume=_volume(p) if case["scene"] == "room" else {})
    if kind == "mesh":
        w, h = 640, 480
        p = K.Pipeline(_scene_config(case, w, h))
        scene = _scene(case["scene"], seed, w, h)
        for depth, color, pose in _frames(scene, 0, SEQUENCE, case["color"] == "float"):
            p.integrate(depth, np.linalg.inv(pose), color=color)
        p.synchronize()
        v, t = _mesh_capacity(case)
        out = {"positions": np.zeros((v, 3), np.float32), "normals": np.zeros((v, 3), np.float32),
               "colors": np.zeros((v, 3), np.float32), "triangles": np.zeros((t, 3), np.int32)}
        return _State(case, p=p, out=out)
    pairs, targets = _pairs(case, seed)
    return _State(case, net=PN.PoseNet(PN.PoseNetConfig(batch_capacity=64, seed=seed % (1 << 31))), pairs=pairs,
                  targets=targets)


# ---- one pass ------------------------------------------------------------------------------------
def _level_views(s):
    """The pyramid's device views (kf_pyramid_level), as tensors."""
    out = {}
    for level in range(3):
        lv = N.KfLevelView()
        N.check(N.hip().kf_pyramid_level(s.p.ctx, level, C.byref(lv)), s.p.ctx)
        key = (level, lv.depth, lv.vertices, lv.normals)
        if key not in s.views:
            n = (lv.height, lv.width)
            s.views[key] = {"depth": _view(s.p, lv.depth, n, "<i2"), "vertices": _view(s.p, lv.vertices, n + (4,), "<f4"),
                            "normals": _view(s.p, lv.normals, n + (4,), "<f4")}
        out["level%d" % level] = s.views[key]
    return out


def _maps(m):
    return {"points": m.points, "normals": m.normals, "colors": m.colors}


def _mesh_into(p, out):
    """The mesh copied into the program's own host buffers (kf_mesh_extract, kf_mesh_size, kf_mesh_copy)."""
    lib, h, nv, nt = N.hip(), C.c_void_p(), C.c_int64(), C.c_int64()
    N.check(lib.kf_mesh_extract(p.ctx, 0.0, C.byref(h)), p.ctx)
    try:
        N.check(lib.kf_mesh_size(h, C.byref(nv), C.byref(nt)), p.ctx)
        if nv.value > len(out["positions"]) or nt.value > len(out["triangles"]):
            raise RuntimeError("the mesh (%d vertices, %d triangles) exceeds the buffers" % (nv.value, nt.value))
        N.check(lib.kf_mesh_copy(h, *(out[k].ctypes.data_as(C.c_void_p) for k in
                                      ("positions", "normals", "colors", "triangles"))), p.ctx)
    finally:
        lib.kf_mesh_free(h)
    return dict(out, vertex_count=nv.value, triangle_count=nt.value)


def _to12(pose):
    return np.asarray(pose, np.float64)[:3].reshape(12)


def run(s):
    kind = s.case["kind"]
    if kind == "sums":
        sums, count = s.tracker.normal_equations(s.live[0], s.live[1], s.model[0], s.model[1], s.k,
                                                 _to12(np.eye(4)), _to12(np.eye(4)))
        return {"sums": sums, "count": count}
    if kind == "icp":
        out = s.tracker.estimate_pose(s.live[0], s.live[1], s.model[0], s.model[1], s.k, np.eye(4), np.eye(4),
                                      s.case["iterations"])
        r = out.diagnostics
        return {"pose": out.pose, "status": r.status, "trials": r.trials, "correspondences": r.correspondences,
                "mean_distance": r.mean_distance, "mean_squared_residual": r.mean_squared_residual}
    if kind == "pyramid":
        s.src.build(s.frames[s.at % len(s.frames)][0])
        s.at += 1
        return _level_views(s)
    if kind == "integrate":
        depth, color, normals, w2c = s.frames[s.at % len(s.frames)]
        s.at += 1
        s.p.integrate(depth, w2c, color=color, normals=normals)
        return s.outputs
    if kind == "raycast":
        s.at += 1
        return _maps(s.p.raycast(s.poses[s.at % len(s.poses)], s.case["level"]))
    if kind == "frames":
        for i in range(BURST):
            turn = 2 * SEQUENCE - 2  # 0, 1, ..., 23, 22, ..., 1, 0, 1, ...
            at = s.at % turn
            depth, color, _ = s.frames[at if at < SEQUENCE else turn - at]
            s.at += 1
            res = s.p.process_frame(depth, color, report=i + 1 == BURST, sync_inputs=False)
        pose = np.array(res.pose[:], np.float64).reshape(4, 4)
        return {"tracked": res.tracked, "used_learned": res.used_learned, "pose": pose.astype(np.float32),
                "model": _maps(s.p.raycast(pose, 0)), **s.volume}
    if kind == "mesh":
        return _mesh_into(s.p, s.out)
    if s.case["mode"] == "forward":
        return {"twists": s.net.forward(s.pairs)}
    loss, grads = s.net.gradients(s.pairs, s.targets)
    return {"loss": loss, "gradients": grads}


# ---- what a pass cannot do without ---------------------------------------------------------------
def _voxels(case, w, h, voxel, depth):
    """Voxels a frame updates: those from the camera to the surface at `depth` m plus the truncation, inside the
    view of w x h pixels."""
    f = 525.0 * w / 640.0
    return w * h / (f * f) * (depth + TRUNC) ** 3 / 3.0 / voxel**3


def _band_voxels(w, h, voxel, depth):
    """Voxels of the truncation band around the surface at `depth` m."""
    f = 525.0 * w / 640.0
    return w * h / (f * f) * depth**2 * 2.0 * TRUNC / voxel**3


def _integration_bytes(case, w, h, voxel):
    """Depth, colour and normals read once; every updated voxel and colour voxel read and written once."""
    sv = 8 if case["store"] == "float" else 4
    hall = case.get("scene") == "hall"
    updated = _band_voxels(w, h, voxel, 2.5) if hall else _voxels(case, w, h, voxel, 1.2)
    b = w * h * 2 + updated * 2 * sv
    if case["color"] == "float":
        b += w * h * 4 + 0.75 * _band_voxels(w, h, voxel, 1.2) * 32
    return b


def _render_bytes(case, w, h):
    """Each ray's surface cell and its gradient's neighbours (32 voxels), its colour cell, and the maps written."""
    sv = 8 if case["store"] == "float" else 4
    return w * h * (36 + 32 * sv + (8 * 16 if case["color"] == "float" else 0))


def work(case):
    kind = case["kind"]
    if kind in ("sums", "icp"):
        n = case["width"] * case["height"]
        sweeps = case.get("iterations", 1)
        # four maps of three floats read once (they stay in cache between iterations); 27 products and sums a pixel
        return {"bytes": 48 * n, "flops": 150 * n * sweeps}
    if kind == "pyramid":
        n, taps = case["width"] * case["height"], (2 * case["radius"] + 1) ** 2
        return {"bytes": n * 2 + 1.3125 * n * (2 + 24), "flops": n * taps * 20}
    if kind == "integrate":
        voxel = 2.56 / max(case["nx"], case["ny"], case["nz"])
        b = _integration_bytes(case, case["width"], case["height"], voxel)
        share = case["nx"] * case["ny"] * case["nz"] / max(case["nx"], case["ny"], case["nz"]) ** 3
        return {"bytes": case["width"] * case["height"] * 2 + share * b, "flops": share * b / 8 * 40}
    if kind == "raycast":
        w, h = case["width"] >> case["level"], case["height"] >> case["level"]
        return {"bytes": _render_bytes(case, w, h), "flops": w * h * 15 * 60}
    if kind == "frames":
        w, h = case["width"], case["height"]
        voxel = (10.24 if case["scene"] == "hall" else 2.56) / case["res"]
        integrate, render = _integration_bytes(case, w, h, voxel), _render_bytes(case, w, h)
        levels = 1.0 if case["init"] == "learned" else 1.3125
        sweeps = 2 if case["init"] == "learned" else 10 + 5 / 4 + 4 / 16
        flops = integrate / 8 * 40 + w * h * (levels * 15 * 60 + 150 * sweeps + 49 * 20)
        return {"bytes": BURST * (integrate + levels * render) + render, "flops": BURST * flops}
    if kind == "mesh":
        voxel = (10.24 if case["scene"] == "hall" else 2.56) / case["res"]
        sv = 8 if case["store"] == "float" else 4
        # every stored voxel read once; about one vertex per surface voxel face crossed, two triangles a vertex
        area = 20.0 if case["scene"] == "hall" else 5.0
        vertices = 1.5 * area / voxel**2
        stored = case["res"] ** 3 if case["scene"] == "room" else 4.0 * area * TRUNC / voxel**3
        return {"bytes": stored * sv + vertices * (36 + 24), "flops": stored + vertices * 500}
    passes = 1 if case["mode"] == "forward" else 3
    return {"bytes": case["batch"] * 2 * 160 * 120 * 2 + 793_000 * (2 if passes == 1 else 6),
            "flops": passes * case["batch"] * 35e6}


# ---- the same outputs in 64 bits -----------------------------------------------------------------
def exact(case, seed):
    """Plain torch and numpy in 64 bits on the same inputs.  Rays and whole frames have no such value: which samples
    a ray takes, and so whether it meets a surface, is decided by the rounding of every step before.  Mesh vertices
    come in the order of the traversal, with fused attributes of the rendered volume: they are compared bit by bit."""
    kind = case["kind"]
    if kind in ("sums", "icp"):
        return _exact_icp(case, seed)
    if kind == "pyramid":
        return _exact_pyramid(case, seed)
    if kind == "integrate":
        return _exact_integrate(case, seed)
    if kind == "posenet":
        return _exact_posenet(case, seed)
    return None


def _exact_sweep(live_v, live_n, model_v, model_n, k, pose, model_inv):
    """J^T J, J^T r, the distance sum, the residual's square sum and the count of one correspondence sweep."""
    h, w = model_v.shape[:2]
    lv, ln = live_v.reshape(-1, 3), live_n.reshape(-1, 3)
    ok = torch.isfinite(lv).all(1) & torch.isfinite(ln).all(1)
    lv, ln = lv[ok], ln[ok]
    src = lv @ pose[:3, :3].T + pose[:3, 3]
    sim = src @ model_inv[:3, :3].T + model_inv[:3, 3]
    front = sim[:, 2] > 0
    src, ln, sim = src[front], ln[front], sim[front]
    u = torch.floor(k.fx * sim[:, 0] / sim[:, 2] + k.cx + 0.5)
    v = torch.floor(k.fy * sim[:, 1] / sim[:, 2] + k.cy + 0.5)
    ok = (u >= 0) & (u < w) & (v >= 0) & (v < h)
    src, ln = src[ok], ln[ok]
    at = (v[ok] * w + u[ok]).long()
    mv, mn = model_v.reshape(-1, 3)[at], model_n.reshape(-1, 3)[at]
    sn = ln @ pose[:3, :3].T
    sn = sn / sn.norm(dim=1, keepdim=True)
    dist = (src - mv).norm(dim=1)
    ok = torch.isfinite(mv).all(1) & torch.isfinite(mn).all(1) & (dist <= MAX_DIST) & ((sn * mn).sum(1) >= MIN_DOT)
    src, mv, mn, dist = src[ok], mv[ok], mn[ok], dist[ok]
    J = torch.cat([torch.linalg.cross(src, mn), mn], dim=1)
    r = (mn * (mv - src)).sum(1)
    A = (J.T @ J).cpu().numpy()
    return A, (J.T @ r).cpu().numpy(), float(dist.sum()), float((r * r).sum()), int(ok.sum())


def _exact_icp(case, seed):
    p, (model, live) = _pair_maps(case, seed)
    p.close()
    maps = [m[..., :3].double() for m in (live[0], live[1], model[0], model[1])]
    k = _camera(case["width"], case["height"])
    eye = torch.eye(4, dtype=torch.float64, device="cuda")
    if case["kind"] == "sums":
        A, b, dist, res2, count = _exact_sweep(*maps, k, eye, eye)
        return {"sums": np.concatenate([A[np.triu_indices(6)], b, [dist, res2]]), "count": None}
    pose = np.eye(4)
    for _ in range(case["iterations"]):
        A, b, dist, res2, count = _exact_sweep(*maps, k, torch.from_numpy(pose).cuda(), eye)
        x = np.linalg.solve(A, b)
        inc = np.eye(4)
        inc[:3, :3] = PN.rotation_from_vector(x[:3])
        inc[:3, 3] = x[3:]
        pose = inc @ pose
        if np.linalg.norm(x[3:]) < 1e-5 and np.linalg.norm(x[:3]) < 1e-5:
            break
    return {"pose": pose, "status": None, "trials": None, "correspondences": None, "mean_distance": dist / count,
            "mean_squared_residual": res2 / count}


def _shift(t, dy, dx, fill):
    """t[y + dy, x + dx], `fill` outside."""
    h, w = t.shape[:2]
    out = torch.full_like(t, fill)
    y0, y1, x0, x1 = max(0, -dy), min(h, h - dy), max(0, -dx), min(w, w - dx)
    out[y0:y1, x0:x1] = t[y0 + dy:y1 + dy, x0 + dx:x1 + dx]
    return out


def _exact_pyramid(case, seed):
    w, h, radius = case["width"], case["height"], case["radius"]
    raw = _frames(_scene("room", seed, w, h), 0, 6, False)[0][0].to(torch.int64) & 0xFFFF
    m = raw.double() / SCALE
    usable = (raw != 0) & (m >= MIN_DEPTH) & (m <= MAX_DEPTH)
    vals, wsum = torch.zeros_like(m), torch.zeros_like(m)
    for dy in range(-radius, radius + 1):
        for dx in range(-radius, radius + 1):
            mm, use = _shift(m, dy, dx, 0.0), _shift(usable, dy, dx, False) & usable
            wt = torch.exp(-0.5 * (dx * dx + dy * dy) / SIGMA_S**2 - 0.5 * (mm - m) ** 2 / SIGMA_R**2) * use
            vals += wt * _shift(raw.double(), dy, dx, 0.0)
            wsum += wt
    depth = torch.where(wsum > 0, torch.floor(vals / wsum.clamp_min(1e-300) + 0.5), 0.0).to(torch.int64)
    out = {}
    k = _camera(w, h)
    for level in range(3):
        if level > 0:
            a = depth[: depth.shape[0] // 2 * 2, : depth.shape[1] // 2 * 2]
            four = torch.stack([a[0::2, 0::2], a[0::2, 1::2], a[1::2, 0::2], a[1::2, 1::2]])
            cnt, hi = (four != 0).sum(0), four.amax(0)
            lo = torch.where(four == 0, 1 << 20, four).amin(0)
            # whether a block or a difference jumps is decided in 32 bits, as the limit is given in them
            jump = hi.float() / SCALE - torch.minimum(lo, hi).float() / SCALE > np.float32(JUMP)
            depth = torch.where((cnt > 0) & ~jump, (four.sum(0) + cnt // 2) // cnt.clamp_min(1), 0)
        hh, ww = depth.shape
        s = 1.0 / (1 << level)
        fx, fy, cx, cy = k.fx * s, k.fy * s, k.cx * s, k.cy * s
        z = depth.double() / SCALE
        bad = (depth == 0) | (z < MIN_DEPTH) | (z > MAX_DEPTH)
        z = torch.where(bad, math.nan, z)
        ys = torch.arange(hh, device="cuda", dtype=torch.float64)[:, None]
        xs = torch.arange(ww, device="cuda", dtype=torch.float64)[None, :]
        v = torch.stack([(xs - cx) * z / fx, (ys - cy) * z / fy, z], dim=-1)
        nb = {d: _shift(v, d[0], d[1], math.nan) for d in ((0, -1), (0, 1), (-1, 0), (1, 0))}
        left, right, top, bottom = nb[(0, -1)], nb[(0, 1)], nb[(-1, 0)], nb[(1, 0)]
        z32 = {d: t[..., 2].float() for d, t in nb.items()}
        n = torch.linalg.cross(bottom - top, right - left)
        n = n / n.norm(dim=-1, keepdim=True)
        jump = ((z32[(0, 1)] - z32[(0, -1)]).abs() > np.float32(JUMP)) | ((z32[(1, 0)] - z32[(-1, 0)]).abs() > np.float32(JUMP))
        n = torch.where((jump | torch.isnan(v[..., 2]))[..., None], math.nan, n)
        pad = torch.zeros(hh, ww, 1, device="cuda", dtype=torch.float64)
        out["level%d" % level] = {"depth": None, "vertices": torch.cat([v, pad], -1), "normals": torch.cat([n, pad], -1)}
    return out


def _exact_integrate(case, seed):
    p = _volume_config(case)
    g, k = p.volume, p.intrinsics
    frames = _integration_frames(case, seed)
    frames.append(frames[0])  # prepare() fuses all of them, the pass the first one again
    nx, ny, nz = g.resolution
    w, h, trunc = case["width"], case["height"], g.truncation_distance
    color = case["color"] == "float"
    dev = {"device": "cuda", "dtype": torch.float64}
    xs, ys = torch.arange(nx, **dev), torch.arange(ny, **dev)
    per_pixel = []
    for depth, image, normals, w2c in frames:
        d = (depth.to(torch.int64) & 0xFFFF).double() / SCALE
        v, u = torch.meshgrid(torch.arange(h, **dev), torch.arange(w, **dev), indexing="ij")
        ray = torch.stack([(u - k.cx) / k.fx, (v - k.cy) / k.fy, torch.ones_like(u)], -1)
        lam = ray.norm(dim=-1)
        wt = torch.ones_like(d)
        if case["rule"] == "angle-weighted":
            n = normals[..., :3].double()
            cos = -(n * ray).sum(-1) / (lam * n.norm(dim=-1))
            wt = torch.where(torch.isfinite(cos), cos.clamp_min(0.0) / d, 1.0)
        ok = (d >= MIN_DEPTH) & (d <= MAX_DEPTH) & (wt > 0)
        rgb = None
        if color:
            px = image.to(torch.int64)
            rgb = torch.stack([px & 255, (px >> 8) & 255, (px >> 16) & 255], -1).double().reshape(-1, 3)
        m = torch.from_numpy(np.asarray(w2c, np.float64)[:3].astype(np.float32).astype(np.float64)).cuda()
        per_pixel.append((d.reshape(-1), lam.reshape(-1), wt.reshape(-1), ok.reshape(-1), rgb, m))
    whole = case["store"] != "float"  # the packed voxels are bytes
    vox = None if whole else torch.empty(nz, ny, nx, 2, **dev)
    col = torch.empty(nz, ny, nx, 4, **dev) if color else None
    slab = max(1, (1 << 23) // (nx * ny))
    for z0 in range(0, nz if color or not whole else 0, slab):
        zs = torch.arange(z0, min(nz, z0 + slab), **dev)
        c = [g.origin[a] + (t + 0.5) * g.voxel_size for a, t in enumerate((xs, ys, zs))]
        tsdf, weight = torch.ones(len(zs), ny, nx, **dev), torch.zeros(len(zs), ny, nx, **dev)
        cc = torch.zeros(len(zs), ny, nx, 4, **dev) if color else None
        for d, lam, wt, ok, rgb, m in per_pixel:
            cam = [m[r, 0] * c[0][None, None, :] + m[r, 1] * c[1][None, :, None] + m[r, 2] * c[2][:, None, None]
                   + m[r, 3] for r in range(3)]
            u, v = torch.floor(k.fx * cam[0] / cam[2] + k.cx + 0.5), torch.floor(k.fy * cam[1] / cam[2] + k.cy + 0.5)
            use = (cam[2] > 0) & (u >= 0) & (u < w) & (v >= 0) & (v < h)
            at = torch.where(use, v * w + u, 0.0).long()
            sd = d[at] - torch.sqrt(cam[0] ** 2 + cam[1] ** 2 + cam[2] ** 2) / lam[at]
            use &= ok[at] & (sd >= -trunc)
            t, wn = (sd / trunc).clamp(-1.0, 1.0), torch.where(use, wt[at], 0.0)
            tsdf = torch.where(use, (tsdf * weight + t * wn) / (weight + wn).clamp_min(1e-300), tsdf)
            weight = torch.where(use, (weight + wn).clamp_max(196.0), weight)
            if color:
                near = use & (sd <= 0.5 * trunc)
                cw, den = cc[..., 3:], (cc[..., 3:] + wn[..., None]).clamp_min(1e-300)
                new = torch.cat([(cc[..., :3] * cw + rgb[at] * wn[..., None]) / den,
                                 (cw + wn[..., None]).clamp_max(196.0)], -1)
                cc = torch.where(near[..., None], new, cc)
        if not whole:
            vox[z0:z0 + len(zs)] = torch.stack([tsdf, weight], -1)
        if color:
            col[z0:z0 + len(zs)] = cc
    out = {"voxels": None if whole else vox.reshape(-1, 2)}
    if color:
        out["colors"] = col.reshape(-1, 4)
    return out if color or not whole else None


def _exact_posenet(case, seed):
    pairs, targets = _pairs(case, seed)
    net = PN.PoseNet(PN.PoseNetConfig(batch_capacity=1, seed=seed % (1 << 31)))
    flat = torch.from_numpy(net.parameters().astype(np.float64)).requires_grad_(True)
    net.close()
    raw = (pairs.to(torch.int64) & 0xFFFF).cpu().double()
    x = torch.where(raw == 0, 0.0, raw / SCALE - 1.5)
    scale = torch.tensor([0.1, 0.1, 0.1, 0.03, 0.03, 0.03], dtype=torch.float64)
    at = 0

    def take(*shape):
        nonlocal at
        n = int(np.prod(shape))
        at += n
        return flat[at - n:at].reshape(shape)

    channels = (2, 16, 32, 64, 64, 128)
    for cin, cout in zip(channels, channels[1:]):
        wt, b = take(cout, 3, 3, cin).permute(0, 3, 1, 2), take(cout)
        x = torch.relu(torch.nn.functional.conv2d(x, wt, b, stride=2, padding=1))
    x = x.permute(0, 2, 3, 1).reshape(x.shape[0], -1)
    wt, b = take(256, 2560), take(256)
    x = torch.relu(x @ wt.T + b)
    wt, b = take(6, 256), take(6)
    x = x @ wt.T + b
    if case["mode"] == "forward":
        return {"twists": (x * scale).detach()}
    loss = ((x - targets.cpu().double() / scale) ** 2).mean()
    loss.backward()
    return {"loss": float(loss), "gradients": flat.grad.numpy()}
