"""Shared helpers for the parity tests: configurations of the synthetic
workloads and conversions between the oracle's host arrays and the
library's device tensors."""
import ctypes as C

import numpy as np

INTR = (525.0, 525.0, 319.5, 239.5)
W, H = 640, 480


def config1_geometry(res=128, voxel=0.01, margin=0.5, trunc=0.05):
    """Volume of the 5-frame small workload: res^3 voxels, origin
    (-res*v/2, -res*v/2, -margin) (src/app/app_options.cpp:33-38)."""
    half = np.float32(0.5) * np.float32(res) * np.float32(voxel)
    return res, voxel, (-float(half), -float(half), -margin), trunc


def pipeline_config(K, res=128, voxel=0.01, margin=0.5, trunc=0.05, store="float", rule="angle-weighted",
                    color="float", radius=3, sigma_s=4.5, sigma_r=0.03, levels=3, **kw):
    r, v, origin, t = config1_geometry(res, voxel, margin, trunc)
    # sparse storage integrates its band (Pipeline::require_valid_storage)
    mode = "band" if kw.get("storage") == "hashed" else "full"
    return K.PipelineConfig(
        voxel=store, tsdf_rule=rule, color=color,
        volume=K.VolumeGeometry((r, r, r), v, origin, t),
        integration=K.TsdfIntegrationOptions(depth_scale=1000.0, mode=mode),
        depth=K.DepthProcessingOptions(levels=levels, bilateral_radius=radius, bilateral_spatial_sigma=sigma_s,
                                       bilateral_depth_sigma=sigma_r),
        intrinsics=K.CameraIntrinsics(*INTR), width=W, height=H, **kw)


def oracle_volume(ko, res=128, voxel=0.01, margin=0.5, trunc=0.05, kind=0, color=True):
    r, v, origin, t = config1_geometry(res, voxel, margin, trunc)
    return ko.Volume.create(r, v, origin, t, kind, color)


STORE_KIND = {"float": 0, "quantized": 1, "bf16": 2}
RULE = {"classic": 0, "angle-weighted": 1}


def to_dev(torch, a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16)).cuda()
    if a.dtype == np.uint32:
        return torch.from_numpy(a.view(np.int32)).cuda()
    return torch.from_numpy(a).cuda()


def f4(a3):
    """(H, W, 3) float32 -> (H, W, 4) float32 with w = 0."""
    out = np.zeros(a3.shape[:2] + (4,), np.float32)
    out[..., :3] = a3
    return out


def host(t):
    return t.detach().cpu().numpy()


def same_bits(a, b):
    """Bitwise equality of float arrays (NaN payloads compared as bits)."""
    a = np.ascontiguousarray(a)
    b = np.ascontiguousarray(b)
    return a.shape == b.shape and np.array_equal(a.view(np.uint8), b.view(np.uint8))


def first_mismatch(a, b):
    a32 = np.ascontiguousarray(a).view(np.uint32).reshape(-1)
    b32 = np.ascontiguousarray(b).view(np.uint32).reshape(-1)
    idx = np.nonzero(a32 != b32)[0]
    return (len(idx), idx[:5], a.reshape(-1)[idx[:5]], b.reshape(-1)[idx[:5]]) if len(idx) else None


def noisy_pipeline(K, res, seed=0):
    """A pipeline over res^3 voxels of random signs: about two triangles a voxel."""
    p = K.Pipeline(K.PipelineConfig(voxel="bf16", color="none",
                                    volume=K.VolumeGeometry((res,) * 3, 0.01, (0, 0, 0), 0.05)))
    t = np.random.default_rng(seed).uniform(-1.0, 1.0, res ** 3).astype(np.float32)
    vox = np.empty((res ** 3, 2), np.uint16)
    vox[:, 0], vox[:, 1] = t.view(np.uint32) >> 16, 256
    p.upload_volume(vox)
    return p


def extract_mesh(p):
    """A mesh by the C entry points: its handle, vertices and triangles."""
    from kinectfusion_amd import _native as N

    lib, h, nv, nt = N.hip(), C.c_void_p(), C.c_int64(), C.c_int64()
    N.check(lib.kf_mesh_extract(p.ctx, 0.0, C.byref(h)), p.ctx)
    N.check(lib.kf_mesh_size(h, C.byref(nv), C.byref(nt)))
    return h, nv.value, nt.value


def copy_mesh(mesh):
    """The status of kf_mesh_copy and its four arrays."""
    from kinectfusion_amd import _native as N

    h, nv, nt = mesh
    out = [np.zeros((nv, 3), np.float32) for _ in range(3)] + [np.zeros((nt, 3), np.uint32)]
    return N.hip().kf_mesh_copy(h, *(a.ctypes.data_as(C.c_void_p) for a in out)), out


def same_mesh(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))
