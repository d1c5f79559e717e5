"""The work a program gives this framework, as cases whose time can be measured.

Each case stands for one way the ray-casting path is used: frames of a viewer
from a thumbnail to the 28M-triangle benchmark frame, a scene of many objects,
a set of frames rendered as one batch, frames bounded by a trained proposal
network, the ray queries, the voxel grid, point clouds, the training of a
proposal network, and loading a mesh.  Meshes, cameras, lights, rays and points
come from the seed; the generators are the package's own displaced tori and
icospheres.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call
    run(state)           one pass through the public entry points
    work(case)           bytes and operations that no implementation can avoid
    exact(case, seed)    the same outputs in 64 bits, by plain torch, where feasible
"""
import ctypes as C
import math

import numpy as np
import torch

import j3d_amd as J
from j3d_amd import ffi

FLT_MAX = float(np.finfo(np.float32).max)
DEVICE = "cuda"


def listed():
    return [
        # a thumbnail or preview of a small model: launches and latency
        {"name": "frame_thumbnail", "kind": "frame", "mesh": "torus", "tris": 20000, "objects": 1, "w": 256, "h": 192,
         "shadow": "none", "builder": "host"},
        # a viewer's window on a scanned model without shadows (the 327,680-triangle icosphere at 1024x768)
        {"name": "frame_window", "kind": "frame", "mesh": "icosphere", "tris": 327680, "objects": 1, "w": 1024,
         "h": 768, "shadow": "none", "builder": "host"},
        # the benchmark frame: 28M triangles, full HD, one directional shadow ray per hit
        {"name": "frame_hd_28m", "kind": "frame", "mesh": "torus", "tris": 28000000, "objects": 1, "w": 1920,
         "h": 1080, "shadow": "directional", "builder": "device"},
        # an assembly of 256 parts under the scene's point light: the top-level tree
        {"name": "frame_256_objects", "kind": "frame", "mesh": "torus", "tris": 20000, "objects": 256, "w": 1366,
         "h": 767, "shadow": "point", "builder": "host"},
        # a frame whose primary rays a trained proposal network bounds
        {"name": "frame_learned", "kind": "learned", "mesh": "torus", "tris": 4000000, "w": 1280, "h": 720,
         "shadow": "directional", "builder": "device"},
        # views of several models of uneven size rendered together (contact sheet, data generation)
        {"name": "batch_24_frames", "kind": "batch", "meshes": 8, "frames": 24, "tris_lo": 10000, "tris_hi": 4000000,
         "builder": "device"},
        # closest-hit queries on device buffers: picking, distance fields, simulation
        {"name": "rays_closest_1m", "kind": "closest", "mesh": "torus", "tris": 4000000, "rays": 1048576,
         "builder": "device"},
        # visibility queries of a host program
        {"name": "rays_visible_200k", "kind": "visible", "mesh": "icosphere", "tris": 327680, "rays": 200003,
         "builder": "host"},
        # a mesh to a voxel grid
        {"name": "voxels_256", "kind": "voxels", "mesh": "torus", "tris": 2000000, "dim": 256, "builder": "device"},
        # a scanned point cloud with normals and colours
        {"name": "points_12m", "kind": "points", "points": 12000000, "w": 1920, "h": 1080},
        # fitting a mesh's proposal network
        {"name": "train_512k_rays", "kind": "train", "mesh": "torus", "tris": 1000000, "rays": 524288, "epochs": 2,
         "batch": 16384, "builder": "device"},
        # opening a model: upload, tree on the GPU, a first query, and closing it again
        {"name": "load_2m", "kind": "load", "tris": 2000000, "rays": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "scene", "learned", "batch", "closest", "visible", "voxels", "points",
                       "train", "load"])
    w, h = rng.choice([(_log(rng, 160, 1920), _log(rng, 120, 1080)), (1280, 720), (640, 480), (1920, 1080)])
    mesh = rng.choice(["torus", "torus", "icosphere"])
    if kind == "frame":
        tris = _log(rng, 2000, 8000000)
        return {"kind": "frame", "mesh": mesh, "tris": tris, "objects": rng.choice([1, 1, 2, 3]), "w": w, "h": h,
                "shadow": rng.choice(["none", "directional", "point"]),
                "builder": "host" if tris < 500000 else "device"}
    if kind == "scene":
        return {"kind": "frame", "mesh": "torus", "tris": _log(rng, 1000, 30000), "objects": _log(rng, 17, 300),
                "w": w, "h": h, "shadow": rng.choice(["none", "directional", "point"]), "builder": "host"}
    if kind == "learned":
        return {"kind": "learned", "mesh": mesh, "tris": _log(rng, 50000, 6000000), "w": w, "h": h,
                "shadow": rng.choice(["none", "directional"]), "builder": "device"}
    if kind == "batch":
        return {"kind": "batch", "meshes": rng.randint(1, 8), "frames": rng.randint(2, 32), "tris_lo": 5000,
                "tris_hi": _log(rng, 20000, 4000000), "builder": rng.choice(["device", "host"])}
    if kind == "closest":
        return {"kind": "closest", "mesh": mesh, "tris": _log(rng, 5000, 6000000), "rays": _log(rng, 1000, 2000000),
                "builder": "device"}
    if kind == "visible":
        return {"kind": "visible", "mesh": mesh, "tris": _log(rng, 5000, 1000000), "rays": _log(rng, 500, 500000),
                "builder": "device"}
    if kind == "voxels":
        return {"kind": "voxels", "mesh": mesh, "tris": _log(rng, 5000, 4000000), "dim": _log(rng, 24, 320),
                "builder": "device"}
    if kind == "points":
        return {"kind": "points", "points": _log(rng, 20000, 16000000), "w": w, "h": h}
    if kind == "train":
        return {"kind": "train", "mesh": mesh, "tris": _log(rng, 20000, 2000000), "rays": _log(rng, 20000, 1000000),
                "epochs": rng.randint(1, 2), "batch": rng.choice([4096, 8192, 16384]), "builder": "device"}
    return {"kind": "load", "tris": _log(rng, 5000, 4000000), "rays": _log(rng, 64, 20000)}


# ------------------------------------------------------------------ inputs ----

def _mesh(kind, tris, seed):
    """A displaced icosphere of the level nearest to `tris` triangles, or a displaced torus of about that many."""
    if kind == "icosphere":
        level = max(1, min(8, int(round(math.log(max(tris, 80) / 20.0, 4)))))
        return J.icosphere(level, seed=seed + 1, amplitude=0.02)
    nv = max(4, int(round(math.sqrt(tris / 2.0 / 1.8))))
    nu = max(4, int(round(tris / 2.0 / nv)))
    return J.torus(nu, nv, seed=seed + 1)


def _in_box(v, size):
    """The vertices in a box of the given size from the origin (the same grid for every seed)."""
    lo, hi = v.min(axis=0), v.max(axis=0)
    return np.ascontiguousarray((v - lo) / (hi - lo) * np.asarray(size, np.float32), np.float32)


def _builder(case):
    return ffi.BUILD_DEVICE if case["builder"] == "device" else ffi.BUILD_HOST


def _poses(n, rng, side):
    out = []
    for _ in range(n):
        q, r = np.linalg.qr(rng.normal(size=(3, 3)))
        q = q * np.sign(np.diag(r))
        if np.linalg.det(q) < 0:
            q[:, 0] = -q[:, 0]
        m = np.eye(4)
        m[:3, :3] = q
        m[:3, 3] = rng.uniform(-side, side, 3)
        out.append(np.ascontiguousarray(m.T, np.float32).reshape(16))
    return out


FLAGS = {"none": ffi.EDGES | ffi.SHADING, "point": ffi.EDGES | ffi.SHADING | ffi.SHADOW,
         "directional": ffi.EDGES | ffi.SHADING | ffi.SHADOW | ffi.DIRECTIONAL_LIGHT}


def _view(rng, dist, w, h, pivot, diag, slots, shadow, seed, **kw):
    az, el = rng.uniform(0.0, 2.0 * math.pi), rng.uniform(0.2, 0.8)
    cs, ci = J.orbit_camera(dist * rng.uniform(0.9, 1.1), az, el)
    cam = J.camera_with_vertical_fov(60.0)
    flags = FLAGS[shadow] | kw.pop("flags", 0)
    return J.make_frame(w, h, cam, cs, ci, pivot, diag, slots, flags=flags, light_dir=J.random_hemisphere(seed + 12),
                        **kw)


class _DeviceArray:
    """A buffer of the renderer's as an array that torch wraps without a copy; the tensor keeps the renderer alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (int(ptr), False), "version": 2,
                                         "strides": None}


def _target(r, w, h):
    """A target and its G-buffer (8 words per pixel, as int32 and as float32) and image, where they lie on the GPU."""
    tg = r.create_target(w, h)
    g, im = C.c_void_p(), C.c_void_p()
    rc = r.lib.j3dg_target_device_ptrs(r.ctx, tg, C.byref(g), C.byref(im))
    assert rc == 0
    words = torch.as_tensor(_DeviceArray(r, g.value, (h, w, 8), "<i4"), device=DEVICE)
    rgba = torch.as_tensor(_DeviceArray(r, im.value, (h, w), "<i4"), device=DEVICE)
    return tg, words, words.view(torch.float32), rgba


def _frame_outputs(words, floats, rgba):
    """The whole G-buffer by field (j3dg_pixel) and the image."""
    return {"mark": words[..., 0], "surface": floats[..., 1:4], "object_id": words[..., 4], "bary": floats[..., 5:7],
            "db_id": words[..., 7], "rgba": rgba}


def _scene(case, seed, rng):
    """(meshes, poses, camera distance, half side of the scene) of a frame case."""
    n = case["objects"]
    if n == 1:
        return [_mesh(case["mesh"], case["tris"], seed)], [None], 3.0, 1.5
    distinct = [_mesh(case["mesh"], case["tris"], seed + 7 * k) for k in range(min(n, 4))]
    side = 1.2 * n ** (1.0 / 3.0)
    return [distinct[i % len(distinct)] for i in range(n)], _poses(n, rng, side), 2.5 * side + 2.0, side


def _rays(n, rng, radius, spread):
    """Rays from a shell around the origin towards points near it; every 16th aims anywhere."""
    o = rng.normal(size=(n, 3))
    o = o / np.linalg.norm(o, axis=1, keepdims=True) * rng.uniform(radius, 1.5 * radius, (n, 1))
    d = rng.uniform(-spread, spread, (n, 3)) - o
    d[::16] = rng.normal(size=d[::16].shape)
    d = d / np.linalg.norm(d, axis=1, keepdims=True)
    r = np.zeros((n, 8), np.float32)
    r[:, :3], r[:, 3:6], r[:, 7] = o, d, FLT_MAX
    return r


def _cloud(case, seed):
    """Points of a displaced sphere, as a scanner gives them (rows along a helix), with normals and colours."""
    n = case["points"]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    i = torch.arange(n, device=DEVICE, dtype=torch.float64)
    z = 1.0 - 2.0 * (i + 0.5) / n
    phi = i * (2.0 * math.pi * max(8.0, math.sqrt(n)) / n)
    rho = torch.sqrt(1.0 - z * z)
    nrm = torch.stack([rho * torch.cos(phi), rho * torch.sin(phi), z], 1)
    k = torch.randn((4, 3), generator=g, device=DEVICE, dtype=torch.float64) * 3.0
    r = 1.0 + 0.05 * torch.sin(nrm @ k.T).sum(1, keepdim=True)
    r = r + 0.004 * torch.randn((n, 1), generator=g, device=DEVICE, dtype=torch.float64)
    xyz = (nrm * r).float()
    col = torch.randint(0, 1 << 24, (n,), generator=g, device=DEVICE, dtype=torch.int64) | 0xFF000000
    return xyz.cpu().numpy(), nrm.float().cpu().numpy(), col.cpu().numpy().astype(np.uint32)


def _points_view(case, seed):
    rng = np.random.default_rng(seed)
    cs, ci = J.orbit_camera(2.6 * rng.uniform(0.95, 1.05), rng.uniform(0.0, 6.28), rng.uniform(0.2, 0.8))
    cam = J.camera_with_vertical_fov(60.0)
    P, Pi = J.projection(cam, case["w"], case["h"])
    frame = J.Frame(case["w"], case["h"], Pi, cs, ci, np.zeros(3, np.float32), 2.2, [], flags=FLAGS["none"],
                    near_plane=cam.near_plane)
    return P, ci, frame


# ----------------------------------------------------------------- prepare ----

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    r = J.Renderer(0)
    s = {"kind": kind, "r": r}
    if kind in ("frame", "learned", "batch", "points"):
        r.set_matcap(*J.make_matcap(0))
    if kind == "frame":
        meshes, poses, dist, side = _scene(case, seed, rng)
        slots = [r.upload_mesh(v, t, db_id=J.make_db_id(1, i), cs=cs, builder=_builder(case))
                 for i, ((v, t), cs) in enumerate(zip(meshes, poses))]
        diag, pivot = J.scene_framing(meshes[0][0]) if case["objects"] == 1 else (2.0 * side, np.zeros(3, np.float32))
        s["frame"] = _view(rng, dist, case["w"], case["h"], pivot, diag, slots, case["shadow"], seed)
        s["target"], s["words"], s["floats"], s["rgba"] = _target(r, case["w"], case["h"])
    elif kind == "learned":
        v, t = _mesh(case["mesh"], case["tris"], seed)
        slot = r.upload_mesh(v, t, db_id=J.make_db_id(1, 0), builder=_builder(case))
        r.train_proposal(slot, n_rays=1 << 20, epochs=4, seed=seed + 1, n_validation=0)
        diag, pivot = J.scene_framing(v)
        s["frame"] = _view(rng, 3.0, case["w"], case["h"], pivot, diag, [slot], case["shadow"], seed,
                           flags=ffi.LEARNED, margin=0.05)
        s["target"], s["words"], s["floats"], s["rgba"] = _target(r, case["w"], case["h"])
    elif kind == "batch":
        lo, hi = math.log(case["tris_lo"]), math.log(case["tris_hi"])
        k = case["meshes"]
        sizes = [int(math.exp(lo + (hi - lo) * (i + 0.5) / k)) for i in range(k)]
        meshes = [_mesh("torus", n, seed + 7 * i) for i, n in enumerate(sizes)]
        slots = [r.upload_mesh(v, t, db_id=J.make_db_id(1, i), builder=_builder(case))
                 for i, (v, t) in enumerate(meshes)]
        framing = [J.scene_framing(v) for v, _ in meshes]
        sizes = [(256, 256), (640, 480), (1280, 720), (1920, 1080)]
        s["frames"], s["targets"], s["buffers"] = [], [], []
        for i in range(case["frames"]):
            w, h = sizes[(i // 2) % 4]
            diag, pivot = framing[i % k]
            s["frames"].append(_view(rng, 3.0, w, h, pivot, diag, [slots[i % k]], "none", seed + i))
            tg, words, _, rgba = _target(r, w, h)
            s["targets"].append(tg)
            s["buffers"].append((words, rgba))
    elif kind in ("closest", "visible", "voxels", "train"):
        v, t = _mesh(case["mesh"], case["tris"], seed)
        if kind == "voxels":
            v = _in_box(v, (2.0, 1.75, 1.0))
        s["slot"] = r.upload_mesh(v, t, builder=_builder(case))
        if kind == "closest":
            _device_query(s, _rays(case["rays"], rng, 2.5, 1.0))
        elif kind == "visible":
            s["rays"] = _rays(case["rays"], rng, 1.3, 1.0)
        elif kind == "voxels":
            s["dim"] = case["dim"]
        else:
            s["opts"] = {"n_rays": case["rays"], "epochs": case["epochs"], "batch": case["batch"], "seed": seed + 1,
                         "n_validation": 8192}
    elif kind == "points":
        xyz, nrm, col = _cloud(case, seed)
        s["cloud"] = r.upload_points(xyz, normals=nrm, colors=col, db_id=J.make_db_id(2, 0))
        s["proj"], s["cs_inv"], s["frame"] = _points_view(case, seed)
        s["target"], s["words"], s["floats"], s["rgba"] = _target(r, case["w"], case["h"])
    else:  # load
        s["mesh"] = _mesh("torus", case["tris"], seed)
        _device_query(s, _rays(case["rays"], rng, 2.5, 1.0))
    return s


def _device_query(s, rays):
    s["d_rays"] = torch.from_numpy(rays).to(DEVICE)
    n = rays.shape[0]
    s["hits"] = {"obj": torch.zeros(n, dtype=torch.int32, device=DEVICE),
                 "tri": torch.zeros(n, dtype=torch.int32, device=DEVICE), "t": torch.zeros(n, device=DEVICE),
                 "u": torch.zeros(n, device=DEVICE), "v": torch.zeros(n, device=DEVICE)}


# --------------------------------------------------------------------- run ----

def run(s):
    kind, r = s["kind"], s["r"]
    if kind in ("frame", "learned"):
        r.render(s["frame"], s["target"], readback=False)
        return _frame_outputs(s["words"], s["floats"], s["rgba"])
    if kind == "batch":
        r.render_batch(s["frames"], s["targets"])
        return s["buffers"]
    if kind == "closest":
        return _trace_device(s, s["slot"])
    if kind == "visible":
        return r.any_hit([s["slot"]], s["rays"])
    if kind == "voxels":
        return r.voxelize(s["slot"], s["dim"])
    if kind == "points":
        r.render(s["frame"], s["target"], readback=False)
        r.splat_points(s["target"], s["proj"], s["cs_inv"], ffi.SHADING, [s["cloud"]])
        return _frame_outputs(s["words"], s["floats"], s["rgba"])
    if kind == "train":
        rep = r.train_proposal(s["slot"], **s["opts"])
        params, norm = r.get_proposal(s["slot"])
        return {"params": params, "norm": norm, "loss": [rep["loss_first"], rep["loss_last"]],
                "hit_fraction": rep["hit_fraction"], "accuracy": rep["val_hit_accuracy"],
                "error": rep["val_mean_abs_error"], "resolved": rep["val_resolved"]}
    v, t = s["mesh"]
    slot = r.upload_mesh(v, t, builder=ffi.BUILD_DEVICE)
    info = r.mesh_info(slot)
    out = dict(_trace_device(s, slot))
    r.remove_mesh(slot)
    out["box"] = info["bb_min"] + info["bb_max"]
    return out


def _trace_device(s, slot):
    r, h = s["r"], s["hits"]
    slots = np.array([slot], np.uint32)
    rc = r.lib.j3dg_trace_rays_device(r.ctx, ffi.ptr(slots), 1, s["d_rays"].data_ptr(), s["d_rays"].shape[0],
                                      h["obj"].data_ptr(), h["tri"].data_ptr(), h["t"].data_ptr(), h["u"].data_ptr(),
                                      h["v"].data_ptr())
    if rc:
        raise RuntimeError("j3dg_trace_rays_device: %d" % rc)
    return h


# -------------------------------------------------------------------- work ----

def _trace_flops(rays, tris):
    """A ray through an 8-wide tree at its least: one path to a leaf (8 box tests of 18 operations per level) and two
    triangle tests of about 50."""
    return rays * (8 * 18 * max(1.0, math.log(max(tris, 8), 8)) + 100)


def work(case):
    kind = case["kind"]
    if kind in ("frame", "learned"):
        px = case["w"] * case["h"]
        tris = case["tris"] * case["objects"] if kind == "frame" else case["tris"]
        # the G-buffer and image written, the G-buffer read for shading, at most a triangle per pixel of the mesh read
        b = px * (32 + 32 + 4) + min(px, tris) * 48
        f = _trace_flops(px, tris) + px * 100
        if kind == "learned":
            f += 0.2 * px * 2 * 13312  # the rays that enter the object's box
        return {"bytes": b, "flops": f}
    if kind == "batch":
        area = [65536, 307200, 921600, 2073600]
        px = sum(area[(i // 2) % 4] for i in range(case["frames"]))
        tris = math.sqrt(case["tris_lo"] * case["tris_hi"])
        return {"bytes": px * 68 + min(px, tris * case["meshes"]) * 48, "flops": _trace_flops(px, tris) + px * 100}
    if kind == "closest":
        return {"bytes": case["rays"] * (32 + 20 + 48), "flops": _trace_flops(case["rays"], case["tris"])}
    if kind == "visible":
        return {"bytes": case["rays"] * (32 + 1 + 48), "flops": _trace_flops(case["rays"], case["tris"])}
    if kind == "voxels":
        rays, cells = 3 * case["dim"] ** 2 * 0.6, case["dim"] ** 3 * 0.3
        return {"bytes": cells + case["tris"] * 48, "flops": _trace_flops(rays, case["tris"])}
    if kind == "points":
        px = case["w"] * case["h"]
        return {"bytes": case["points"] * 12 + px * (32 + 32 + 4 + 16 + 16), "flops": case["points"] * 90}
    if kind == "train":
        n = case["rays"] * case["epochs"]
        return {"bytes": n * 40, "flops": n * 6 * 13312 + _trace_flops(case["rays"], case["tris"])}
    # the arrays up, read for the tree, the records and nodes written
    return {"bytes": case["tris"] * (6 + 12 + 18 + 24 + 48 + 48 + 12 + 24), "flops": case["tris"] * 200}


# ------------------------------------------------------------------- exact ----

def _mat(m):
    return torch.tensor(np.asarray(m, np.float64).reshape(4, 4).T.copy(), device=DEVICE)


def _closest(o, d, v, t, t_near):
    """Closest hit by testing every triangle, in 64 bits: (found, t, u, v, unit normal)."""
    v = torch.from_numpy(np.ascontiguousarray(v)).to(DEVICE).double()
    t = torch.from_numpy(t.astype(np.int64)).to(DEVICE)
    a, e1, e2 = v[t[:, 0]], v[t[:, 1]] - v[t[:, 0]], v[t[:, 2]] - v[t[:, 0]]
    nrm = torch.linalg.cross(e1, e2)
    n = d.shape[0]
    out = [torch.zeros(n, dtype=torch.bool, device=DEVICE)] + [torch.zeros(n, dtype=torch.float64, device=DEVICE)
                                                              for _ in range(3)]
    best = torch.zeros(n, dtype=torch.int64, device=DEVICE)
    step = max(1, 32000000 // t.shape[0])
    for i in range(0, n, step):
        dd, oo = d[i:i + step], o[i:i + step]
        det = dd @ nrm.T
        tt = ((a * nrm).sum(1)[None, :] - oo @ nrm.T) / det
        # with s = o - a: u = -e2 . (s x d) / (d . n), v = e1 . (s x d) / (d . n), e . (a x d) = d . (e x a)
        q = torch.linalg.cross(oo, dd)
        u = (dd @ torch.linalg.cross(e2, a).T - q @ e2.T) / det
        w = (q @ e1.T - dd @ torch.linalg.cross(e1, a).T) / det
        ok = (det != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (tt >= t_near)
        tt = torch.where(ok, tt, torch.full_like(tt, math.inf))
        m, k = tt.min(1)
        rows = torch.arange(m.shape[0], device=DEVICE)
        out[0][i:i + step] = m < math.inf
        out[1][i:i + step], out[2][i:i + step], out[3][i:i + step] = m, u[rows, k], w[rows, k]
        best[i:i + step] = k
    n1 = nrm[best]
    return out + [n1 / torch.linalg.norm(n1, dim=1, keepdim=True)]


def _exact_frame(case, seed):
    rng = np.random.default_rng(seed)
    w, h = case["w"], case["h"]
    (v, t), = _scene(case, seed, rng)[0]
    diag, pivot = J.scene_framing(v)
    f = _view(rng, 3.0, w, h, pivot, diag, [0], case["shadow"], seed)
    y, x = torch.meshgrid(torch.arange(h, device=DEVICE).double(), torch.arange(w, device=DEVICE).double(),
                          indexing="ij")
    one = torch.ones_like(x)
    sp = torch.stack([2 * (x + 0.5) / w - 1, 2 * (y + 0.5) / h - 1, one * f.near_plane, one], -1).reshape(-1, 4)
    d = sp @ _mat(f.proj_inv).T
    d[:, 3] = 0
    cs = _mat(f.cs)
    d = (d @ cs.T)[:, :3]
    o = cs[:3, 3].expand_as(d)
    hit, dist, u, b, n = _closest(o, d, v, t, f.diagonal / 100.0)
    n4 = torch.cat([n, torch.zeros_like(n[:, :1])], 1) @ _mat(f.cs_inv).T
    zero = torch.zeros_like(dist)
    surface = torch.stack([torch.where(hit, n4[:, 0], zero), torch.where(hit, n4[:, 1], zero),
                           torch.where(hit, dist, zero + FLT_MAX)], -1)
    bary = torch.stack([torch.where(hit, u, zero), torch.where(hit, b, zero)], -1)
    return {"mark": None, "surface": surface.reshape(h, w, 3), "object_id": None, "bary": bary.reshape(h, w, 2),
            "db_id": None, "rgba": None}


def _exact_points(case, seed):
    w, h = case["w"], case["h"]
    P, ci, _ = _points_view(case, seed)
    xyz = torch.from_numpy(_cloud(case, seed)[0]).to(DEVICE).double()
    c = torch.cat([xyz, torch.ones_like(xyz[:, :1])], 1) @ (_mat(P) @ _mat(ci)).T
    cw = c[:, 3]
    ok = (cw > 0) & (c[:, 0].abs() <= cw) & (c[:, 1].abs() <= cw)
    x = torch.floor((c[:, 0] / cw + 1) * 0.5 * w)
    y = torch.floor((c[:, 1] / cw + 1) * 0.5 * h)
    ok &= (x < w) & (y < h)
    z = torch.zeros(w * h, dtype=torch.float64, device=DEVICE)
    z.scatter_reduce_(0, (y[ok] * w + x[ok]).long(), 1 / cw[ok], "amax")
    depth = torch.where(z > 0, 1 / z, torch.full_like(z, FLT_MAX))
    surface = torch.stack([torch.zeros_like(depth), torch.zeros_like(depth), depth], -1)
    return {"mark": None, "surface": surface.reshape(h, w, 3), "object_id": None,
            "bary": torch.zeros((h, w, 2), dtype=torch.float64, device=DEVICE), "db_id": None, "rgba": None}


def _exact_closest(rays, mesh, extra=None):
    q = torch.from_numpy(rays).to(DEVICE).double()
    hit, t, u, v, _ = _closest(q[:, :3], q[:, 3:6], mesh[0], mesh[1], 0.0)
    zero = torch.zeros_like(t)
    out = {"obj": None, "tri": None, "t": torch.where(hit, t, zero + FLT_MAX), "u": torch.where(hit, u, zero),
           "v": torch.where(hit, v, zero)}
    out.update(extra or {})
    return out


def exact(case, seed):
    """Every triangle against every ray in 64 bits where that ends in seconds, the points' nearest per pixel, and
    nothing for what a tree alone makes feasible, for whole numbers and for a trained network."""
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "frame" and case["objects"] == 1 and case["w"] * case["h"] * case["tris"] <= 2e9:
        return _exact_frame(case, seed)
    if kind == "points":
        return _exact_points(case, seed)
    if kind == "closest" and case["rays"] * case["tris"] <= 1e10:
        mesh = _mesh(case["mesh"], case["tris"], seed)
        return _exact_closest(_rays(case["rays"], rng, 2.5, 1.0), mesh)
    if kind == "load" and case["rays"] * case["tris"] <= 1e10:
        mesh = _mesh("torus", case["tris"], seed)
        lo, hi = mesh[0].min(axis=0), mesh[0].max(axis=0)
        return _exact_closest(_rays(case["rays"], rng, 2.5, 1.0), mesh,
                              {"box": [float(x) for x in np.concatenate([lo, hi])]})
    return None
