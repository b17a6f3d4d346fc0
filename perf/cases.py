"""Workloads of the framework's hot path, each one call sequence of a user's program on device-resident data.

A program keeps one context, its inputs and outputs as device arrays, and the handles of the trees it builds (builds
of a changing scene reuse their handle).  The C ABI is called through its ctypes binding with torch tensors as device
arrays.  Scenes follow the benchmark's recipes (soup, heightfield with boxes, long thin triangles, icospheres) with
the same sizes, generated on the device from the seed.  Tree bytes, primitive orders and hit ids are whole numbers;
hit distances are float32.
"""
import ctypes as C
import math

import numpy as np
import torch

import obvhs_amd as ob
from obvhs_amd import native

DEV = "cuda"
TMAX = 1e30

PRESETS = {
    # the benchmark's plain build: distance 14, no quality passes, 3 primitives per leaf
    "plain": lambda: ob.BvhBuildParams(ploc_search_distance=14, max_prims_per_leaf=3),
    "fastest": ob.BvhBuildParams.fastest_build,
    "fast": ob.BvhBuildParams.fast_build,
    "medium": ob.BvhBuildParams.medium_build,
    "slow": ob.BvhBuildParams.slow_build,
    # the benchmark's large scene: pre-splits capped at 1.3x the triangles, reinsertion 0.05 x [1, 1/3]
    "large": lambda: ob.BvhBuildParams(pre_split=True, ploc_search_distance=14, reinsertion_batch_ratio=0.05,
                                       max_prims_per_leaf=3),
}


def listed():
    return [
        # a small object rebuilt on its own: launches and host round trips are most of it
        {"name": "build_small", "kind": "build", "soup": 1501, "grid": 0, "boxes": 0, "thin": 0, "preset": "plain"},
        # the soup of the benchmark's plain leg
        {"name": "build_soup", "kind": "build", "soup": 65536, "grid": 0, "boxes": 0, "thin": 0, "preset": "plain"},
        # the heightfield with boxes (1,288,352 triangles) rebuilt each frame
        {"name": "build_heightfield", "kind": "build", "soup": 0, "grid": 724, "boxes": 20000, "thin": 0,
         "preset": "plain"},
        # an asset of the kitchen's size (56,939 triangles) built once at high quality: pre-splits, distance 24,
        # 128-bit sort keys, reinsertion over the default ratio sequence
        {"name": "build_slow", "kind": "build", "soup": 0, "grid": 150, "boxes": 0, "thin": 11939, "preset": "slow"},
        # the large scene (17,273,632 triangles) with its quality passes
        {"name": "build_large", "kind": "build", "soup": 0, "grid": 2896, "boxes": 0, "thin": 500000,
         "preset": "large"},
        # a deforming mesh: leaf boxes from the moved triangles, refit, conversion
        {"name": "refit_heightfield", "kind": "refit", "soup": 0, "grid": 724, "boxes": 20000, "thin": 0,
         "preset": "plain"},
        # many independent meshes rebuilt, their triangles reordered and a few rays traced, in shared launches
        {"name": "batch_build", "kind": "batch_build", "meshes": 4096, "max_level": 5, "rays_per_mesh": 64},
        # the plain leg's 256 x 256 primary rays
        {"name": "trace_small", "kind": "trace", "soup": 65536, "grid": 0, "boxes": 0, "thin": 0, "preset": "plain",
         "rays": "primary", "width": 256, "height": 256},
        # one 1080p frame: coherent primary rays, then a diffuse bounce per hit
        {"name": "trace_frame", "kind": "trace", "soup": 0, "grid": 724, "boxes": 20000, "thin": 0,
         "preset": "plain", "rays": "frame", "width": 1920, "height": 1080},
        # occlusion of an odd number of surface points toward a point light
        {"name": "trace_shadow", "kind": "trace", "soup": 0, "grid": 724, "boxes": 20000, "thin": 0,
         "preset": "plain", "rays": "shadow", "width": 1000003, "height": 1},
        # the headline: incoherent closest-hit rays against the large scene
        {"name": "trace_incoherent", "kind": "trace", "soup": 0, "grid": 2896, "boxes": 0, "thin": 500000,
         "preset": "large", "rays": "incoherent", "width": 1 << 22, "height": 1},
        # rays of many meshes in one launch
        {"name": "batch_trace", "kind": "batch_trace", "meshes": 4096, "max_level": 5, "rays_per_mesh": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case between the smallest and the largest sizes of the listed kinds."""
    kind = rng.choice(["build", "build", "build", "refit", "batch_build", "trace", "trace", "trace", "batch_trace"])
    if kind.startswith("batch"):
        per_mesh = rng.randint(8, 100) if kind == "batch_build" else _log_int(rng, 64, 2048)
        return {"kind": kind, "meshes": _log_int(rng, 16, 3000), "max_level": rng.randint(2, 5),
                "rays_per_mesh": per_mesh}
    n = _log_int(rng, 300, 2_500_000)
    case = {"kind": kind, "soup": 0, "grid": 0, "boxes": 0, "thin": 0}
    if rng.random() < 0.4:
        case["soup"] = n
    else:
        share = rng.uniform(0.6, 1.0)
        case["grid"] = max(3, int(math.sqrt(share * n / 2)))
        rest = max(0, n - 2 * case["grid"] ** 2)
        case["thin" if rng.random() < 0.5 else "boxes"] = rest // 24
    if kind == "build" and n < 700_000:
        case["preset"] = rng.choice(["plain", "plain", "fastest", "fast", "medium", "slow"])
    else:
        case["preset"] = rng.choice(["plain", "plain", "fastest"] if kind == "build" else ["plain", "plain", "fast"])
    if kind == "trace":
        case["rays"] = rng.choice(["primary", "frame", "shadow", "incoherent"])
        if case["rays"] in ("primary", "frame"):
            case["width"] = _log_int(rng, 32, 2048)
            case["height"] = max(1, int(case["width"] * rng.uniform(0.5, 1.0)))
        else:
            case["width"], case["height"] = _log_int(rng, 1000, 4_000_000), 1
            case["tuned"] = rng.random() < 0.4
    return case


# ---- the device side of the program ----

_contexts = {}
_tuned = False  # whether the case at hand uses the context whose table is set for incoherent rays


def context():
    if _tuned not in _contexts:
        ctx = _contexts[_tuned] = ob.Context(0)
        if _tuned:  # what the tuning run keeps for incoherent rays
            ctx.set_tune_table(dict(ctx.tune_table(), trav_chunk=[1] * 4))
    return _contexts[_tuned]


def _call(fn, *args):
    h = context().handle
    native.check(fn(h, *args), h)


def _p(t):
    return C.c_void_p(t.data_ptr())


def _tree_buffers(leaves, max_prims):
    """The program's own arrays for a tree: node words and primitive indices, with room to spare."""
    nodes = (leaves // 4 if max_prims > 1 else leaves) + 64
    return {"nodes": torch.zeros(nodes, 20, device=DEV, dtype=torch.int32),
            "primitive_indices": torch.zeros(leaves, device=DEV, dtype=torch.int32)}


def _copy_tree(cw, out):
    """Copies the CWBVH into the program's arrays (on the device, in stream order)."""
    lib = native.lib()
    nn, pn, a, b = C.c_uint32(), C.c_uint32(), C.c_void_p(), C.c_void_p()
    native.check(lib.obvhs_cwbvh_info(cw.handle, C.byref(nn), C.byref(pn), None))
    native.check(lib.obvhs_cwbvh_device_arrays(cw.handle, C.byref(a), C.byref(b)))
    if nn.value > out["nodes"].shape[0] or pn.value > out["primitive_indices"].shape[0]:
        raise MemoryError("tree arrays too small")
    _call(lib.obvhs_memcpy_dtod, _p(out["nodes"]), a, nn.value * 80)
    _call(lib.obvhs_memcpy_dtod, _p(out["primitive_indices"]), b, pn.value * 4)
    return {"node_count": nn.value, **out}


# ---- scenes ----

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float32)


def _pack(v):
    """(n, 3, 3) vertices as Triangle rows; adding 0 leaves no negative zero."""
    out = torch.zeros(v.shape[0], 3, 4, device=DEV, dtype=torch.float32)
    out[:, :, :3] = v.to(torch.float32) + 0.0
    return out


def _soup(n, g):
    return _pack(_rand(g, n, 1, 3) + (_rand(g, n, 3, 3) - 0.5) * 0.01)


def _sines(g):
    u = _rand(g, 3, 8).double()
    f = 1.0 + 31.0 * u[0]
    return f, 2 * math.pi * u[1], 2 * math.pi * u[2], 0.05 / f


def _height(x, z, sines):
    h = torch.zeros_like(x)
    for f, phase, ang, amp in zip(*(s.tolist() for s in sines)):
        h += amp * torch.sin(2 * math.pi * f * (x * math.cos(ang) + z * math.sin(ang)) + phase)
    return h


def _heightfield(grid, sines):
    c = torch.arange(grid + 1, device=DEV, dtype=torch.float64) / grid
    z, x = torch.meshgrid(c, c, indexing="ij")
    v = torch.stack([x, _height(x, z, sines), z], dim=-1).float()
    v00, v10, v01, v11 = v[:-1, :-1], v[:-1, 1:], v[1:, :-1], v[1:, 1:]
    t = torch.stack([torch.stack([v00, v01, v10], dim=-2), torch.stack([v10, v01, v11], dim=-2)], dim=2)
    return _pack(t.reshape(-1, 3, 3))


_CUBE = [(a, b, c) for q in ((0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3))
         for a, b, c in ((q[0], q[1], q[2]), (q[0], q[2], q[3]))]


def _boxes(n, sines, g):
    u = _rand(g, n, 3).double()
    s = 0.001 + 0.003 * u[:, 2]
    c = torch.stack([u[:, 0], _height(u[:, 0], u[:, 1], sines) + s, u[:, 1]], dim=-1)
    corner = torch.tensor([[(k >> 2) & 1, (k >> 1) & 1, k & 1] for k in range(8)], device=DEV).double() * 2 - 1
    v = c[:, None, :] + s[:, None, None] * corner[None]
    return _pack(v[:, torch.tensor(_CUBE, device=DEV)].reshape(-1, 3, 3))


def _sphere(g, n):
    u = _rand(g, 2, n)
    z = 1 - 2 * u[0]
    r = torch.sqrt(torch.clamp(1 - z * z, min=0))
    a = 2 * math.pi * u[1]
    return torch.stack([r * torch.cos(a), r * torch.sin(a), z], dim=-1)


def _thin(n, g):
    """Long thin triangles, length 0.05 to 0.5, aspect ratio 50 to 200."""
    u = _rand(g, 5, n)
    start = torch.stack([u[0], u[1] * 0.3, u[2]], dim=-1)
    length = (0.05 + 0.45 * u[3])[:, None]
    d = _sphere(g, n)
    helper = torch.zeros_like(d)
    helper[torch.arange(n, device=DEV), (d[:, 0].abs() >= 0.9).long()] = 1
    perp = torch.nn.functional.normalize(torch.linalg.cross(d, helper), dim=-1) * (length / (50 + 150 * u[4][:, None]) / 2)
    return _pack(torch.stack([start - perp, start + perp, start + d * length], dim=1))


def _scene(case, g):
    if case["soup"]:
        return _soup(case["soup"], g)
    sines = _sines(g)
    parts = [_heightfield(case["grid"], sines)]
    if case["boxes"]:
        parts.append(_boxes(case["boxes"], sines, g))
    if case["thin"]:
        parts.append(_thin(case["thin"], g))
    return torch.cat(parts)


# ---- rays ----

def _rays(origins, directions, tmax=TMAX):
    n = origins.shape[0]
    rows = [torch.zeros(n, 4, device=DEV, dtype=torch.float32) for _ in range(2)]
    rows[0][:, :3], rows[1][:, :3] = origins, directions
    out = torch.empty(n, 16, device=DEV, dtype=torch.float32)
    torch.cuda.synchronize()
    _call(native.lib().obvhs_rays_new, _p(rows[0]), _p(rows[1]), n, 0.0, tmax, _p(out))
    context().synchronize()
    return out


def _pinhole(width, height, eye, target):
    eye, target = (torch.tensor(v, device=DEV, dtype=torch.float64) for v in (eye, target))
    fwd = torch.nn.functional.normalize(target - eye, dim=0)
    right = torch.nn.functional.normalize(
        torch.linalg.cross(fwd, torch.tensor([0.0, 1.0, 0.0], device=DEV, dtype=torch.float64)), dim=0)
    up = torch.linalg.cross(right, fwd)
    k = math.tan(math.radians(60.0) / 2)
    y, x = torch.meshgrid(torch.arange(height, device=DEV), torch.arange(width, device=DEV), indexing="ij")
    sx = ((x + 0.5) / width * 2 - 1) * k * width / height
    sy = (1 - (y + 0.5) / height * 2) * k
    d = fwd + sx[..., None].double() * right + sy[..., None].double() * up
    d = torch.nn.functional.normalize(d.reshape(-1, 3), dim=-1).float()
    return _rays(eye.float().expand_as(d), d)


def _normals(t):
    a = t[:, 1, :3] - t[:, 0, :3]
    return torch.nn.functional.normalize(torch.linalg.cross(a, t[:, 2, :3] - t[:, 0, :3]), dim=-1)


def _bounce(rays, hits, bvh_tris, g):
    """One cosine-weighted bounce per hit."""
    prim, t = hits[:, 0], hits[:, 3].view(torch.float32)
    i = torch.nonzero(prim != -1)[:, 0]
    d = rays[i, 4:7]
    n = _normals(bvh_tris[prim[i].long()])
    n = torch.where((n * d).sum(-1, keepdim=True) > 0, -n, n)
    w = torch.nn.functional.normalize(n + _sphere(g, i.shape[0]) * 0.999, dim=-1)
    return _rays(rays[i, 0:3] + d * t[i][:, None] + n * 1e-4, w)


def _shadow(tris, n, g):
    """Surface points toward a light above the scene, ending at the light."""
    i = torch.randint(0, tris.shape[0], (n,), generator=g, device=DEV)
    b = _rand(g, 2, n).sqrt()
    v = tris[i][:, :, :3]
    u = torch.stack([1 - b[0], b[0] * (1 - b[1]), b[0] * b[1]], dim=-1)
    p = (v * u[..., None]).sum(1)
    light = torch.tensor([0.4, 0.9, 0.3], device=DEV) + 0.2 * _rand(g, 3)
    nrm = _normals(tris[i])
    nrm = torch.where((nrm * (light - p)).sum(-1, keepdim=True) < 0, -nrm, nrm)
    p = p + nrm * 1e-4
    d = light - p
    dist = torch.linalg.vector_norm(d, dim=-1)
    r = _rays(p, d / dist[:, None])
    r[:, 13] = dist
    return r


def _incoherent(n, g):
    """Origins on a sphere around the scene, uniform directions."""
    o = torch.tensor([0.5, 0.1, 0.5], device=DEV) + 0.8 * _sphere(g, n)
    return _rays(o, _sphere(g, n))


# ---- icosphere batches ----

_ico_cache = {}


def _icosphere(level):
    """Unit icosphere of 20 * 4^level triangles: vertices and faces."""
    if level not in _ico_cache:
        if level == 0:
            f = (1 + 5 ** 0.5) / 2
            v = np.array([[-1, f, 0], [1, f, 0], [-1, -f, 0], [1, -f, 0], [0, -1, f], [0, 1, f], [0, -1, -f],
                          [0, 1, -f], [f, 0, -1], [f, 0, 1], [-f, 0, -1], [-f, 0, 1]])
            t = np.array([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9], [5, 11, 4],
                          [11, 10, 2], [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2], [3, 2, 6], [3, 6, 8], [3, 8, 9],
                          [4, 9, 5], [2, 4, 11], [6, 2, 10], [8, 6, 7], [9, 8, 1]])
        else:
            v, t = (x.cpu().numpy() for x in _icosphere(level - 1))
            edges = np.sort(np.concatenate([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]]), axis=1)
            uniq, inv = np.unique(edges, axis=0, return_inverse=True)
            m = len(v) + inv.reshape(3, -1)
            v = np.concatenate([v, (v[uniq[:, 0]] + v[uniq[:, 1]]) / 2])
            a, b, c = t.T
            t = np.concatenate([np.stack(q, axis=1) for q in ((a, m[0], m[2]), (b, m[1], m[0]), (c, m[2], m[1]),
                                                              (m[0], m[1], m[2]))])
        v = v / np.linalg.norm(v, axis=1, keepdims=True)
        _ico_cache[level] = (torch.from_numpy(v).to(DEV), torch.from_numpy(t).to(DEV))
    return _ico_cache[level]


def _levels(case):
    """Subdivision levels: triangle counts log-uniform in [64, 65,536], rounded down to 20 * 4^level."""
    u = np.random.RandomState(case["meshes"]).rand(case["meshes"])
    s = np.floor(np.log(np.exp(np.log(64) + u * np.log(1024)) / 20) / np.log(4)).astype(int)
    return np.clip(s, 0, case["max_level"])


def _batch(case, seed):
    """Jittered icospheres, concatenated in mesh order, and rays from around each toward its inside."""
    g = _gen(seed)
    levels = _levels(case)
    m = case["meshes"]
    counts = 20 * 4 ** levels
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    tris = torch.zeros(int(offsets[-1]), 3, 4, device=DEV, dtype=torch.float32)
    for s in np.unique(levels):
        v, t = _icosphere(int(s))
        ids = np.nonzero(levels == s)[0]
        for part in np.array_split(ids, max(1, len(ids) * len(t) // 4_000_000)):  # bounded temporaries
            r = 0.9 + 0.2 * _rand(g, len(part), len(v), 1)
            at = torch.from_numpy(offsets[part].astype(np.int64)).to(DEV)[:, None] + torch.arange(len(t), device=DEV)
            tris[at.reshape(-1)] = _pack((v.float() * r)[:, t].reshape(-1, 3, 3))
    n = m * case["rays_per_mesh"]
    o = 2 * _sphere(g, n)
    rays = _rays(o, torch.nn.functional.normalize(2 * _rand(g, n, 3) - 1 - o, dim=-1))
    ray_mesh = torch.arange(m, device=DEV, dtype=torch.int32).repeat_interleave(case["rays_per_mesh"])
    return tris, offsets, rays, ray_mesh


# ---- what is measured ----

def _build(s):
    lib = native.lib()
    p, out = s["params"], C.c_void_p()
    ext = s["ext"]
    reuse = s["cw"].handle if s["cw"] is not None else None
    _call(lib.obvhs_build_cwbvh_from_tris_ex, _p(s["tris"]), s["n"], C.byref(p),
          None if ext is None else C.byref(ext), reuse, C.byref(out), None)
    if s["cw"] is None:
        s["cw"] = ob.CwBvh(context(), out)
    return s["cw"].handle


def _build_batch(s):
    out = C.c_void_p()
    reuse = s["batch"].handle if s["batch"] is not None else None
    _call(native.lib().obvhs_batch_build_cwbvh, _p(s["tris"]), s["offsets"].ctypes.data_as(C.c_void_p),
          len(s["offsets"]) - 1, C.byref(s["params"]), reuse, C.byref(out))
    if s["batch"] is None:
        s["batch"] = ob.CwBvhBatch(context(), out)
    return s["batch"].handle


def _hits(n):
    return torch.zeros(n, 4, device=DEV, dtype=torch.int32)


def _hit_outputs(hits):
    return {"ids": hits[:, :3], "t": hits.view(torch.float32)[:, 3]}


def prepare(case, seed):
    global _tuned
    _tuned = bool(case.get("tuned"))
    context()
    s = {"kind": case["kind"], "tuned": _tuned, "cw": None, "batch": None, "ext": None}
    if case["kind"].startswith("batch"):
        s["tris"], s["offsets"], s["rays"], s["ray_mesh"] = _batch(case, seed)
        s["params"] = PRESETS["plain"]().to_c()
        s["bvh_tris"] = torch.empty_like(s["tris"])
        s["hits"] = _hits(s["rays"].shape[0])
        torch.cuda.synchronize()
        if case["kind"] == "batch_trace":
            _call(native.lib().obvhs_batch_reorder_triangles, _build_batch(s), _p(s["tris"]), _p(s["bvh_tris"]))
            context().synchronize()
        return s
    g = _gen(seed)
    s["tris"] = _scene(case, g)
    s["n"] = s["tris"].shape[0]
    s["params"] = PRESETS[case["preset"]]().to_c()
    if case["preset"] == "large":
        s["seq"] = np.array([1.0, 1.0 / 3.0], np.float32)
        s["ext"] = native.BuildExt(int(s["n"] * 1.3), s["seq"].ctypes.data_as(C.c_void_p), 2)
    torch.cuda.synchronize()
    if case["kind"] in ("build", "refit"):
        leaves = s["n"] if not s["params"].pre_split else int(s["n"] * 1.3) if s["ext"] else 3 * s["n"]
        s["tree"] = _tree_buffers(leaves, s["params"].max_prims_per_leaf)
        torch.cuda.synchronize()
    if case["kind"] == "build":
        return s
    handle = _build(s)
    if case["kind"] == "refit":
        s["bvh2"] = s["cw"].bvh2
        extent = (s["tris"][:, :, :3].amax((0, 1)) - s["tris"][:, :, :3].amin((0, 1))).max()
        s["moved"] = s["tris"].clone()
        s["moved"][:, :, :3] += (_rand(g, s["n"], 3, 3) - 0.5) * (extent * 0.002)
        s["out"] = None
        torch.cuda.synchronize()
        return s
    info = C.c_uint32()
    native.check(native.lib().obvhs_cwbvh_info(handle, None, C.byref(info), None))
    s["bvh_tris"] = torch.empty(info.value, 3, 4, device=DEV, dtype=torch.float32)
    _call(native.lib().obvhs_cwbvh_reorder_triangles, handle, _p(s["tris"]), _p(s["bvh_tris"]))
    context().synchronize()
    n = case["width"] * case["height"]
    if case["rays"] == "incoherent":
        s["rays"] = [_incoherent(n, g)]
    elif case["rays"] == "shadow":
        s["rays"] = [_shadow(s["tris"], n, g)]
    elif case["soup"]:
        s["rays"] = [_pinhole(case["width"], case["height"], (0.5, 0.5, -1.5), (0.5, 0.5, 0.0))]
    else:
        s["rays"] = [_pinhole(case["width"], case["height"], (0.5, 0.45, -0.35), (0.5, 0.0, 0.55))]
    s["miss"] = case["rays"] == "shadow"
    if case["rays"] == "frame":
        first = _hits(n)
        _trace(s, s["rays"][0], first)
        context().synchronize()
        s["rays"].append(_bounce(s["rays"][0], first, s["bvh_tris"], g))
    # a bounce has a result for every pixel whose primary ray hit, packed at the front
    s["results"] = [torch.zeros(n, device=DEV, dtype=torch.uint8) if s["miss"] else _hits(n) for _ in s["rays"]]
    del s["tris"]
    torch.cuda.synchronize()
    return s


def _trace(s, rays, out):
    lib = native.lib()
    fn = lib.obvhs_cwbvh_ray_traverse_miss if s["miss"] else lib.obvhs_cwbvh_ray_traverse
    _call(fn, s["cw"].handle, _p(s["bvh_tris"]), _p(rays), rays.shape[0], _p(out))


def run(s):
    global _tuned
    _tuned = s["tuned"]
    lib = native.lib()
    if s["kind"] == "build":
        _build(s)
        return _copy_tree(s["cw"], s["tree"])
    if s["kind"] == "refit":
        _call(lib.obvhs_bvh2_refit_from_triangles, s["bvh2"].handle, _p(s["moved"]))
        out = C.c_void_p()
        _call(lib.obvhs_bvh2_to_cwbvh, s["bvh2"].handle, 3, 1, 0, s["out"].handle if s["out"] is not None else None,
              C.byref(out))
        if s["out"] is None:
            s["out"] = ob.CwBvh(context(), out)
        return _copy_tree(s["out"], s["tree"])
    if s["kind"].startswith("batch"):
        outputs = {}
        if s["kind"] == "batch_build":
            _call(lib.obvhs_batch_reorder_triangles, _build_batch(s), _p(s["tris"]), _p(s["bvh_tris"]))
            outputs["bvh_tris"] = s["bvh_tris"].view(torch.int32)
        _call(lib.obvhs_batch_ray_traverse, s["batch"].handle, _p(s["bvh_tris"]), _p(s["rays"]), _p(s["ray_mesh"]),
              s["rays"].shape[0], _p(s["hits"]))
        outputs.update(_hit_outputs(s["hits"]))
        return outputs
    for rays, out in zip(s["rays"], s["results"]):
        _trace(s, rays, out)
    return [out if s["miss"] else _hit_outputs(out) for out in s["results"]]


def _triangles(case):
    return case["soup"] or 2 * case["grid"] ** 2 + 12 * case["boxes"] + case["thin"]


def work(case):
    """Inputs read once, outputs written once; about one CWBVH node per ten primitives."""
    if case["kind"].startswith("batch"):
        n = 20 * 4 ** case["max_level"] * case["meshes"] // 4
        rays = case["meshes"] * case["rays_per_mesh"]
        build = n * (48 + 4 + 8 + 96) if case["kind"] == "batch_build" else 0
        return {"bytes": build + rays * (64 + 4 + 16) + min(56 * n, 1500 * rays), "flops": 2000 * rays}
    n = _triangles(case)
    if case["kind"] == "build":
        leaves = 1.1 * n if case["preset"] in ("slow", "large") else n
        return {"bytes": 48 * n + 12 * leaves, "flops": 1000 * leaves}
    if case["kind"] == "refit":
        return {"bytes": (48 + 64 + 4 + 64 + 12) * n, "flops": 500 * n}
    rays = case["width"] * case["height"] * (2 if case["rays"] == "frame" else 1)
    return {"bytes": rays * (64 + (1 if case["rays"] == "shadow" else 16)) + min(56 * n, 1500 * rays),
            "flops": 2000 * rays}


def exact(case, seed):
    """Hit distances of the closest hits by testing every triangle in 64 bits, where that is quick."""
    if case["kind"] != "trace" or case["rays"] not in ("primary", "incoherent"):
        return None
    rays_n = case["width"] * case["height"]
    if rays_n * _triangles(case) > 8e9:
        return None
    g = _gen(seed)
    tris = _scene(case, g)[:, :, :3].double()
    if case["rays"] == "incoherent":
        rays = _incoherent(rays_n, g)
    elif case["soup"]:
        rays = _pinhole(case["width"], case["height"], (0.5, 0.5, -1.5), (0.5, 0.5, 0.0))
    else:
        rays = _pinhole(case["width"], case["height"], (0.5, 0.45, -0.35), (0.5, 0.0, 0.55))
    v0, a, b = tris[:, 0], tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0]
    n = torch.linalg.cross(a, b)
    t = torch.full((rays_n,), math.inf, device=DEV, dtype=torch.float64)
    step = max(1, 30_000_000 // len(tris))
    for i in range(0, rays_n, step):
        o, d = rays[i:i + step, None, 0:3].double(), rays[i:i + step, None, 4:7].double()
        det = -(d * n).sum(-1)
        s = o - v0
        m = torch.linalg.cross(s, d.expand_as(s))
        u, v, tt = (b * m).sum(-1) / det, -(a * m).sum(-1) / det, (s * n).sum(-1) / det
        tt[~((u >= 0) & (v >= 0) & (u + v <= 1) & (tt >= 0))] = math.inf
        t[i:i + step] = tt.amin(-1)
    return [{"ids": None, "t": t}]
