"""Large launches split by rows of 64 rays: rows whose directions agree are traced a lane per ray, the others by the
chunked kernel.  Every entry point's results equal the allocation-free entry point's (one lane per ray) and the
chunked form's for launches that are all coherent, all incoherent, mixed row by row, and not a multiple of a row."""
import ctypes as C

import numpy as np
import pytest

import obvhs_amd as ob
from obvhs_amd import native, scenes
from obvhs_amd.api import rt_triangles

pytestmark = pytest.mark.gpu

# at least two rows per resident wave, whatever the kernel's occupancy: 256 compute units x 32 waves x 64 rays x 2
N = 2 * 256 * 32 * 64 + 37


def rays_of(kind, seed):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(N, 3))
    o = rng.random((N, 3)) * 1.5 - 0.25
    rows = np.arange(N) // 64
    agree = {"coherent": rows >= 0, "incoherent": rows < 0, "mixed": (rows * 2654435761 >> 7) % 3 == 0}[kind]
    base = rng.normal(size=(rows[-1] + 1, 3))
    d[agree] = base[rows[agree]] + 0.02 * d[agree]
    d[::9973] = [0.0, 0.0, 1.0]  # a row of its own kind here and there, and zero components
    r = np.zeros(N, dtype=ob.RAY)
    r["origin"][:, :3], r["direction"][:, :3] = o, d
    r["inv_direction"][:, :3] = ob.types.safe_inverse(d.astype(np.float32))
    r["tmax"] = 1e30
    return r


@pytest.mark.parametrize("kind", ["coherent", "incoherent", "mixed"])
def test_rows(kind):
    tris = scenes.soup(3000, seed=4)
    with ob.Context(0) as ctx:
        cw = ob.build_cwbvh_from_tris(ctx, tris, ob.BvhBuildParams(max_prims_per_leaf=3))
        d_tris, d_rays = cw.reorder_triangles(tris), ctx.upload(rays_of(kind, 7))
        d_rt = rt_triangles(ctx, d_tris)
        hits = ob.DeviceArray(ctx, ob.RAY_HIT, N)
        native.check(native.lib().obvhs_cwbvh_ray_traverse_noalloc(ctx.handle, cw.handle, d_tris.ptr, d_rays.ptr, N,
                                                                   hits.ptr), ctx.handle)
        want = hits.to_host()
        assert 1000 < (want["primitive_id"] != ob.INVALID_ID).sum() < N - 1000  # hits and misses
        calls = {"closest": lambda: cw.ray_traverse(d_rays, d_tris), "rt": lambda: cw.ray_traverse_rt(d_rays, d_rt),
                 "miss": lambda: cw.ray_traverse_miss(d_rays, d_tris),
                 "rt miss": lambda: cw.ray_traverse_rt(d_rays, d_rt, miss=True),
                 "wt": lambda: cw.ray_traverse_watertight(d_rays, d_tris),
                 "wt miss": lambda: cw.ray_traverse_watertight(d_rays, d_tris, miss=True)}
        for depth in (4, 8, 16):
            got = {}
            for chunk in (0, 1):
                ctx.set_tune_table(dict(ctx.tune_table(), trav_chunk=[chunk] * 4, trav_lds_depth=[depth] * 4))
                got[chunk] = {k: f() for k, f in calls.items()}
            for k in calls:
                np.testing.assert_array_equal(got[0][k], got[1][k], err_msg=k)
            assert got[0]["closest"].tobytes() == want.tobytes() and got[0]["rt"].tobytes() == want.tobytes()
            np.testing.assert_array_equal(got[0]["miss"], want["primitive_id"] == ob.INVALID_ID)
