"""Large launches share a step's triangle tests over the wave through LDS.  Overlapping triangles, up to 24 pending per
visited node, fill those lists: most lanes have more pending than a step takes.  Hits equal the oracle's."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd.api import rt_triangles
from obvhs_amd.types import triangles_from_vertices

pytestmark = pytest.mark.gpu

N = 16 * 256 * 64 + 5  # 16 rows of 64 rays per compute unit of 256, and a few rays more


@pytest.mark.parametrize("spread", [0.05, 1.0])
def test_many_pending_tests(spread):
    rng = np.random.default_rng(int(spread * 100))
    c = rng.random((400, 1, 3))
    v = (c + spread * rng.normal(size=(400, 3, 3))).astype(np.float32)
    tris = triangles_from_vertices(v[:, 0], v[:, 1], v[:, 2])
    o = rng.normal(size=(N, 3))
    o *= 4.0 / np.linalg.norm(o, axis=1, keepdims=True)
    d = rng.random((N, 3)) - o
    r = np.zeros(N, dtype=ob.RAY)
    r["origin"][:, :3], r["direction"][:, :3] = o, d
    r["inv_direction"][:, :3] = ob.types.safe_inverse(d.astype(np.float32))
    r["tmin"], r["tmax"] = np.where(np.arange(N) % 3 == 0, 0.9, 0.0), np.where(np.arange(N) % 5 == 0, 1.0, 1e30)
    with ob.Context(0) as ctx:
        cw = ob.build_cwbvh_from_tris(ctx, tris, ob.BvhBuildParams(max_prims_per_leaf=3))
        bt = cw.reorder_triangles(tris)
        want = O.traverse(cw.nodes, tris[cw.primitive_indices], r, 0)
        assert (want["primitive_id"] != ob.INVALID_ID).sum() > N // 4
        assert cw.ray_traverse(r, bt).tobytes() == want.tobytes()
        assert cw.ray_traverse_rt(r, rt_triangles(ctx, bt)).tobytes() == want.tobytes()
        np.testing.assert_array_equal(cw.ray_traverse_miss(r, bt), want["primitive_id"] == ob.INVALID_ID)
