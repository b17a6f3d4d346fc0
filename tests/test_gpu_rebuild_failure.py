"""A rebuild that fails half way (a leaf whose box is NaN has no neighbour) leaves nodes that are no tree: what follows
on the handle is refused, as for any other graph that is no tree, until it is built again."""
import numpy as np
import pytest

import obvhs_amd as ob
from obvhs_amd import scenes
from obvhs_amd.types import AABB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 5000])
def test_refit_after_a_failed_rebuild(ctx, n):
    tris = scenes.soup(n, seed=n)
    builder = ob.PlocBuilder(ctx)
    bvh = builder.build(14, tris)
    want = bvh.nodes.tobytes()
    leaf = np.nonzero(bvh.nodes["prim_count"] != 0)[0][n // 2:n // 2 + 1].astype(np.uint32)
    box = np.zeros(1, dtype=AABB)
    for k in AABB.names:
        box[k] = np.nan
    bvh.set_node_aabbs(leaf, box)
    with pytest.raises(ob.ObvhsError):
        builder.full_rebuild(bvh, 14)
    with pytest.raises(ob.ObvhsError):
        bvh.refit_from_triangles(tris)
    with pytest.raises(ob.ObvhsError):
        ob.bvh2_to_cwbvh(bvh, 3)
    builder.build_with_bvh(bvh, 14, tris)
    assert bvh.nodes.tobytes() == want
    bvh.refit_from_triangles(tris)
    assert bvh.nodes.tobytes() == want
