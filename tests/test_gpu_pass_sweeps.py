"""Refit and cost table of trees in pass order: launches over the slots of the large passes, then one workgroup for the
last 2,048 slots (1,024 leaves).  Sizes around that edge, every search distance (the number of passes), a chain with a
pass per leaf, and the level lists after the order is gone; nodes and CWBVH equal the oracle's."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from obvhs_amd.types import triangles_from_vertices
from test_gpu_parity import assert_same_bytes

pytestmark = pytest.mark.gpu


def moved_copy(tris):
    out = tris.copy()
    for k, name in enumerate(("v0", "v1", "v2")):
        out[name][:, :3] = out[name][:, :3] * np.float32(1.0 + 0.01 * k) + np.float32(0.25)
    return out


def refit_reference(nodes, prims, tris):
    expect = nodes.copy()
    leaves = np.nonzero(expect["prim_count"] != 0)[0]
    boxes = O.tri_aabbs(tris)
    for side in ("min", "max"):
        expect[side][leaves] = boxes[side][prims[expect["first_index"][leaves]]]
    return O.refit_all(expect)


def check(ctx, tris, sd, convert=True):
    bvh2 = ob.PlocBuilder(ctx).build(sd, tris)
    ref = O.ploc_build(O.tri_aabbs(tris), sd, 0)
    assert_same_bytes(bvh2.nodes, ref["nodes"], "BVH2")
    moved = moved_copy(tris)
    bvh2.refit_from_triangles(moved)
    expect = refit_reference(ref["nodes"], ref["prim_indices"], moved)
    assert_same_bytes(bvh2.nodes, expect, "refit BVH2")
    bvh2.refit_all()
    assert_same_bytes(bvh2.nodes, expect, "refit of the inner nodes")
    for mp in (3, 1) if convert else ():
        cw = ob.bvh2_to_cwbvh(bvh2, mp, True, False)
        rcw, rprims, _ = O.bvh2_to_cwbvh(expect, ref["prim_indices"], mp, True)
        assert_same_bytes(cw.nodes, rcw, f"CWBVH, at most {mp} per leaf")
        np.testing.assert_array_equal(cw.primitive_indices, rprims)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 257, 1023, 1024, 1025, 1026, 2049, 5000, 70000])
def test_sizes(ctx, n):
    check(ctx, scenes.soup(n, seed=n), 14)


@pytest.mark.parametrize("sd", [1, 2, 6, 24, 32])
def test_distances(ctx, sd):
    check(ctx, scenes.soup(3000, seed=sd), sd)


@pytest.mark.parametrize("n", [30, 120])
def test_chain(ctx, n):
    """Boxes at growing distances merge one at a time: about a pass per leaf (too deep for a CWBVH)."""
    x = 1.5 ** np.arange(n, dtype=np.float64)
    v = np.stack([np.stack([x, x * 0, x * 0], 1), np.stack([x, x * 0 + 0.1, x * 0], 1),
                  np.stack([x, x * 0, x * 0 + 0.1], 1)], 1).astype(np.float32)
    check(ctx, triangles_from_vertices(v[:, 0], v[:, 1], v[:, 2]), 14, convert=False)


def test_after_reinsertion(ctx):
    tris = scenes.soup(4000, seed=3)
    params = ob.BvhBuildParams(ploc_search_distance=14, max_prims_per_leaf=3, reinsertion_batch_ratio=0.05)
    b2 = ob.build_cwbvh_from_tris(ctx, tris, params).bvh2
    ref, _, _ = O.build_cwbvh(tris, 14, 0, 3, reinsertion_batch_ratio=0.05)
    moved = moved_copy(tris)
    b2.refit_from_triangles(moved)
    expect = refit_reference(ref["nodes"], ref["prim_indices"], moved)
    assert_same_bytes(b2.nodes, expect, "refit BVH2")
    cw = ob.bvh2_to_cwbvh(b2, 3, True, False)
    rcw, _, _ = O.bvh2_to_cwbvh(expect, ref["prim_indices"], 3, True)
    assert_same_bytes(cw.nodes, rcw, "CWBVH")
