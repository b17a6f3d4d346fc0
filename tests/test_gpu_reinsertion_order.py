"""Reinsertion of trees on either side of the size (2^20 nodes) from which the candidates are walked in node order, with
more candidates than the walk has lanes (2^18) and with fewer: the BVH2 after two steps equals the oracle's."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from test_gpu_parity import assert_same_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ratio", [(524288, 0.02), (524289, 0.02), (524289, 0.3), (60000, 0.9)])
def test_reinsertion_around_the_size(ctx, n, ratio):
    tris = scenes.soup(n, seed=n)
    params = ob.BvhBuildParams(ploc_search_distance=14, max_prims_per_leaf=3, reinsertion_batch_ratio=ratio)
    seq = [1.0, 1.0 / 3.0]
    cw = ob.build_cwbvh_from_tris(ctx, tris, params, ratio_sequence=seq)
    ref, rcw, rprims = O.build_cwbvh(tris, 14, 0, 3, reinsertion_batch_ratio=ratio, ratio_sequence=seq)
    assert_same_bytes(cw.bvh2.nodes, ref["nodes"], "BVH2")
    assert_same_bytes(cw.nodes, rcw, "CWBVH")
    np.testing.assert_array_equal(cw.primitive_indices, rprims)


def caterpillar(n):
    """A chain of n leaves, one level each: deeper than the walk that finds the levels goes (512) from 513 leaves on."""
    ref = O.ploc_build(O.tri_aabbs(scenes.soup(n, seed=n)), 14, 0)
    nodes = ref["nodes"].copy()
    leaves = ref["nodes"][ref["nodes"]["prim_count"] != 0]
    for k in range(n - 1):  # inner node at 0, 2, 4, ...; its children at 2k + 1 (leaf) and 2k + 2
        at = 0 if k == 0 else 2 * k
        nodes[at]["prim_count"], nodes[at]["first_index"] = 0, 2 * k + 1
        nodes[2 * k + 1] = leaves[k]
    nodes[2 * n - 2] = leaves[n - 1]
    return O.refit_all(nodes), ref["prim_indices"]


@pytest.mark.parametrize("n", [200, 511, 512, 513, 900])
def test_deep_tree(ctx, n):
    nodes, prims = caterpillar(n)
    bvh = ob.Bvh2.from_host(ctx, nodes, prims)
    assert_same_bytes(bvh.nodes, nodes, "uploaded")
    bvh.reinsertion(0.2, [1.0, 0.5, 1.0])
    assert_same_bytes(bvh.nodes, O.reinsertion(nodes, 0.2, [1.0, 0.5, 1.0]), "BVH2 after reinsertion")
    bvh.refit_all()
    assert_same_bytes(bvh.nodes, O.refit_all(O.reinsertion(nodes, 0.2, [1.0, 0.5, 1.0])), "BVH2 after a refit")


@pytest.mark.parametrize("n", [2, 3, 4, 600, 1100, 2500, 9000])
def test_small_trees(ctx, n):
    """Levels of up to 1,024 inner nodes are refitted by one workgroup."""
    tris = scenes.soup(n, seed=n)
    bvh = ob.PlocBuilder(ctx).build(14, tris)
    ref = O.ploc_build(O.tri_aabbs(tris), 14, 0)
    bvh.reinsertion(1.0, [1.0, 1.0, 0.5])
    assert_same_bytes(bvh.nodes, O.reinsertion(ref["nodes"], 1.0, [1.0, 1.0, 0.5]), "BVH2 after reinsertion")
