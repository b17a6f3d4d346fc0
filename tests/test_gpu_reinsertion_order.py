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
