"""Reinsertion steps that find nothing to move, before, between and after steps that do: the step after one reads the
number of moves before it launches the conflict rounds.  The BVH2 equals the oracle's."""
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from test_gpu_parity import assert_same_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 600, 5000])
def test_steps_without_moves(ctx, n):
    tris = scenes.soup(n, seed=n)
    bvh = ob.PlocBuilder(ctx).build(14, tris)
    want = O.ploc_build(O.tri_aabbs(tris), 14, 0)["nodes"]
    # one candidate, the node after the root, then all again
    mixed, settling = [1e-9, 1.0, 1e-9, 1e-9, 0.5], [1.0] * 12
    for seq in (mixed, settling, mixed):
        bvh.reinsertion(0.6, seq)
        want = O.reinsertion(want, 0.6, seq)
        assert_same_bytes(bvh.nodes, want, f"BVH2 after {len(seq)} steps")
