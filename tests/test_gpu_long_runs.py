"""Long runs of equal top words (more than 64 leaves in a cell of the codes' top 32 bits) where the passes have other
forms than in small builds: passes without work in one launch each (up to 1,024 tiles), with sums over groups of tiles,
and with a scan (above 16,384 tiles), then the same passes again over the order by whole codes.  And rebuilds, of trees
that met such runs when they were built and of uploaded ones."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from test_gpu_parity import assert_same_bytes, check_build
from test_gpu_rebuild import pick_leaves
from test_gpu_sort_runs import clumps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sp", [(70000, 64), (70000, 128), (300001, 64), (300001, 128), (4194400, 64)])
def test_builds(ctx, n, sp):
    check_build(ctx, clumps(n, 100, 1.0, seed=n), 14, 0, 3, sp)


@pytest.mark.parametrize("uploaded", [False, True])
@pytest.mark.parametrize("n,frac,sp", [(1500, 0.4, 64), (9000, 0.3, 128), (60000, 0.5, 64), (400000, 0.9, 64)])
def test_rebuilds(ctx, n, frac, sp, uploaded):
    tris = clumps(n, 200, 1.0, seed=n)
    bvh = ob.PlocBuilder(ctx).build(14, tris, None, ob.SortPrecision(sp))
    nodes = bvh.nodes
    if uploaded:
        bvh = ob.Bvh2.from_host(ctx, nodes, bvh.primitive_indices)
    flags = ob.compute_rebuild_path_flags(bvh, pick_leaves(nodes, frac, seed=n))
    ob.PlocBuilder(ctx).partial_rebuild(bvh, flags, 14, ob.SortPrecision(sp))
    rc, want, _ = O.partial_rebuild(nodes, flags.to_host(), 14, 0, sort_precision=sp)
    assert rc == 0
    assert_same_bytes(bvh.nodes, want, "partial rebuild")
    ob.PlocBuilder(ctx).full_rebuild(bvh, 6, ob.SortPrecision(sp))
    rc, want, _ = O.full_rebuild(want, 6, 0, sort_precision=sp)
    assert rc == 0
    assert_same_bytes(bvh.nodes, want, "full rebuild")
