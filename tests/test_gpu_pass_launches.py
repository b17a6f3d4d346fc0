"""Builds where a PLOC pass changes form: one launch per pass up to 1,024 tiles of 256 clusters, tile edges, and the
one-workgroup tail's steps (2,048 clusters, two clusters per thread above 1,024, two and four lanes per cluster below 512
and 256, one wave below 64), for every search distance and with the distance-1 passes first.  And CWBVHs deeper than the
21 levels whose node bound (8 per level) fits 64 bits.  Nodes equal the oracle's."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from test_gpu_parity import assert_same_bytes, check_build
from test_gpu_sort_runs import clumps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 17, 32, 33, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048])
@pytest.mark.parametrize("sd", [1, 2, 14, 32])
def test_tail(ctx, n, sd):
    check_build(ctx, scenes.soup(n, seed=n), sd, 0, 3, 64)


@pytest.mark.parametrize("sd,sdt", [(1, 0), (2, 0), (6, 3), (14, 0), (14, 2), (24, 0), (32, 1)])
@pytest.mark.parametrize("n", [2049, 2304, 2305, 10000])
def test_passes(ctx, n, sd, sdt):
    check_build(ctx, scenes.soup(n, seed=n + sd), sd, sdt, 3, 64)


@pytest.mark.parametrize("n", [262144, 262145])
def test_pass_limit(ctx, n):
    check_build(ctx, scenes.soup(n, seed=n), 14, 0, 3, 64)


@pytest.mark.parametrize("run", [25, 40])
def test_deep_conversion(ctx, run):
    """Clumps of identical triangles merge into chains: more levels than an evenly filled CWBVH has."""
    tris = clumps(1200, run, 0.0, seed=run)
    ref = O.ploc_build(O.tri_aabbs(tris), 14, 0)
    bvh = ob.PlocBuilder(ctx).build(14, tris)
    assert_same_bytes(bvh.nodes, ref["nodes"], "BVH2")
    rcw, rprims, _ = O.bvh2_to_cwbvh(ref["nodes"], ref["prim_indices"], 3, True)
    cw = ob.bvh2_to_cwbvh(bvh, 3, True, False)
    assert_same_bytes(cw.nodes, rcw, "CWBVH")
    np.testing.assert_array_equal(cw.primitive_indices, rprims)
