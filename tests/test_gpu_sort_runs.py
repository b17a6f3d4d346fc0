"""Builds whose Morton codes share their top 32 bits in runs: the sort by the tops orders each run where the leaves are
gathered, and long runs send the build to the sort of the whole codes.  Codes, permutation, nodes and CWBVH equal the
oracle's for run lengths around the limit (64), runs across tile edges (256), equal codes, and the one-workgroup front
(at most 2,048 leaves)."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd.types import triangles_from_vertices
from test_gpu_parity import assert_same_bytes, check_build

pytestmark = pytest.mark.gpu


def clumps(n, run, spread, seed):
    """n small triangles in the unit cube (two of them at its corners): groups of `run` triangles inside a cell of the
    codes' top bits (2^-14 wide at most), `spread` of that cell apart (0: identical triangles)."""
    rng = np.random.default_rng(seed)
    groups = -(-n // run)
    cell = (rng.integers(0, 1 << 10, (groups, 3)) + 0.25) / 1024.0
    at = np.repeat(cell, run, axis=0)[:n]
    at = at + spread * 2.0 ** -14 * rng.random((n, 3))
    off = 1e-7 * rng.random((n, 3, 3)) * (1.0 if spread else 0.0)
    v = at[:, None, :] + off
    v[0], v[1] = 0.0, 1.0
    v = v[rng.permutation(n)].astype(np.float32)
    return triangles_from_vertices(v[:, 0], v[:, 1], v[:, 2])


def check(ctx, tris, spread, sp):
    if spread:
        check_build(ctx, tris, 14, 0, 3, sp)
        return
    # identical triangles merge into chains deeper than a CWBVH may be: codes, permutation and BVH2 only
    ref = O.ploc_build(O.tri_aabbs(tris), 14, 0, sort_precision=sp)
    bvh2 = ob.PlocBuilder(ctx).build(14, tris, None, ob.SortPrecision(sp), 0)
    codes, order = bvh2.sort_trace()
    np.testing.assert_array_equal(codes, ref["codes"])
    np.testing.assert_array_equal(order, ref["sorted_index"])
    assert_same_bytes(bvh2.nodes, ref["nodes"], "BVH2 nodes")


@pytest.mark.parametrize("sp", [64, 128])
@pytest.mark.parametrize("n,run,spread", [(2049, 2, 1.0), (5000, 33, 1.0), (5000, 63, 1.0), (5120, 64, 1.0),
                                          (5001, 65, 1.0), (4097, 4097, 1.0), (3000, 40, 0.0), (3000, 3000, 0.0)])
def test_runs(ctx, n, run, spread, sp):
    check(ctx, clumps(n, run, spread, seed=n + run), spread, sp)


@pytest.mark.parametrize("sp", [64, 128])
@pytest.mark.parametrize("n,run,spread", [(64, 3, 1.0), (65, 65, 1.0), (1023, 7, 1.0), (1025, 300, 1.0),
                                          (2048, 2048, 1.0), (2047, 5, 0.0), (2048, 2048, 0.0)])
def test_small_front(ctx, n, run, spread, sp):
    check(ctx, clumps(n, run, spread, seed=n + run), spread, sp)
