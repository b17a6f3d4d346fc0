"""Batched builds where the sort and the last passes change form: runs of equal sort keys around the limit of the
ranking (64), a mesh too large for the 32-bit keys, and meshes of cluster counts around the steps of the one-workgroup
passes (1,024 clusters at most, several lanes per cluster below 256 and 128, one wave below 64).  Every mesh's CWBVH
equals the oracle's build of that mesh alone."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from test_gpu_batch import assert_same_bytes, check_batch_build, concat, mesh_slices
from test_gpu_sort_runs import clumps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("run", [2, 33, 63, 64, 65, 300])
def test_runs(ctx, run):
    """Three meshes: 30 bits of the code beside 2 of the mesh number; the clumps share them."""
    check_batch_build(ctx, [clumps(3000, run, 1.0, seed=run), scenes.soup(700, seed=run), clumps(259, run, 1.0, seed=9)])


@pytest.mark.parametrize("size", [6501, 6502])
def test_many_meshes_one_large(ctx, size):
    """65,536 meshes leave 16 bits for the code: 4 * 2^(32/3) = 6,501 triangles are the most a mesh may have then."""
    meshes = [np.zeros(0, dtype=ob.TRIANGLE)] * 65536
    full = {0: scenes.soup(40, seed=1), 40000: scenes.soup(size, seed=2), 65535: scenes.soup(1300, seed=3)}
    for i, m in full.items():
        meshes[i] = m
    tris, offsets = concat(meshes)
    params = ob.BvhBuildParams(ploc_search_distance=14, max_prims_per_leaf=3)
    batch = ob.build_cwbvh_batch(ctx, tris, offsets, params)
    nodes, prims = batch.all_nodes(), batch.all_primitive_indices()
    for i, m in full.items():
        n_i, p_i = mesh_slices(batch, nodes, prims, i)
        _, rcw, rprims = O.build_cwbvh(m, 14, 0, 3)
        assert_same_bytes(n_i, rcw, f"mesh {i} nodes")
        np.testing.assert_array_equal(p_i, rprims)


EDGES = [1, 2, 3, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024]


@pytest.mark.parametrize("more", [[], [1025, 2500]])
@pytest.mark.parametrize("sd,sdt", [(1, 0), (2, 0), (6, 0), (14, 0), (14, 3), (24, 2), (32, 0)])
def test_tail_edges(ctx, sd, sdt, more):
    check_batch_build(ctx, [scenes.soup(n, seed=n) for n in EDGES + more], sd, sdt, 3)
