"""Batched builds where the sort changes form: runs of equal sort keys around the limit of the ranking (64) and a mesh
too large for the 32-bit keys.  Every mesh's CWBVH equals the oracle's build of that mesh alone."""
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
