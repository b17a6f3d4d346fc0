"""The tail of a batched build by the size of the meshes: workgroups for 128, 512 and 1,024 clusters, with a launch of
its own for a class of many meshes beside larger ones.  Every mesh checked equals the oracle's build of it alone."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes

pytestmark = pytest.mark.gpu


def check(ctx, counts, sd, picks):
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    tris = scenes.soup(int(offsets[-1]), seed=int(offsets[-1]) + sd)
    batch = ob.build_cwbvh_batch(ctx, tris, offsets, ob.BvhBuildParams(ploc_search_distance=sd, max_prims_per_leaf=3))
    nodes, prims = batch.all_nodes(), batch.all_primitive_indices()
    for i in picks:
        no, nc, po, pc = batch.mesh_info(i)
        _, rcw, rprims = O.build_cwbvh(tris[offsets[i]:offsets[i + 1]], sd, 0, 3)
        assert nodes[no:no + nc].tobytes() == rcw.tobytes(), f"mesh {i} of {counts[i]} triangles"
        np.testing.assert_array_equal(prims[po:po + pc], rprims)


@pytest.mark.parametrize("sd", [1, 2, 14, 32])
def test_sizes(ctx, sd):
    for n in (1, 63, 64, 65, 127, 128, 129, 255, 511, 512, 513, 1023, 1024):
        check(ctx, [n] * 5, sd, range(5))


@pytest.mark.parametrize("small,middle,large", [(4095, 3, [1]), (4096, 3, []), (4097, 4096, [1024]),
                                                (4100, 4200, [5000]), (100, 4200, [600]), (5000, 0, [3000])])
def test_mixed(ctx, small, middle, large):
    rng = np.random.default_rng(small + middle)
    counts = np.concatenate([rng.integers(0, 7, small - 2), [128, 127], rng.integers(129, 140, max(middle - 2, 0)),
                             [129, 512][:middle], large]).astype(np.int64)
    order = rng.permutation(len(counts))
    counts = counts[order]
    big = np.argsort(counts, kind="stable")
    check(ctx, counts, 14, list(big[-6:]) + list(big[::max(1, len(big) // 12)]))
