"""Pre-splits of triangles whose areas grow along the array: the running sum leaves its binade every few thousand
elements to the end, so it goes serially in small tiles, in large ones, or in passes by the distance of the stops.
Split boxes and indices equal the oracle's, whose thresholds come from the sum in order."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd.types import triangles_from_vertices
from test_gpu_parity import assert_same_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,octaves", [(150000, 75), (200000, 20), (400000, 30), (400000, 13), (600001, 10),
                                       (600001, 0)])
def test_growing_areas(ctx, n, octaves):
    rng = np.random.default_rng(n + octaves)
    size = 1e-4 * np.exp2(np.arange(n) * (octaves / 2 / n))
    v = (size[:, None, None] * rng.random((n, 3, 3))).astype(np.float32)
    tris = triangles_from_vertices(v[:, 0], v[:, 1], v[:, 2])
    aabbs, idx = ob.split_aabbs_preset(ctx, tris, 0)
    ra, ri, _, _ = O.presplit(tris, 0)
    assert_same_bytes(aabbs, ra, "split boxes")
    np.testing.assert_array_equal(idx, ri)
