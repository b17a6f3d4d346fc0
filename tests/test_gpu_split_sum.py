"""Pre-splits of triangle counts around the running sum's head (4,096 elements), its tiles of 4,096 and its span (65,536):
split boxes and indices equal the oracle's, whose thresholds come from the sum in order."""
import numpy as np
import pytest

import obvhs_amd as ob
import oracle_lib as O
from obvhs_amd import scenes
from test_gpu_parity import assert_same_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 5, 4095, 4096, 4097, 8192, 8193, 65535, 65536, 65537, 140001])
def test_sum_edges(ctx, n):
    tris = scenes.soup(n, seed=n)
    aabbs, idx = ob.split_aabbs_preset(ctx, tris, 0)
    ra, ri, _, _ = O.presplit(tris, 0)
    assert_same_bytes(aabbs, ra, "split boxes")
    np.testing.assert_array_equal(idx, ri)


def test_equal_triangles(ctx):
    """Equal half areas: ties in plenty."""
    tris = np.repeat(scenes.soup(1, seed=4), 70000)
    tris["v0"][:, 0] += np.arange(70000, dtype=np.float32) % 7
    aabbs, idx = ob.split_aabbs_preset(ctx, tris, 0)
    ra, ri, _, _ = O.presplit(tris, 0)
    assert_same_bytes(aabbs, ra, "split boxes")
    np.testing.assert_array_equal(idx, ri)
