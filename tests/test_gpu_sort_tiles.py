"""Builds around the sizes where the sort changes form: one workgroup up to 8,192 keys, no scan launch up to 64 tiles of
2,048 keys."""
import pytest

from obvhs_amd import scenes
from test_gpu_parity import check_build
from test_gpu_sort_runs import clumps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2049, 4097, 131072, 131073, 133121])
def test_tiles(ctx, n):
    check_build(ctx, scenes.soup(n, seed=n), 14, 0, 3, 64)


@pytest.mark.parametrize("n", [2050, 4095, 4096, 8191, 8192, 8193])
def test_one_workgroup(ctx, n):
    """Up to 8,192 keys the sort is one launch of 2, 4 or 8 keys per thread."""
    check_build(ctx, scenes.soup(n, seed=n), 14, 0, 3, 64)
    check_build(ctx, clumps(n, 50, 1.0, seed=n), 14, 0, 3, 64)
