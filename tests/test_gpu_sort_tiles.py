"""Builds around the number of sort tiles (64 of 2,048 keys) up to which a sort pass has no scan launch."""
import pytest

from obvhs_amd import scenes
from test_gpu_parity import check_build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2049, 4097, 131072, 131073, 133121])
def test_tiles(ctx, n):
    check_build(ctx, scenes.soup(n, seed=n), 14, 0, 3, 64)
