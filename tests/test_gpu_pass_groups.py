"""PLOC passes of more than 1,024 tiles of 256 clusters: search and compaction as launches of their own, a tile's place
from sums over groups of tiles up to 16,384 tiles and from a scan above.  Trees equal the oracle's."""
import pytest

from obvhs_amd import scenes
from test_gpu_parity import check_build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sd,sdt", [(1, 0), (2, 0), (32, 2)])
def test_tile_merges(ctx, sd, sdt):
    """Distance-1 passes merge up to half of a tile's clusters: every wave of a tile has table entries to write."""
    check_build(ctx, scenes.soup(300001, seed=sd), sd, sdt, 3, 64)


@pytest.mark.parametrize("n", [4194304, 4194305])
def test_group_limit(ctx, n):
    """16,384 tiles and one more: the first passes go by group sums, or by the scan and later ones by sums."""
    check_build(ctx, scenes.soup(n, seed=n), 14, 0, 3, 64)
