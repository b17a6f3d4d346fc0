"""The sort tuner times what the builds run: sorts of 32-bit keys, which have no tiles up to 8,192 keys."""
import pytest

import obvhs_amd as ob

pytestmark = pytest.mark.gpu


def test_no_tiles_nothing_to_choose():
    with ob.Context(0) as ctx:
        for n in (1, 4095, 4096, 8192):
            for items in (4, 8, 16):
                table = dict(ctx.tune_table(), sort_items=[items] * 4)
                ctx.set_tune_table(table)
                assert ob.tune_sort(ctx, n) == items
                assert ctx.tune_table() == table


@pytest.mark.parametrize("n", [8193, 300000, 2000000])
def test_choice_is_stored(n):
    with ob.Context(0) as ctx:
        items = ob.tune_sort(ctx, n)
        assert items in (4, 8, 16)
        want = [8] * 4
        want[ob.size_class(n)] = items
        assert ctx.tune_table()["sort_items"] == want
