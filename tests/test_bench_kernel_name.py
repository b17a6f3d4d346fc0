"""The benchmark names the kernel form that a launch of its rays takes: below 16 rows of 64 rays per compute unit one
lane per ray in k_traverse, k_traverse_chunk from there on."""
import importlib.util
import os

import pytest

import obvhs_amd as ob

spec = importlib.util.spec_from_file_location(
    "bench", os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bench.py"))
bench = importlib.util.module_from_spec(spec)
spec.loader.exec_module(bench)


class Table:
    def tune_table(self):
        return {"trav_lds_depth": [4, 8, 16, 8], "trav_chunk": [0, 1, 0, 1]}


@pytest.mark.parametrize("n_prims,n_rays,want", [
    (100, 262080, "k_traverse<closest, lds 4>"), (100, 262081, "k_traverse_chunk<closest, lds 4>"),
    (5000, 65536, "k_traverse<closest, lds 8>"), (100000, 1 << 22, "k_traverse_chunk<closest, lds 16>")])
def test_names(n_prims, n_rays, want):
    assert bench.kernel_name(Table(), ob, n_prims, n_rays) == want
