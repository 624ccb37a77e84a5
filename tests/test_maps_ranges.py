"""Into how many ranges of keys the units of mapped attention are cut, and the results at the edges of that rule."""
import pytest
import torch

import tabupel_mechanisms as mech


def ranges(units, heads, kv_heads, maps, values, keys, tokens=1, window=0):
    from simply_amd.kernels import lib
    return lib.load().sa_paged_attention_maps_ranges(units, heads, kv_heads, maps, values, window, keys, tokens)


def test_a_workgroup_for_each_tile_where_it_is_ahead():
    # (n keys lie in at most (n + 31) // 32 + 1 tiles)
    assert [ranges(1, 16, 1, 1, 512, n) for n in (64, 96, 217, 1024, 1025)] == [2, 4, 8, 33, 17]
    assert [ranges(8, 16, 1, 1, 512, n) for n in (217, 960, 1024)] == [8, 31, 17]       # 256 CUs
    assert [ranges(1, 16, 1, 1, 512, n) for n in (2048, 4096, 8000)] == [33, 64, 64]     # one request with a long context
    assert [ranges(1, 4, 1, 1, 256, n) for n in (1024, 2016, 2048)] == [33, 64, 33]      # units of four rows
    # the merge that walks the ranges of 16 rows one by one: as before, beyond its 64 ranges a tile each
    assert [ranges(1, 16, 1, 1, 256, n) for n in (217, 1024, 2048, 4096)] == [4, 17, 65, 129]
    # two maps: as before at every length
    assert [ranges(1, 8, 1, 2, 128, n) for n in (217, 1024, 2048, 3000)] == [4, 17, 33, 48]
    # a window bounds the tiles
    assert ranges(1, 16, 1, 1, 512, 8000, window=1000) == ranges(1, 16, 1, 1, 512, 1000)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,differential,n", [((16, 1, 64, 272), False, 500), ((16, 1, 64, 272), False, 1030), ((4, 1, 64, 256), False, 2000),
                                                  ((16, 1, 64, 64), False, 2100), ((16, 1, 64, 64), False, 2040), ((8, 1, 64, 128), True, 2100)])
def test_one_request_at_the_edges_of_the_rule(gpu_lib, sizes, differential, n):
    from simply_amd.kernels import ops
    mech.attention_units_on_the_matrix_cores(ops, "cuda", sizes=sizes, differential=differential, n=n)
