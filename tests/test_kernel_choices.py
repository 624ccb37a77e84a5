"""Which kernel of the library takes a call: its host functions, which need the built library and no GPU."""
import pytest

from simply_amd.kernels import build


@pytest.fixture(scope="module")
def lib():
    if build.find_library() is None:
        pytest.skip("the kernel library has not been built here")
    from simply_amd.kernels import lib
    return lib.load()


def test_32_bit_attention_of_long_contexts_keeps_its_ranges(lib):
    """Partial results of a range: its chunks' where there are few, the range's own where those are many or the workspace does not hold
    the chunks', and none only where the units fill the chip or the workspace does not hold a part for every range."""
    from simply_amd.kernels import ops

    parts = ops.attention_f32_parts
    assert parts(4, 4, 256, None, 1023, 1) == 4 and parts(1, 4, 256, None, 8192, 1) == 4 and parts(8, 4, 256, None, 1024, 1) == 4
    assert parts(1, 4, 256, None, 8193, 1) == 1 and parts(16, 4, 256, None, 2048, 1) == 1 and parts(1, 16, 128, None, 4096, 1) == 1
    # 4,097 keys and more of 32 requests, planned for 8,192; two of 131,072 (14.6 ms a launch walked, 0.7 in ranges); a long portion
    assert parts(32, 4, 256, None, 8192, 1) == 1 and parts(2, 4, 256, None, 131072, 1) == 1 and parts(32, 4, 256, None, 16640, 8) == 1
    # a window bounds them
    assert parts(4, 4, 256, 1024, 100000, 1) == 4 and parts(16, 4, 256, 1024, 100000, 1) == 1
    assert parts(64, 4, 256, None, 4096, 1) == 0 and parts(4, 4, 256, None, 256, 1) == 0
    row = 16 * (256 + 4) * 4
    assert [parts(2, 4, 256, None, 2048, 1, n * 8 * 8 * row) for n in (0, 1, 3, 4)] == [0, 1, 1, 4]
    assert parts(2, 4, 256, None, 2048, 1, 8 * 8 * row - 1) == 0


def test_32_bit_attention_of_prompts_fills_the_chip(lib):
    """Units of several tokens: a part for each chunk of short prompts, for each range of longer ones; walked where one range is all there
    is of many units, or the workspace holds no part for every range."""
    from simply_amd.kernels import ops

    parts = ops.attention_f32_parts
    assert parts(8, 4, 256, None, 64, 8) == 4 and parts(64, 4, 256, None, 509, 8) == 4 and parts(88, 4, 256, None, 700, 8) == 4
    assert parts(128, 4, 256, None, 1024, 8) == 1 and parts(64, 4, 256, None, 2557, 8) == 1 and parts(256, 4, 256, None, 2048, 8) == 1
    assert parts(32, 16, 128, None, 256, 8) == 0 and parts(64, 16, 128, None, 512, 8) == 1 and parts(8, 4, 64, None, 128, 8) == 4
    row = 16 * (256 + 4) * 4
    assert [parts(64, 4, 256, None, 509, 8, n * 512 * row) for n in (0, 1, 3, 4)] == [0, 1, 1, 4]


def test_32_bit_attention_of_few_tokens_behind_many_goes_by_ranges(lib):
    """A few units that see many ranges: a part for each chunk would leave the merge four times as many to walk through."""
    from simply_amd.kernels import ops

    parts = ops.attention_f32_parts
    assert parts(3, 4, 256, None, 8017, 8) == 1 and parts(1, 4, 256, None, 30005, 5) == 1 and parts(13, 4, 256, None, 2100, 8) == 1
    assert parts(1, 8, 128, None, 8005, 5) == 1 and parts(1, 1, 128, None, 30005, 5) == 1
    assert parts(8, 4, 256, None, 1088, 8) == 4 and parts(1, 4, 256, None, 4000, 5) == 4 and parts(16, 4, 64, None, 305, 5) == 4


def test_32_bit_products_of_narrow_weights_and_few_rows_take_small_tiles(lib):
    """(M, N, K, gated): where larger tiles took up to twice as long, and the sizes beside them that stay with those."""
    from simply_amd.kernels import ops

    def tile(M, N, K, gated=False):
        return (*ops.gemm_f32_tile(M, N, K, gated=gated), ops.gemm_f32_plan(M, N, K, gated=gated)[1])

    assert tile(1024, 512, 256) == tile(509, 512, 256) == tile(300, 1024, 256, True) == tile(1024, 1024, 1024) == (64, 64, False)
    assert tile(61, 1024, 4096) == tile(100, 512, 256) == tile(61, 1152, 6912) == (64, 64, True)
    assert tile(130, 4096, 512) == tile(256, 2048, 512, True) == tile(130, 3584, 736) == tile(100, 1570, 256, True) == (64, 64, False)
    assert tile(700, 4096, 512) == (128, 128, False) and tile(130, 3840, 1024)[:2] == (128, 256)
    assert tile(17, 9216, 2304, True) == tile(32, 14336, 3584, True) == (32, 128, True)
    assert tile(17, 2048, 1024) == tile(32, 8192, 3584) == (32, 64, True)
    assert tile(33, 9216, 2304, True) == (64, 128, True) and tile(509, 2304, 9216) == (128, 288, True)
    assert tile(509, 9216, 2304, True) == (128, 256, True) and tile(17, 36864, 4608, True)[:2] == (64, 128)


@pytest.mark.parametrize("M,N,K,gated,shape", [
    (2048, 1024, 4096, 0, 4128128), (2048, 2048, 2048, 0, 4128128), (1537, 2048, 8192, 0, 4128128), (4096, 1024, 1024, 0, 4128128),
    (2048, 2304, 2304, 0, 3192128), (1664, 4992, 2048, 0, 4128128), (1664, 5120, 2048, 0, 2256192),
    (129, 512, 1024, 1, 4128128), (300, 2048, 2048, 1, 4128128), (256, 8192, 2048, 1, 4128128), (384, 8192, 2048, 1, 3192128),
    (1025, 2048, 1024, 1, 3192128), (2048, 9216, 2304, 1, 2128192), (128, 8192, 2048, 1, 3128128)])
def test_wide_tiles_of_128_by_128_where_one_round_is_enough(lib, M, N, K, gated, shape):
    """One round of them in place of one of 192 x 128, or two for one of 256 x 192."""
    assert lib.sa_gemm_wide_shape(M, N, K, gated, 256 << 20) == shape


@pytest.mark.parametrize("which", ["q", "rows", "weight", "k_pages", "v_pages"])
def test_latent_rows_look_at_every_buffer_s_alignment(lib, which):
    """Pieces of 16 bytes are read and written at all five: a view that begins elsewhere goes the way of single entries."""
    base = dict(q=4096, rows=8192, weight=12288, k_pages=16384, v_pages=20480)
    takes = lambda **at: lib.sa_latent_rows_takes(16, 512, 64, 64, 16, 16 * 576, 576, *{**base, **at}.values())
    assert takes() and takes(**{which: base[which] + 16}) and not takes(**{which: base[which] + 2}) and not takes(**{which: base[which] + 8})


@pytest.mark.parametrize("D,F,per,rows", [
    (2048, 2048, 11, 16), (2048, 2048, 59, 64), (2048, 2048, 60, 128), (4096, 3584, 64, 128), (3072, 2048, 96, 128),
    # one product of fewer columns than fill the CUs: 64 rows were ahead by up to a third (1,024 x 8,192: 180 us for 235)
    (1024, 4096, 60, 64), (1024, 4096, 128, 64), (4096, 1024, 96, 64), (3072, 1536, 136, 64), (3072, 1536, 272, 64), (1024, 8192, 60, 64),
    (1024, 4096, 336, 128), (3072, 1536, 336, 128), (1024, 8192, 192, 128), (1024, 1024, 400, 64), (2048, 1536, 256, 64)])
def test_rows_of_a_tile_of_routed_experts(lib, D, F, per, rows):
    assert lib.sa_expert_tile_rows(16 * per, 16, D, F, 1, D, 4096) == rows


@pytest.mark.parametrize("T,D,E,top,pays", [
    (1, 2048, 16, 2, True), (16, 2048, 16, 2, True), (16, 4096, 16, 2, True), (16, 512, 8, 2, True), (4, 2048, 16, 8, True),
    (16, 1024, 16, 4, False), (16, 2048, 16, 8, False), (4, 4096, 32, 4, True), (12, 1024, 32, 4, False), (16, 4096, 32, 8, False),
    (4, 1024, 64, 6, True), (8, 1024, 64, 6, False), (16, 2048, 64, 8, False), (1, 960, 128, 8, True), (8, 960, 128, 8, False)])
def test_router_of_few_tokens_where_it_pays(lib, T, D, E, top, pays):
    """Sizes at which one workgroup or three launches were clearly ahead (128 experts, top 8, 16 tokens: 43 us for 22)."""
    assert bool(lib.sa_route_few_pays(T, D, E, E, top)) == pays


def test_routers_that_do_not_pay_go_the_way_of_many_tokens(lib, monkeypatch):
    """With 128 experts a step of 8 tokens is routed by the product, the choice and the sort."""
    import types

    import torch

    from simply_amd.kernels import ops
    from simply_amd.parts.ffn import RoutedExperts

    part, seen = RoutedExperts(960, 128, 8, 16), []
    part.router = types.SimpleNamespace(rows=128, cols=960)
    monkeypatch.setattr(ops, "route_few_takes", lambda *a: True)
    monkeypatch.setattr(ops, "few_rows_experts", lambda *a: True)
    monkeypatch.setattr(ops, "route_few", lambda *a, **k: seen.append("few") or (torch.zeros(1, 128), None, None, ()))
    monkeypatch.setattr(ops, "gemm", lambda x, w, **k: seen.append("product") or torch.zeros(x.shape[0], 128))
    monkeypatch.setattr(ops, "route", lambda *a: (None, None))
    monkeypatch.setattr(ops, "routed_experts", lambda *a, **k: None)
    monkeypatch.setattr(ops, "expert_sums", lambda *a, **k: types.SimpleNamespace(materialize=lambda: None))
    for tokens in (1, 8):
        part.forward(torch.zeros(tokens, 960))
    assert seen == ["few", "product"]


@pytest.mark.parametrize("D,top,pays", [(512, 16, True), (2048, 8, True), (2048, 17, False), (4096, 8, True), (4096, 16, False), (8192, 2, True),
                                        (8192, 4, False), (8192, 16, False)])
def test_sums_over_experts_in_the_norm_where_they_pay(lib, D, top, pays):
    """One workgroup a token for all of its experts' rows, or a sum's kernel with one for each 2,048 entries (8,192, top 16: 15.8 us for 6.6)."""
    assert bool(lib.sa_experts_add_next_norm_pays(D, top)) == pays
