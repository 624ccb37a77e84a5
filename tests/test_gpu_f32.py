"""The 32-bit path's own kernels against 64-bit references, at the edges of their tiles and of their ways of cutting the
work."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def draw(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).cuda()


@pytest.mark.parametrize("N,K", [(16, 4), (7, 32), (100, 36), (130, 256), (333, 260), (96, 2304), (2304, 100)])
def test_products(N, K):
    """Few rows and tiles of 64 rows, whole and cut over K, plain, gated and soft-capped: each within the bound on a sum of K products in
    any order, (K + 2) eps sum |a| |w|; and a row's result is the same to the bit whichever of the ways it went."""
    from simply_amd.kernels import ops

    a, w, w2 = draw((200, K), 1), draw((N, K), 2, 0.1), draw((N, K), 3, 0.1)
    want = a.double() @ w.double().T
    bound = (K + 2) * EPS * (a.double().abs() @ w.double().abs().T)
    gate_want = torch.nn.functional.silu(want) * (a.double() @ w2.double().T)
    # silu's slope is at most 1.1, |silu(x)| <= |x|; its own rounding: a few steps of the result
    gate_bound = 1.1 * bound * (a.double() @ w2.double().T).abs() + want.abs() * (K + 2) * EPS * (a.double().abs() @ w2.double().abs().T) \
        + 8 * EPS * gate_want.abs()
    first = {}
    for M in (1, 4, 8, 9, 16, 17, 64, 65, 128, 200):
        rows = a[200 - M:]
        got = {"plain": ops.gemm(rows, w), "gated": ops.gemm(rows, w, w2=w2, activation=ops.ACT_SILU),
               "capped": ops.gemm(rows, w, soft_cap=2.0)}
        assert ((got["plain"].double() - want[200 - M:]).abs() <= bound[200 - M:]).all(), M
        assert ((got["gated"].double() - gate_want[200 - M:]).abs() <= gate_bound[200 - M:]).all(), M
        assert ((got["capped"].double() - 2.0 * torch.tanh(want[200 - M:] / 2.0)).abs() <= bound[200 - M:] + 8 * EPS * 2.0).all(), M
        for k, v in got.items():
            first.setdefault(k, v[-1])
            assert torch.equal(v[-1], first[k]), (k, M)
    # rows of a wider buffer, and a result that is one
    wide, out = draw((20, K + 24), 4), torch.zeros(20, N + 3, device="cuda")
    got = ops.gemm(wide[:, 8:8 + K], w, out=out[:, :N])
    assert torch.equal(got, ops.gemm(wide[:, 8:8 + K].contiguous(), w)) and not out[:, N:].any()


@pytest.mark.parametrize("M,N,K,gated,cut", [(1000, 3135, 260, False, False), (1000, 1570, 260, True, False),
                                             (333, 1101, 1028, False, True), (333, 1100, 1028, False, True),
                                             (333, 581, 1028, True, True), (333, 580, 1028, True, True)])
def test_products_in_tiles_of_128_rows(M, N, K, gated, cut):
    """Tiles of 128 rows, whole and cut over K, the last rows and columns of their tiles missing, segments that end in the
    middle of a stage of 32 columns (48 and 144 columns long): bounds as above, and the bits of the kernel for few rows."""
    from simply_amd.kernels import ops

    assert ops.gemm_f32_plan(M, N, K, gated=gated) == (128, cut) and ops.gemm_f32_plan(5, N, K, gated=gated) == (16, False)
    a, w, w2 = draw((M, K), 11), draw((N, K), 12, 0.1), draw((N, K), 13, 0.1)
    kw = dict(w2=w2, activation=ops.ACT_SILU) if gated else {}
    got = ops.gemm(a, w, **kw)
    x, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = (K + 2) * EPS * size
    if gated:
        up, up_bound = a.double() @ w2.double().T, (K + 2) * EPS * (a.double().abs() @ w2.double().abs().T)
        want = torch.nn.functional.silu(x) * up
        bound = 1.1 * bound * up.abs() + x.abs() * up_bound + 8 * EPS * want.abs()
    else:
        want = x
    assert ((got.double() - want).abs() <= bound).all()
    for rows in (slice(0, 5), slice(126, 131), slice(M - 5, M)):
        assert torch.equal(ops.gemm(a[rows], w, **kw), got[rows])
    if not gated:
        capped = ops.gemm(a, w, soft_cap=2.0)
        assert ((capped.double() - 2.0 * torch.tanh(want / 2.0)).abs() <= bound + 8 * EPS * 2.0).all()
        assert torch.equal(ops.gemm(a[M - 5:], w, soft_cap=2.0), capped[M - 5:])


@pytest.mark.parametrize("M,N,K,gated,tile,cut", [
    (70, 130, 48, False, (64, 64), False), (333, 581, 272, True, (64, 64), False), (130, 300, 1040, False, (64, 64), True),
    (700, 1500, 272, False, (128, 64), False), (700, 760, 272, True, (128, 64), False), (200, 701, 528, False, (128, 64), True),
    (1500, 2000, 16, False, (128, 96), False), (300, 8003, 80, False, (128, 96), False), (300, 4010, 80, True, (128, 96), False),
    (509, 2300, 2064, False, (128, 96), True), (1000, 3135, 272, False, (128, 128), False), (1000, 1570, 272, True, (128, 128), False)])
def test_products_of_whole_blocks(M, N, K, gated, tile, cut):
    """K in blocks of 16, through the tiles that hold their operands ahead of the products: the last rows and columns missing, a
    last stage of one block, one block in all, segments that end inside a stage.  Bounds as above, the bits of the kernel for few
    rows, and the same from rows of a wider buffer."""
    from simply_amd.kernels import ops

    assert ops.gemm_f32_tile(M, N, K, gated=gated) == tile and ops.gemm_f32_plan(M, N, K, gated=gated) == (tile[0], cut)
    wide, w, w2 = draw((M, K + 12), 21), draw((N, K), 22, 0.1), draw((N, K), 23, 0.1)
    a = wide[:, 8:8 + K]
    kw = dict(w2=w2, activation=ops.ACT_SILU) if gated else {}
    got = ops.gemm(a, w, **kw)
    x, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = (K + 2) * EPS * size
    if gated:
        up, up_bound = a.double() @ w2.double().T, (K + 2) * EPS * (a.double().abs() @ w2.double().abs().T)
        want = torch.nn.functional.silu(x) * up
        bound = 1.1 * bound * up.abs() + x.abs() * up_bound + 8 * EPS * want.abs()
    else:
        want = x
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(ops.gemm(a.contiguous(), w, **kw), got)
    for rows in (slice(0, 5), slice(62, 67), slice(M - 5, M)):
        assert torch.equal(ops.gemm(a[rows], w, **kw), got[rows])


@pytest.mark.parametrize("M,N,K,gated,tile,cut", [
    (17, 1570, 256, True, (64, 128), True), (17, 18433, 160, False, (64, 128), False), (17, 9200, 160, True, (64, 128), False),
    (65, 18433, 160, False, (128, 64), True), (17, 2300, 160, True, (128, 64), False), (257, 8003, 160, False, (128, 128), False),
    (65, 18433, 992, True, (128, 128), True), (200, 18433, 160, False, (128, 192), False), (65, 4100, 992, False, (128, 192), True),
    (130, 3135, 992, False, (128, 256), True), (257, 18433, 160, False, (128, 256), False), (130, 18433, 992, True, (128, 256), True),
    (130, 4100, 992, False, (128, 288), True), (1000, 9200, 160, False, (128, 288), False), (1000, 4100, 160, True, (128, 288), False)])
def test_products_of_parts(M, N, K, gated, tile, cut):
    """K in segments of whole stages of 32 columns (the last one shorter at 992), the products those of bfloat16 parts: every tile, whole,
    cut, and cut behind 256 whole ones, the last rows and columns missing, rows and weights of very different sizes: the bounds of a sum
    in 32 bits, and the bits of the kernel for few rows.  (That all 24 bits of every number count is the next tests' matter: two of three
    parts would stay within these bounds.)"""
    from simply_amd.kernels import ops

    assert ops.gemm_f32_tile(M, N, K, gated=gated) == tile and ops.gemm_f32_plan(M, N, K, gated=gated) == (tile[0], cut)
    wide, w, w2 = draw((M, K + 12), 31), draw((N, K), 32, 0.1), draw((N, K), 33, 0.1)
    a = wide[:, 8:8 + K]
    a[::3] *= 2.0 ** 40
    a[1::3, ::2] *= 2.0 ** -30
    w[::5] *= 2.0 ** -45
    kw = dict(w2=w2, activation=ops.ACT_SILU) if gated else {}
    got = ops.gemm(a, w, **kw)
    x, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = (K + 2) * EPS * size
    if gated:
        up, up_bound = a.double() @ w2.double().T, (K + 2) * EPS * (a.double().abs() @ w2.double().abs().T)
        want = torch.nn.functional.silu(x) * up
        bound = 1.1 * bound * up.abs() + x.abs() * up_bound + 8 * EPS * want.abs()
    else:
        want = x
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(ops.gemm(a.contiguous(), w, **kw), got)
    for rows in (slice(0, 5), slice(0, 16), slice(M // 2, M // 2 + 5), slice(M - 5, M)):
        assert torch.equal(ops.gemm(a[rows], w, **kw), got[rows])
    if not gated:
        capped = ops.gemm(a, w, soft_cap=2.0)
        assert ((capped.double() - 2.0 * torch.tanh(want / 2.0)).abs() <= bound + 8 * EPS * 2.0).all()
        assert torch.equal(ops.gemm(a[M - 5:], w, soft_cap=2.0), capped[M - 5:])


@pytest.mark.parametrize("M,N,K,gated,tile,cut", [
    (33, 1001, 992, False, (64, 64), True), (130, 1000, 160, False, (64, 64), True), (40, 520, 992, True, (64, 64), True),
    (700, 1003, 992, False, (64, 64), False), (300, 1003, 992, True, (64, 64), False), (500, 1530, 160, True, (64, 64), False),
    (17, 1001, 992, False, (32, 64), True), (20, 4100, 992, True, (32, 64), True), (20, 500, 160, False, (32, 64), True),
    (31, 18433, 992, False, (32, 128), True), (20, 9200, 992, True, (32, 128), True)])
def test_products_of_parts_in_small_tiles(M, N, K, gated, tile, cut):
    """Narrow weights and few rows.  A row that holds an infinite entry is done again by such tiles too."""
    from simply_amd.kernels import ops

    test_products_of_parts(M, N, K, gated, tile, cut)
    a, w, w2 = draw((M, K), 34), draw((N, K), 35, 0.1), draw((N, K), 36, 0.1)
    kw = dict(w2=w2, activation=ops.ACT_SILU) if gated else {}
    before = ops.gemm(a, w, **kw)
    a[M - 2, 3] = float("inf")
    got, others = ops.gemm(a, w, **kw), torch.arange(M, device="cuda") != M - 2
    assert torch.equal(got[others], before[others]) and not torch.isfinite(ops.gemm(a, w)[M - 2]).any()
    assert torch.equal(ops.gemm(a[M - 5:], w, **kw).nan_to_num(), got[M - 5:].nan_to_num())


@pytest.mark.parametrize("a_exp,w_exp", [(0, 0), (-60, 70), (-112, 60), (-126, 60), (-140, 100), (60, -116), (90, -126)])
@pytest.mark.parametrize("M,N", [(5, 100), (12, 100), (40, 100), (200, 1000), (300, 4100)])
def test_products_of_parts_keep_every_bit(M, N, a_exp, w_exp):
    """One product for each output, of numbers down to the smallest of 32 bits: all bits of both factors count.  The unit drops what lies
    below the sum's bits (2^-23 of it at most, in the last of the six additions; the others add numbers of 2^-8 and less), the three
    products of parts that are left out are 2^-25 together: 2^-22.  Two parts of three would miss by up to 2^-16, five products of six by
    2^-17 and more.  Rows' bits do not depend on how many there are."""
    from simply_amd.kernels import ops

    K = 256
    columns = torch.randint(0, K, (M,), generator=torch.Generator().manual_seed(41)).cuda()
    scaled = lambda x, e: x * 2.0 ** (e // 2) * 2.0 ** (e - e // 2)
    a, w = torch.zeros((M, K), device="cuda"), scaled(draw((N, K), 42), w_exp)
    a[torch.arange(M, device="cuda"), columns] = scaled(draw((M,), 43), a_exp)
    got = ops.gemm(a, w)
    want = a.double().sum(1)[:, None] * w.double()[:, columns].T
    assert ((got.double() - want).abs() <= 2.0 ** -22 * want.abs() + 2.0 ** -149).all()
    for rows in (slice(0, 5), slice(M - 5, M), slice(0, min(M, 16))):
        assert torch.equal(ops.gemm(a[rows], w), got[rows])


@pytest.mark.parametrize("K", [2304, 9216])
@pytest.mark.parametrize("a_exp,w_exp", [(0, 0), (-120, 60), (60, -120)])
def test_errors_of_products_of_parts(K, a_exp, w_exp):
    """Errors against 64 bits are no larger than the 32-bit unit's, which takes the same rows with 16 columns of zeros behind them."""
    from simply_amd.kernels import ops

    a, w = draw((300, K), 51) * 2.0 ** a_exp, draw((500, K), 52, 0.1) * 2.0 ** w_exp
    want = a.double() @ w.double().T
    error = lambda y, of: (((y.double() - of) ** 2).sum() / (of ** 2).sum()).sqrt().item()
    pad = lambda x: torch.nn.functional.pad(x, (0, 16))
    for M in (4, 12, 300):
        parts, unit = ops.gemm(a[:M], w), ops.gemm(pad(a[:M]), pad(w))
        assert error(parts, want[:M]) <= error(unit, want[:M]), M


@pytest.mark.parametrize("N,rows", [(50, (3, 16, 40, 200)), (4100, (3, 40, 200, 1000))])
def test_products_of_parts_keep_special_values(N, rows):
    """An infinite or undefined entry reaches its own row and column only, as in plain 32-bit arithmetic, and entries next to the
    largest number, whose first part is rounded to an infinite one, give the finite sums that they have."""
    from simply_amd.kernels import ops

    K, largest = 256, torch.finfo(torch.float32).max
    for M in rows:
        a, w, up = draw((M, K), 5), draw((N, K), 6), draw((N, K), 7)
        a[1, 70], a[0, 9], w[7, 3], w[20, 9], up[9, 200] = float("inf"), largest, float("nan"), 0.0, float("-inf")
        a[2, 11], w[20, 11] = -largest, 2.0 ** -20
        got, gated = ops.gemm(a, w), ops.gemm(a, w, w2=up, activation=ops.ACT_SILU)
        assert torch.isnan(got[:, 7]).all() and torch.isnan(gated[:, 7]).all()
        keep = torch.arange(N, device="cuda") != 7
        assert torch.isinf(got[1, keep]).all() and (got[1, keep].sign() == w[keep, 70].sign()).all()
        rest = torch.arange(M, device="cuda") != 1
        want = a[rest].double() @ w[keep].double().T
        size = a[rest].double().abs() @ w[keep].double().abs().T
        y = got[rest][:, keep].double()
        ok = want.abs() < largest / 2
        assert ((y - want).abs()[ok] <= ((K + 2) * EPS * size)[ok]).all()
        assert torch.isfinite(got[0, 20]) and torch.isfinite(got[2, 20])
        # the other factor's column: infinite or, where the gate's factor is zero, undefined
        assert not torch.isfinite(gated[rest][:, 9]).any()
        assert torch.equal(ops.gemm(a[-2:], w)[:, keep], got[-2:, keep])


@pytest.mark.parametrize("M,N,gated", [(5, 100, False), (12, 100, True), (60, 100, True), (200, 4100, False), (300, 4100, True), (600, 2300, False)])
def test_products_of_parts_of_large_numbers(M, N, gated):
    """Entries and sums beyond what scaled parts hold, in some rows, weights and segments: the bound on a sum of K 32-bit products, and
    the bits of rows that are few."""
    from simply_amd.kernels import ops

    K = 992
    a, w, w2 = draw((M, K), 61), draw((N, K), 62, 0.1), draw((N, K), 63, 0.1) * 2.0 ** -100
    a[0] *= 2.0 ** 81
    a[M // 2, 5:9] *= 2.0 ** 110
    a[M - 1, 700] = 2.0 ** 126
    w[N - 2] *= 2.0 ** 30
    w[3, 980:] *= 2.0 ** 100
    a[:, 980:] *= 2.0 ** -20
    kw = dict(w2=w2, activation=ops.ACT_SILU) if gated else {}
    got, largest = ops.gemm(a, w, **kw), torch.finfo(torch.float32).max
    x, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    want, bound = x, (K + 2) * EPS * size
    if gated:
        up, up_bound = a.double() @ w2.double().T, (K + 2) * EPS * (a.double().abs() @ w2.double().abs().T)
        want = torch.nn.functional.silu(x) * up
        bound = 1.1 * bound * up.abs() + x.abs() * up_bound + 8 * EPS * want.abs()
        size = torch.maximum(size, torch.maximum(want.abs(), a.double().abs() @ w2.double().abs().T))
    held = size < largest / 2   # (no partial sum on the way can overflow)
    assert held.any(1).all() and (x.abs() > 2.0 ** 82)[held].any()
    assert ((got.double() - want).abs()[held] <= bound[held]).all()
    for rows in (slice(0, 5), slice(M // 2 - 2, M // 2 + 3), slice(M - 5, M), slice(0, min(16, M))):
        assert torch.equal(ops.gemm(a[rows], w, **kw).nan_to_num(), got[rows].nan_to_num())


@pytest.mark.parametrize("M", [4, 16, 509])
def test_products_of_undefined_rows_take_bounded_time(M):
    """Rows that are not finite are done again by the matrix unit: less than 20 times as long as others (2 to 8 times are measured; by
    single lanes it was 110 to 210)."""
    from simply_amd.kernels import ops

    w, a = draw((2304, 9216), 71, 0.1), draw((M, 9216), 72)
    b = a.clone()
    b[:, 5] = float("nan")
    assert torch.isnan(ops.gemm(b, w)).all()

    def time(x):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(10):
            ops.gemm(x, w)
        end.record()
        end.synchronize()
        return begin.elapsed_time(end)

    time(a)
    assert time(b) < 20 * max(time(a), time(a))


def test_products_keep_special_values():
    """An infinite or undefined entry reaches its own row and column only."""
    from simply_amd.kernels import ops

    for M in (3, 40):
        a, w = draw((M, 72), 5), draw((50, 72), 6)
        a[1, 70], w[7, 3] = float("inf"), float("nan")
        got = ops.gemm(a, w)
        assert torch.isnan(got[:, 7]).all()
        rest = torch.cat([got[:, :7], got[:, 8:]], 1)
        assert torch.isinf(rest[1]).all() and torch.isfinite(rest[torch.arange(M) != 1]).all()


def attention_64(q, kp, vp, table, slot, positions, H, window, cap, scale, sinks):
    """q [T, H, hd] of one request at `positions`, its keys and values gathered from the pages: 64 bits."""
    from torch_ops import stored_keys_as_rows

    kp = stored_keys_as_rows(kp)
    _, Kh, P, hd = kp.shape
    n = int(positions[-1]) + 1
    at = torch.arange(n, device="cuda")
    pages = table[slot, at // P].long().clamp_min(0)
    k, v = kp[pages, :, at % P].double(), vp[pages, :, :, at % P].double()      # [n, Kh, hd]
    k, v = (x.repeat_interleave(H // Kh, 1) for x in (k, v))
    s = torch.einsum("thd,nhd->htn", q.double(), k) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    d = positions[:, None] - at[None]
    seen = (d >= 0) & (d < (window or n))
    s = s.masked_fill(~seen, float("-inf"))
    if sinks is not None:
        s = torch.cat([s, sinks.double()[:, None, None].expand(H, len(positions), 1)], 2)
    p = torch.softmax(s, -1)[..., :n]
    return torch.einsum("htn,nhd->thd", p, torch.where(torch.isnan(v), torch.zeros_like(v), v))


@pytest.mark.parametrize("H,Kh,hd,P,window,cap,sink", [
    (8, 4, 256, 16, None, 50.0, False), (8, 4, 256, 16, 300, 50.0, False), (4, 4, 64, 32, 17, None, True),
    (6, 2, 128, 16, None, None, True), (16, 1, 64, 48, 64, 30.0, False)])
def test_attention(H, Kh, hd, P, window, cap, sink):
    """Portions and single tokens around the ends of chunks (64) and ranges (256) of keys, a workgroup per range and one
    that walks through them.  Bounds: the scores' sums of hd products and the weighted values' sums, each (n + 8) eps of
    the sums of magnitudes, which unit normal entries keep below 1e-5 of the largest value."""
    from simply_amd.kernels import ops
    from test_gpu_kernels import paged_setup

    lens = [1, 63, 64, 65, 256, 257, 700, 1100]
    kp, vp, table = paged_setup(torch.float32, len(lens), H, Kh, hd, P, lens, 31)
    if window:   # pages that no query of the step sees are another's by now
        first = max(lens) - 150 - window
        table[len(lens) - 1, :max(first, 0) // P] = -1
    portions = [(s, max(0, n - (1 if s < 4 else 150)), n) for s, n in enumerate(lens)]
    T = sum(b - a for _, a, b in portions)
    q = draw((T, H * hd + 32), 32, 0.5)[:, :H * hd]
    sinks = draw((H,), 33) if sink else None
    G = H // Kh
    kw = dict(window=window, soft_cap=cap, scale=0.7, sinks=sinks, max_kv_len=max(lens))
    out = torch.zeros(T, H * hd, device="cuda")
    per = 16 // G
    units, row = [], 0
    for s, a, b in portions:
        units += [(s, row + i, min(per, b - a - i), a + i) for i in range(0, b - a, per)]
        row += b - a
    dev = torch.tensor(units, dtype=torch.int32).cuda()
    assert ops.attention_f32_takes(q, kp, vp, H)
    ops.paged_attention_f32(q, kp, vp, table, dev, 0, len(units), H, max_q_len=per, out=out, **kw)
    row = 0
    for s, a, b in portions:
        want = attention_64(q[row:row + b - a].reshape(-1, H, hd), kp, vp, table, s, torch.arange(a, b, device="cuda"), H, window,
                            cap, 0.7, sinks)
        err = (out[row:row + b - a].double().reshape(want.shape) - want).abs().max()
        assert err <= 1e-5 * want.abs().max(), (s, float(err), float(want.abs().max()))
        row += b - a
    # one token at a time, a few units to a launch: the same bits
    single = [(s, r + i, 1, p + i) for s, r, n, p in units for i in range(n)]
    one = torch.zeros_like(out)
    dev = torch.tensor(single, dtype=torch.int32).cuda()
    for i in range(0, len(single), 100):
        ops.paged_attention_f32(q, kp, vp, table, dev, i, min(100, len(single) - i), H, max_q_len=1, out=one, **kw)
    assert torch.equal(one, out)


@pytest.mark.parametrize("H,Kh,hd,window,per", [(8, 4, 256, None, 1), (8, 4, 256, 300, 3), (6, 2, 128, None, 5), (16, 1, 64, 700, 1)])
def test_attention_in_chunks_ranges_and_walks(H, Kh, hd, window, per):
    """The same units with a workgroup for each chunk, for each range, and one that walks through the ranges (a workspace of nothing):
    the same bits, within the bound above, and nothing written behind the rows that there are."""
    from simply_amd.kernels import lib, ops
    from test_gpu_kernels import paged_setup

    P, lens = 16, [per, 64, 255, 256, 257, 513, 1100]
    kp, vp, table = paged_setup(torch.float32, len(lens), H, Kh, hd, P, lens, 71)
    q = draw((per * len(lens), H * hd), 72, 0.5)
    units = torch.tensor([(s, per * s, per, n - per) for s, n in enumerate(lens)], dtype=torch.int32).cuda()
    outs = []
    for parts, count, planned, room in ((4, 1, 1100, None), (1, len(lens), 60000 if window is None else 1100, None), (0, len(lens), 1100, 0)):
        if parts == 1 and window is not None:   # (a window bounds the ranges: more units then, each several times)
            count = 1 + 128 // (Kh * 3)
        assert ops.attention_f32_parts(count, Kh, hd, window, planned, per, room) == parts
        out = torch.full((len(q) + 1, H * hd), 7.0, device="cuda")
        more = units.repeat(-(-count // len(lens)) + 1, 1).contiguous()
        ws = torch.full((64 << 20,), 255, dtype=torch.uint8, device="cuda")   # (undefined numbers)
        for i in range(0, len(lens), count):
            lib.call("sa_paged_attention_f32", q.data_ptr(), q.stride(0), kp.data_ptr(), vp.data_ptr(), table.data_ptr(), table.stride(0),
                     more.data_ptr(), i, count, out.data_ptr(), out.stride(0), H, Kh, hd, P, window or 0, 30.0, 0.7, None, planned, per,
                     ws.data_ptr(), ws.numel() if room is None else room, torch.cuda.current_stream().cuda_stream)
        assert (out[-1] == 7).all()
        outs.append(out[:-1])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    for s, n in enumerate(lens):
        want = attention_64(q[per * s:per * s + per].reshape(-1, H, hd), kp, vp, table, s, torch.arange(n - per, n, device="cuda"), H, window, 30.0,
                            0.7, None)
        assert (outs[0][per * s:per * s + per].double().reshape(want.shape) - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("H,Kh,hd", [(8, 4, 256), (6, 2, 128), (4, 4, 64)])
def test_attention_errors_no_larger_than_row_by_row(H, Kh, hd):
    """Root mean square errors against 64 bits over a prompt of 300 tokens behind 200: no larger than those of the kernel that
    goes row by row on the vector ALU, which serves other sizes (a tenth for the difference of the two sets of roundings)."""
    from simply_amd.kernels import ops
    from test_gpu_kernels import paged_setup

    n, T, P = 500, 300, 16
    kp, vp, table = paged_setup(torch.float32, 1, H, Kh, hd, P, [n], 51)
    q = draw((T, H * hd), 52, 2 * hd ** -0.5)
    pos = torch.arange(n - T, n, dtype=torch.int32, device="cuda")
    one, here = torch.empty(T, H * hd, device="cuda"), torch.empty(T, H * hd, device="cuda")
    ops.paged_attention(q, kp, vp, table, torch.zeros(T, dtype=torch.int32, device="cuda"), pos, H, window=None, soft_cap=50.0, out=one)
    per = 16 // (H // Kh)
    units = torch.tensor([(0, i, min(per, T - i), n - T + i) for i in range(0, T, per)], dtype=torch.int32).cuda()
    ops.paged_attention_f32(q, kp, vp, table, units, 0, len(units), H, window=None, soft_cap=50.0, max_kv_len=n, max_q_len=per, out=here)
    want = attention_64(q.view(T, H, hd), kp, vp, table, 0, pos.long(), H, None, 50.0, 1.0, None).reshape(T, -1)
    rms = lambda x: float((x.double() - want).square().mean().sqrt())
    print(rms(one), rms(here))
    assert rms(here) <= 1.1 * rms(one)


def test_attention_keeps_special_values():
    """Values that are not finite reach the queries that see them and no others of the same unit."""
    from simply_amd.kernels import ops
    from test_gpu_kernels import paged_setup

    H, Kh, hd, P, n, window = 2, 1, 64, 16, 40, 12
    kp, vp, table = paged_setup(torch.float32, 1, H, Kh, hd, P, [n], 41)
    at = 27
    vp[table[0, at // P].long(), 0, 5, at % P] = float("inf")
    q = draw((8, H * hd), 42)
    for first in (20, 24, 32):   # the key becomes visible within the unit, or leaves its window
        units = torch.tensor([[0, 0, 8, first]], dtype=torch.int32).cuda()
        out = torch.empty(8, H * hd, device="cuda")
        ops.paged_attention_f32(q, kp, vp, table, units, 0, 1, H, window=window, soft_cap=None, max_kv_len=n, max_q_len=8, out=out)
        sees = torch.tensor([first + i >= at and first + i - window < at for i in range(8)], device="cuda")
        bad = ~torch.isfinite(out.view(8, H, hd))
        assert torch.equal(bad[:, :, 5], sees[:, None].expand(8, H)) and not bad[:, :, :5].any() and not bad[:, :, 6:].any()
