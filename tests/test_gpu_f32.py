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
    """Few rows, tiles and tiles cut over K, plain, gated and soft-capped: each within the bound on a sum of K products in
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
