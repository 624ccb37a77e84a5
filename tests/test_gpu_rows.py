"""Row kernels at widths around the pieces that a thread takes, aligned and not: against 64-bit references."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def draw(shape, seed, dtype=torch.float32, mean=0.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) + mean).to(dtype).cuda()


@pytest.mark.parametrize("D", [8, 72, 100, 504, 512, 520, 2040, 2048, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_and_norms(D, dtype):
    """residual + mult y, its norm (root mean square, and centred with a mean that is large beside the spread), and the sum
    of a normed y.  Bounds: a sum of D squares in 32 bits is off by at most (D / 256 + 16) steps of 2^-24, results are
    rounded once to their type."""
    from simply_amd.kernels import ops

    T = 3
    step = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -8
    w, b = draw((D,), 1, dtype, 1.0), draw((D,), 2, dtype)
    for offset in (0, 3):   # rows of a wider buffer whose start is not aligned
        y = draw((T, D + 8), 3, dtype)[:, offset:offset + D]
        h = draw((T, D), 4, mean=20.0)
        total = h.double() + 0.7 * y.double()
        for bias in (None, b):
            for add in (y, None):
                got_h, x = h.clone(), total if add is not None else h.double()
                got = ops.residual_add_next_norm(add, got_h, w, eps=1e-5, bias=bias, mult=0.7, out_dtype=dtype)
                c = x - x.mean(1, keepdim=True) if bias is not None else x
                want = c / (c.square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double() + (b.double() if bias is not None else 0.0)
                assert (got_h.double() - x).abs().max() <= 2.0 ** -24 * 4 * x.abs().max()
                # centring takes away a mean of 20: what is left carries the sum's rounding, 20 * 2^-23, to its unit spread
                assert ((got.double() - want).abs() <= (step + (D / 256 + 16 + 60) * 2.0 ** -23) * (want.abs() + 1)).all(), (offset, bias is None)
        got_h = h.clone()
        out = ops.residual_add_norm(y, got_h, weight=w, eps=1e-5, mult=0.7, out_dtype=dtype)
        want = h.double() + 0.7 * y.double() / (y.double().square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double()
        assert ((got_h.double() - want).abs() <= (D / 256 + 20) * 2.0 ** -24 * 25).all()
        assert ((out.double() - want).abs() <= (step + (D / 256 + 20) * 2.0 ** -24) * 30).all()


@pytest.mark.parametrize("H,I,O,tail,gates", [(3, 128, 512, 64, None), (2, 512, 128, 0, "outputs"), (4, 32, 20, 4, "heads"),
                                              (2, 96, 68, 0, "outputs"), (1, 192, 16, 32, None), (2, 40, 36, 0, None)])
def test_head_products(H, I, O, tail, gates):
    """Tokens around the tiles of 16 and 64, heads apart from each other (the last case: inputs that the matrix cores do not
    take).  Sums of I bfloat16 products in 32 bits, rounded once; and a token's result does not depend on the others."""
    from simply_amd.kernels import ops

    w = draw((H, O, I), 1, torch.bfloat16)
    for T in (1, 16, 17, 64, 65, 150):
        x = draw((T, H * (I + tail + 8) + 16), 2, torch.bfloat16)[:, 8:]
        gate = None if gates is None else draw((T, (H if gates == "heads" else H * O) + 8), 3, torch.bfloat16)[:, 8:]
        got = ops.head_product(x, w, in_stride=I + tail + 8, tail=tail, gate=gate)
        rows = torch.stack([x[:, h * (I + tail + 8):h * (I + tail + 8) + I + tail] for h in range(H)], 1).double()
        want = torch.einsum("thi,hoi->tho", rows[:, :, :I], w.double())
        size = torch.einsum("thi,hoi->tho", rows[:, :, :I].abs(), w.double().abs())
        if gates is not None:
            g = torch.sigmoid(gate.double()).reshape(T, H, -1)
            want, size = want * g, size * g
        got = got.double().reshape(T, H, O + tail)
        assert ((got[:, :, :O] - want).abs() <= 2.0 ** -8 * want.abs() + (I + 8) * 2.0 ** -24 * size).all(), T
        assert torch.equal(got[:, :, O:], rows[:, :, I:])
        if T > 1 and I % 32 == 0:
            alone = ops.head_product(x[T - 1:], w, in_stride=I + tail + 8, tail=tail, gate=None if gate is None else gate[T - 1:])
            assert torch.equal(alone.double().reshape(H, -1), got[T - 1])


@pytest.mark.parametrize("H,size,dtype,weight,offset", [
    (3, 128, torch.float32, "shared", 0), (5, 32, torch.bfloat16, "own", 0), (1, 512, torch.bfloat16, None, 0),
    (7, 64, torch.float32, "own 32", 0), (2, 256, torch.bfloat16, "shared 32", 0), (3, 128, torch.float32, "shared", 3), (3, 96, torch.bfloat16, "own", 0)])
def test_gated_heads(H, size, dtype, weight, offset):
    """Heads in pieces of eight entries, and the sizes and alignments that are left to a wave a head (the last two): a norm's
    sum of squares is off by (size / 64 + 8) steps of 2^-24 at most, the rest by a few; the result is rounded once."""
    from simply_amd.kernels import ops

    w = None
    if weight is not None:
        w = draw((size * (H if "own" in weight else 1),), 2, torch.float32 if "32" in weight else torch.bfloat16, 1.0)
    for T in (1, 5, 67):
        x, g = draw((T, H * size + 8), 3, dtype)[:, offset:offset + H * size], draw((T, H * size + 16), 4, torch.bfloat16)[:, 8:8 + H * size]
        for kind in (0, 1):
            got = ops.gated_heads(x, g, H, size, kind=kind, weight=w, eps=1e-5, out_dtype=torch.bfloat16).double()
            v = x.double().reshape(T, H, size)
            if w is not None:
                v = v / (v.square().mean(2, keepdim=True) + 1e-5).sqrt() * w.double().reshape(-1, size)
            gd = g.double().reshape(T, H, size)
            want = (v * torch.sigmoid(gd) * (gd if kind == 1 else 1.0)).reshape(T, -1)
            assert ((got - want).abs() <= (2.0 ** -8 + (size / 64 + 24) * 2.0 ** -24) * want.abs() + 1e-30).all()


@pytest.mark.parametrize("D,dtype,out_dtype,gated,offset", [
    (2048, torch.bfloat16, torch.bfloat16, True, 0), (1028, torch.float32, torch.float32, False, 0), (4, torch.bfloat16, torch.float32, True, 0),
    (100, torch.float32, torch.bfloat16, True, 0), (64, None, torch.bfloat16, False, 0), (1030, torch.bfloat16, torch.bfloat16, True, 0),
    (64, torch.bfloat16, torch.bfloat16, False, 2)])
def test_expert_combine(D, dtype, out_dtype, gated, offset):
    """Four entries a thread, and the widths and alignments that are left to one (the last two): top products and two sums
    in 32 bits, rounded once."""
    from simply_amd.kernels import lib, ops

    for T, top in ((1, 1), (3, 4), (70, 9)):
        y, weights = draw((T * top, D), 1), draw((T, top), 2).abs()
        shared = None if dtype is None else draw((T, D + 8), 3, dtype)[:, offset:offset + D]
        gate = draw((T, 3), 4)[:, 1:2] if gated else None
        out = torch.empty((T, D), dtype=out_dtype, device="cuda")
        code = lambda t: 0 if t is None else ops._code(t)
        lib.call("sa_expert_combine", y.data_ptr(), weights.data_ptr(), top, None if shared is None else shared.data_ptr(), code(shared),
                 0 if shared is None else shared.stride(0), None if gate is None else gate.data_ptr(), 3, out.data_ptr(), code(out), D, T, D,
                 ops._stream())
        got = out.double()
        terms = y.double().reshape(T, top, D) * weights.double()[:, :, None]
        extra = torch.zeros(T, D, dtype=torch.float64, device="cuda") if shared is None else shared.double()
        if gate is not None:
            extra = extra * torch.sigmoid(gate.double())
        step = 2.0 ** -24 if out_dtype == torch.float32 else 2.0 ** -8
        room = terms.abs().sum(1) + extra.abs()
        assert ((got - terms.sum(1) - extra).abs() <= step * (terms.sum(1) + extra).abs() + (top + 12) * 2.0 ** -23 * room).all()


@pytest.mark.parametrize("M,N,K", [(65, 16, 256), (65, 64, 2048), (130, 4, 1000), (300, 256, 2048), (1025, 32, 4096), (2047, 16, 2048),
                                   (2047, 128, 520), (9000, 16, 1024), (17000, 8, 512)])
def test_narrow_products(M, N, K):
    """Many rows of few outputs, the inner dimension cut or not: sums of K bfloat16 products in 32 bits."""
    from simply_amd.kernels import ops
    from simply_amd.parts.base import as_product_weight

    x, w = draw((M, K + 8), 1, torch.bfloat16)[:, :K], draw((N, K), 2, torch.bfloat16)
    got = ops.gemm(x, as_product_weight(w), out_dtype=torch.float32).double()
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert ((got - want).abs() <= (K / 32 + 16) * 2.0 ** -24 * size).all()
