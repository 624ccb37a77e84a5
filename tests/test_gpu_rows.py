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
