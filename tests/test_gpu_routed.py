"""Routed experts' products on tiles of 16, 64 and 128 rows: against 32-bit products of the same operands, and to the bit
against one another."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def draw(shape, seed, std=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std


@pytest.mark.parametrize("T,E,top,D,F,gated", [(300, 2, 2, 192, 320, True), (200, 4, 1, 64, 100, False), (700, 8, 2, 128, 64, True),
                                               (260, 3, 2, 320, 196, True), (150, 4, 2, 80, 72, True)])
def test_tiles_agree(monkeypatch, T, E, top, D, F, gated):
    """All tokens at once (tiles of 64 rows, in the wide kernel but for the last case, whose sizes it does not take), in tiles of 128
    where the kernel takes them, and few at a time (tiles of 16): the same bits.  Against the reference: an expert's output is a sum of F products of a
    bfloat16 row h, itself off by at most two bfloat16 steps (2^-7 relative) of its factors' products."""
    from simply_amd.kernels import lib, ops
    from simply_amd.kernels.packing import stack_experts

    x = draw((T, D + 8), 1).bfloat16().cuda()[:, :D]
    ws = [[draw((r, c), 10 + 100 * i + e, c ** -0.5).bfloat16().cuda() for e in range(E)] for i, (r, c) in
          enumerate(((F, D), (F, D), (D, F)))]
    gate, up, down = (stack_experts(w) for w in ws)
    experts = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)])
    experts[: T // 3, 0], experts[: T // 3, 1:] = 0, experts[: T // 3, 1:].clamp_min(1)   # (one expert gets many rows)
    experts, weights = experts.to(torch.int32).cuda(), torch.rand(T, top, generator=torch.Generator().manual_seed(2)).cuda()
    args = (gate if gated else None, up, down, ops.ACT_SILU)
    got = ops.routed_experts(x, experts, weights, *args, out_dtype=torch.float32)
    if D % 64 == 0 and F % 64 == 0:
        monkeypatch.setattr(lib.load(), "sa_expert_tile_rows", lambda *a: 128)
        assert torch.equal(ops.routed_experts(x, experts, weights, *args, out_dtype=torch.float32), got)
        monkeypatch.undo()
    n = max(1, 10 * E // top)   # (pairs below 12 an expert)
    parts = [ops.routed_experts(x[i:i + n], experts[i:i + n].contiguous(), weights[i:i + n].contiguous(), *args,
                                out_dtype=torch.float32) for i in range(0, T, n)]
    assert torch.equal(got, torch.cat(parts))
    want, size = torch.zeros(T, D, device="cuda"), torch.zeros(T, D, device="cuda")
    for e in range(E):
        for k in range(top):
            rows = (experts[:, k] == e).nonzero()[:, 0]
            u = x[rows].float() @ ws[1][e].float().T
            h = torch.nn.functional.silu(x[rows].float() @ ws[0][e].float().T) * u if gated else torch.nn.functional.silu(u)
            want[rows] += weights[rows, k, None] * (h @ ws[2][e].float().T)
            size[rows] += weights[rows, k, None] * (h.abs() @ ws[2][e].float().abs().T)
    assert ((got - want).abs() <= 2.0 ** -6 * size + 1e-5).all()


@pytest.mark.parametrize("dtype,tile_rows", [(torch.float32, 16), (torch.float32, 64), (torch.bfloat16, 16), (torch.bfloat16, 64)])
def test_more_tiles_than_a_grid_s_second_index(dtype, tile_rows):
    """More than 65,535 tiles of rows; the last rows of the last tiles among them.  Whole numbers that both types hold: exact."""
    from simply_amd.kernels import lib, ops
    from simply_amd.kernels.packing import stack_experts

    P, E, N, K = 65536 * tile_rows + 5, 2, 16, 64
    a = torch.randint(-2, 3, (P, K), generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    w = [torch.randint(-2, 3, (N, K), generator=torch.Generator().manual_seed(e)).to(dtype).cuda() for e in (2, 3)]
    stack = stack_experts(w)
    experts = (torch.arange(P, dtype=torch.int32) % 7 == 0).int().cuda()
    max_tiles = lib.load().sa_expert_tiles_max(P, E, tile_rows)
    order = torch.empty(P, dtype=torch.int32, device="cuda")
    plan = torch.empty(1 + 3 * max_tiles, dtype=torch.int32, device="cuda")
    out = torch.full((P, N), -1.0, device="cuda")
    lib.call("sa_expert_sort", experts.data_ptr(), P, E, tile_rows, order.data_ptr(), plan.data_ptr(), plan.numel(), ops._stream())
    lib.call("sa_expert_product", a.data_ptr(), ops._code(a), K, 1, 1, stack.data.data_ptr(), None, N, K, order.data_ptr(),
             plan.data_ptr(), P, E, tile_rows, 0, 0.0, out.data_ptr(), N, 1, 0, ops._stream())
    assert int(plan[0]) > 65535
    a = a.float()
    want = torch.where(experts[:, None] == 0, a @ w[0].float().T, a @ w[1].float().T)
    assert torch.equal(out, want)
