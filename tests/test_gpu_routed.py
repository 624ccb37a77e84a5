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


@pytest.mark.parametrize("T,E,top,D,F,S,gated,options", [
    (1, 1, 1, 32, 16, 16, True, None), (16, 128, 8, 960, 64, 96, True, None), (8, 16, 2, 2048, 128, 128, True, dict(groups=4, keep=2, softmax=True, group_best=1, renorm=1e-20)),
    (5, 17, 3, 96, 40, 24, False, dict(softmax=False, correction=True, bias=True)), (16, 9, 3, 160, 48, 320, True, dict(softmax="chosen")),
    (3, 128, 40, 64, 32, 8, False, dict(groups=16, keep=7))])
def test_few_tokens(T, E, top, D, F, S, gated, options):
    """The router in one launch and the shared feed-forward beside the experts, against the separate kernels on the same logits: the
    same experts, weights and order of experts.  The sum over experts with the norm behind it: what the experts and the shared
    feed-forward give differs by the roundings of a bfloat16 run alone (2^-8 of the shared rows, which the separate kernels round)."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_gate_up, pack_tiles, stack_experts

    x = draw((T, D + 8), 1).bfloat16().cuda()[:, :D]
    router = pack_tiles(draw((E + 1, D), 2, 3 * D ** -0.5).bfloat16().cuda())
    o = None if options is None else dict(options)
    for name in ("correction", "bias"):
        if o and o.get(name):
            o[name] = draw((E,), 3).cuda()
    assert ops.route_few_takes(x, router, E, top)
    logits, experts, weights, order = ops.route_few(x, router, E, top, 1.5, options=o)
    # (sums of D products in another order: 2^-24 of their sizes for each of at most D steps)
    want = ops.gemm(x, router, out_dtype=torch.float32)
    assert torch.allclose(logits, want, rtol=0, atol=D * 2.0 ** -24 * 3 * D ** 0.5)
    e, w = ops.route(logits[:, :E], top, 1.5) if o is None else ops.route_choice(logits[:, :E], top, 1.5, **o)
    assert torch.equal(experts, e) and torch.equal(weights, w)
    flat, (pairs, plan) = experts.flatten().cpu(), (order[0].cpu().long(), order[1].cpu())
    assert sorted(pairs.tolist()) == list(range(T * top)) and bool((flat[pairs].diff() >= 0).all())
    tiles, at = [], 0
    for n in range(E):
        rows = int((flat == n).sum())
        for i in range(0, rows, 16):
            tiles += [n, at + i, min(16, rows - i)]
        at += rows
    assert plan[0] == len(tiles) // 3 and plan[1:1 + len(tiles)].tolist() == tiles

    ws = [[draw((r, c), 10 + 100 * i + n, c ** -0.5).bfloat16().cuda() for n in range(E)] for i, (r, c) in
          enumerate(((F, D), (F, D), (D, F)))]
    gate, up, down = (stack_experts(v) for v in ws)
    sg, su, sd = draw((S, D), 5, D ** -0.5).bfloat16().cuda(), draw((S, D), 6, D ** -0.5).bfloat16().cuda(), draw((D, S), 7, S ** -0.5).bfloat16().cuda()
    first = pack_gate_up(sg, su) if gated else pack_tiles(su)
    args = (x, experts, weights, gate if gated else None, up, down, ops.ACT_SILU)
    hidden = ops.gemm(x, first, activation=ops.ACT_SILU) if gated else ops.gemm(x, first, activate=ops.ACT_SILU)
    shared = ops.gemm(hidden, pack_tiles(sd), out_dtype=torch.float32)
    kw = dict(shared_gate=logits[:, E:], out_dtype=torch.float32)
    beside = ops.route_few(x, router, E, top, 1.5, options=o, dense=(first, ops.ACT_SILU, None))
    assert all(torch.equal(a, b) for a, b in zip(beside, (logits, experts, weights)))
    assert torch.equal(beside[3][0], order[0]) and torch.equal(beside[3][1][:1 + len(tiles)], order[1][:1 + len(tiles)])
    # (a bfloat16 step where a sum of D products in another order rounds the other way)
    assert torch.allclose(beside[4].float(), hidden.float(), rtol=2.0 ** -7, atol=2.0 ** -12)
    got = ops.expert_sums(*args, order=order, dense=(beside[4], pack_tiles(sd)), **kw).materialize()
    want = ops.routed_experts(*args, shared=shared, **kw)
    # (hidden entries of the shared feed-forward may round the other way where their sums are taken in another order)
    assert torch.allclose(got, want, rtol=0, atol=2.0 ** -8 * float(shared.abs().max()))
    h = draw((T, D), 8).cuda()
    h2, scale = h.clone(), draw((D,), 9).bfloat16().cuda()
    sums = ops.expert_sums(*args, shared=shared, shared_gate=logits[:, E:])
    a = ops.residual_add_next_norm(sums, h, scale, eps=1e-5, mult=0.7)
    b = ops.residual_add_next_norm(want, h2, scale, eps=1e-5, mult=0.7, out_dtype=torch.bfloat16)
    assert torch.equal(h, h2) and torch.equal(a, b)


@pytest.mark.parametrize("T,D,E", [(1, 1024, 16), (1, 4096, 16), (3, 992, 16), (16, 1024, 16), (8, 2048, 64), (5, 7168, 16), (16, 96, 16)])
def test_router_of_few_tokens_errors_no_larger_than_the_product_kernel_s(T, D, E):
    """Logits against 64 bits, root mean squares over 24 drawings: no larger than those of the product kernel that takes more tokens (a
    twentieth for the difference of the two sets of roundings)."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles

    here = there = 0.0
    for seed in range(24):
        x, w = draw((T, D), 50 + seed).bfloat16().cuda(), draw((E, D), 90 + seed, D ** -0.5).bfloat16().cuda()
        tiled, want = pack_tiles(w), x.double() @ w.double().T
        assert ops.route_few_takes(x, tiled, E, 2)
        here += float((ops.route_few(x, tiled, E, 2, 1.0)[0].double() - want).square().mean())
        there += float((ops.gemm(x, tiled, out_dtype=torch.float32).double() - want).square().mean())
    assert 0 < here <= 1.05 ** 2 * there, (here / there) ** 0.5


@pytest.mark.parametrize("shared", [16, 5120, 5136])
def test_shared_feed_forwards_beside_the_experts_and_apart(shared):
    """Up to and beyond the widest that runs beside the router and the experts, against 64 bits: half a bfloat16 step of 2^-8 for the
    hidden entries and for the result, and another for the shared rows where they come by themselves."""
    from simply_amd.parts.ffn import RoutedExperts

    T, D, E, F = 5, 64, 4, 48
    part = RoutedExperts(D, E, 2, F, shared_size=shared, shared_gate=False)
    tensors = {n: draw(s.shape, 200 + i, s.shape[1] ** -0.5).bfloat16().cuda() for i, (n, s) in enumerate(part.param_specs().items())}
    part.load(tensors)
    x = draw((T, D), 199).bfloat16().cuda()
    got = part.forward(x).double()
    w = {n: t.double() for n, t in tensors.items()}
    ff = lambda p, up: (torch.nn.functional.silu(x.double() @ w[p + "gate" + up].T) * (x.double() @ w[p + "up" + up].T)) @ w[p + "down" + up].T
    scores = torch.softmax(x.double() @ w["router"].T, -1)
    best = scores.topk(2, -1)
    want = ff("shared.", "_proj")
    for k in range(2):
        every = torch.stack([ff(f"e{e}.", "") for e in range(E)])
        want += best.values[:, k:k + 1] * every[best.indices[:, k], torch.arange(T, device="cuda")]
    assert float((got - want).norm() / want.norm()) <= 1.5 * 2.0 ** -8


@pytest.mark.parametrize("T,F,shared_F", [(600, 2048, 64), (1031, 2112, 2048), (1801, 2048, 4160)])
def test_shared_product_beside_the_experts_of_many_tokens(gpu_lib, T, F, shared_F):
    """The second product of a shared feed-forward in the launch of the experts' second products: the experts' rows to the bit those of the
    launch without it, its own those of the wide kernel by itself with K uncut (the same order of sums)."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles, stack_experts
    D, E, top = 2048, 16, 2
    gen = torch.Generator(device="cuda").manual_seed(5)
    draw = lambda *shape: (torch.randn(shape, generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
    gate, up, down = (stack_experts([draw(r, c) for _ in range(E)]) for r, c in ((F, D), (F, D), (D, F)))
    x, hidden, w = draw(T, D), draw(T, shared_F + 8)[:, :shared_F], draw(D, shared_F)
    experts = torch.stack([torch.randperm(E, generator=gen, device="cuda")[:top] for _ in range(T)]).int().contiguous()
    weights = torch.rand((T, top), generator=gen, device="cuda")
    assert ops.experts_beside(T, top, up, down, x, pack_tiles(w))
    args = (x, experts, weights, gate, up, down, ops.ACT_SILU)
    apart, beside = ops.expert_sums(*args), ops.expert_sums(*args, dense=(hidden, pack_tiles(w)))
    assert torch.equal(apart.y, beside.y)
    assert torch.equal(beside.shared, ops.gemm(hidden, pack_tiles(w), algo=ops.ALGO_WIDE, shape=3128128))
