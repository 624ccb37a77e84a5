"""Recurrences worked through in pieces of tokens on the matrix cores, against their token-by-token definition in 64 bits:
pieces that are full, short, alone and many; sizes that fill no block; decays near one, near zero, zero and one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def uniform(shape, seed, lo=0.0, hi=1.0):
    g = torch.Generator().manual_seed(seed)
    return torch.rand(shape, generator=g) * (hi - lo) + lo


def normal(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def delta_64(qkv, gates, state, meta, H, G, dk, dv):
    """The definition, token by token."""
    T = qkv.shape[0]
    out, state = torch.zeros(T, H, dv, dtype=torch.float64), state.double().clone()
    q, k, v = (t.reshape(T, -1, d).double() for t, d in zip(qkv[:, :2 * G * dk + H * dv].split([G * dk, G * dk, H * dv], 1), (dk, dk, dv)))
    q, k = (t.repeat_interleave(H // G, 1) for t in (q, k))
    beta, decay = gates.double().split(H, 1)
    for slot, first, count, _ in meta:
        S = state[slot, :H * dk * dv].reshape(H, dv, dk).transpose(1, 2).clone()
        for t in range(first, first + count):
            S = decay[t][:, None, None] * S
            u = beta[t][:, None] * (v[t] - (k[t][:, :, None] * S).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
            out[t] = (q[t][:, :, None] * S).sum(1)
        state[slot, :H * dk * dv] = S.transpose(1, 2).reshape(-1)
    return out.reshape(T, H * dv), state


@pytest.mark.parametrize("H,G,dk,dv,kind", [(2, 1, 128, 128, "slow"), (4, 4, 64, 64, "fast"), (3, 1, 20, 24, "ends"),
                                            (2, 2, 100, 130, "slow"), (2, 1, 128, 40, "alike"), (1, 1, 4, 3, "fast")])
def test_delta_rule(H, G, dk, dv, kind):
    """The kernel's error against 64 bits stays within three times that of the token-by-token kernel (both are sums of 32-bit
    products in another order; three for the exponentials and the substitution) and below 1e-5 of the largest result."""
    from simply_amd.kernels import ops

    counts, before = [1, 15, 64, 65, 130, 200], 3
    T = before + sum(counts)
    meta, row = [], before
    for i, n in enumerate(counts):
        meta.append((5 - i if i else 6, row, n, 0))
        row += n
    C = 2 * G * dk + H * dv
    C += -C % 4
    qkv = normal((T, C), 51)
    heads = qkv[:, :2 * G * dk].reshape(T, 2 * G, dk)
    if kind == "alike":   # keys that nearly repeat, taken whole: what the triangular system is hardest on
        heads[:, G:] = heads[:1, G:] + 0.05 * heads[:, G:]
    heads = heads / heads.square().sum(-1, keepdim=True).sqrt()
    heads[:, :G] *= dk ** -0.5
    qkv[:, :2 * G * dk] = heads.reshape(T, -1)
    beta = uniform((T, H), 52) if kind != "alike" else uniform((T, H), 52, 0.95, 1.0)
    decay = {"slow": 1.0 - 0.01 * uniform((T, H), 53), "fast": uniform((T, H), 53), "alike": torch.ones(T, H),
             "ends": torch.randint(0, 2, (T, H), generator=torch.Generator().manual_seed(53)).float()}[kind]
    gates = torch.cat([beta, decay], 1).contiguous()
    state = torch.cat([normal((7, H * dk * dv), 54), torch.zeros(7, 4 + -(H * dk * dv) % 4)], 1)
    want, want_state = delta_64(qkv, gates, state, meta, H, G, dk, dv)
    dev_meta = torch.tensor(meta, dtype=torch.int32).cuda()
    args = (qkv.cuda(), gates.cuda())
    s1, s2 = state.cuda(), state.cuda()
    one = ops.delta_rule(*args, s1, dev_meta, len(meta), H, G, dk, dv)
    out = torch.zeros(T, H * dv, device="cuda")
    assert ops.delta_chunks_takes(args[0], s2, len(meta), H, G, dk, dv)
    ops.delta_chunks(*args, s2, dev_meta, len(meta), before, max(counts), H, G, dk, dv, out=out)
    assert not out[:before].any()
    for got, ref, plain in ((out[before:], want[before:], one[before:]), (s2, want_state, s1)):
        err, base, top = ((x.double().cpu() - ref).abs().max() for x in (got, plain, torch.zeros_like(got)))
        print(kind, float(err / top), float(base / top))
        assert err <= 3 * base and err <= 1e-5 * top, (float(err), float(base), float(top))


def linear_64(p, at, q_mult, decay, bonus, state, meta, H, dk, dv):
    out, state = torch.zeros(len(p), H, dv, dtype=torch.float64), state.double().clone()
    q, k, v = (p[:, a:a + H * d].double().reshape(-1, H, d) for a, d in zip(at, (dk, dk, dv)))
    a = decay.double().reshape(-1, H, dk)
    for slot, first, count, _ in meta:
        S = state[slot, :H * dk * dv].reshape(H, dv, dk).transpose(1, 2).clone()
        for t in range(first, first + count):
            kv = k[t][:, :, None] * v[t][:, None, :]
            behind = a[t][:, :, None] * S + kv
            read = behind if bonus is None else S + bonus.double().reshape(H, dk, 1) * kv
            out[t], S = (q[t][:, :, None] * q_mult * read).sum(1), behind
        state[slot, :H * dk * dv] = S.transpose(1, 2).reshape(-1)
    return out.reshape(len(p), H * dv), state


@pytest.mark.parametrize("H,dk,dv,kind,bonus", [(2, 128, 128, "slow", True), (4, 64, 64, "fast", False), (3, 20, 24, "ends", True),
                                                (2, 100, 130, "spread", False), (1, 4, 3, "fast", True),
                                                (2, 128, 40, "spread", True)])
def test_channel_decays(H, dk, dv, kind, bonus):
    """As above: within three times the error of the kernel that goes token by token, and below 1e-5 of the largest result."""
    from simply_amd.kernels import ops

    counts, before = [1, 15, 64, 65, 130, 200], 3
    T = before + sum(counts)
    meta, row = [], before
    for i, n in enumerate(counts):
        meta.append((5 - i if i else 6, row, n, 0))
        row += n
    at = (4, 4 + H * dk + 8, 13 + 2 * H * dk)
    proj = normal((T, at[2] + H * dv + -(at[2] + H * dv) % 4), 61).bfloat16()
    decay = {"slow": 1.0 - 0.01 * uniform((T, H * dk), 62), "fast": uniform((T, H * dk), 62),
             "spread": torch.exp(-torch.exp(uniform((T, H * dk), 62, -8.0, 4.0))),
             "ends": torch.randint(0, 2, (T, H * dk), generator=torch.Generator().manual_seed(62)).float()}[kind]
    u = normal((H * dk,), 63) if bonus else None
    q_mult = 1.0 if bonus else dk ** -0.5
    state = torch.cat([normal((7, H * dk * dv), 64), torch.zeros(7, 4 + -(H * dk * dv) % 4)], 1)
    want, want_state = linear_64(proj, at, q_mult, decay, u, state, meta, H, dk, dv)
    dev_meta, dev_u = torch.tensor(meta, dtype=torch.int32).cuda(), u.cuda() if bonus else None
    s1, s2, p, g = state.cuda(), state.cuda(), proj.cuda(), decay.cuda()
    one = ops.linear_state(p, *at, q_mult, g, False, H, dk, dv, False, s1, dev_meta, len(meta), bonus=dev_u)
    out = torch.zeros(T, H * dv, device="cuda")
    assert ops.linear_chunks_takes(p, at[0], at[1], g, s2, len(meta), H, dk, dv)
    ops.linear_chunks(p, *at, q_mult, g, H, dk, dv, s2, dev_meta, len(meta), before, max(counts), bonus=dev_u, out=out)
    assert not out[:before].any()
    for got, ref, plain in ((out[before:], want[before:], one[before:]), (s2, want_state, s1)):
        err, base, top = ((x.double().cpu() - ref).abs().max() for x in (got, plain, torch.zeros_like(got)))
        print(kind, float(err / top), float(base / top))
        assert err <= 3 * base and err <= 1e-5 * top, (float(err), float(base), float(top))


def test_decays_from_their_logits():
    """a = sigmoid(z + bias)^(1 / tau) is computed as the token-by-token kernel does it: results agree to 32-bit rounding."""
    from simply_amd.kernels import ops

    H, dk, dv, T = 2, 64, 32, 150
    proj, z = normal((T, 2 * H * dk + H * dv), 71).bfloat16().cuda(), normal((T, H * dk), 72).cuda()
    bias, meta = normal((H * dk,), 73).bfloat16().cuda(), torch.tensor([[0, 0, T, 0]], dtype=torch.int32).cuda()
    at, kw = (0, H * dk, 2 * H * dk), dict(decay_bias=bias, tau=16.0)
    s1, s2 = torch.zeros(1, H * dk * dv).cuda(), torch.zeros(1, H * dk * dv).cuda()
    want = ops.linear_state(proj, *at, 0.125, z, False, H, dk, dv, False, s1, meta, 1, **kw)
    got = ops.linear_chunks(proj, *at, 0.125, z, H, dk, dv, s2, meta, 1, 0, T, out=torch.zeros_like(want), **kw)
    for x, y in ((got, want), (s2, s1)):
        assert (x - y).abs().max() <= 1e-5 * y.abs().max()


@pytest.mark.parametrize("T,H", [(512, 4), (1000, 8)])
def test_errors_no_larger_than_token_by_token(T, H):
    """Root mean square errors against 64 bits over all results and states, at the values that the recurrences meet (keys that
    have much in common, half-lives from a token to thousands): at most a tenth above the token-by-token kernels' (the mean
    over so many entries is itself steady to a hundredth; the products' sums in one chain each were 1.2 to 1.9 times off)."""
    from simply_amd.kernels import ops

    d, G, meta = 128, H // 2, torch.tensor([[0, 0, T, 0]], dtype=torch.int32).cuda()
    rms = lambda got, ref: (got.double().cpu() - ref).square().mean().sqrt()

    def no_larger(one, pieces, want):
        for name, a, b, ref in zip(("result", "state"), one, pieces, want):
            print(name, float(rms(a, ref)), float(rms(b, ref)))
            assert rms(b, ref) <= 1.1 * rms(a, ref), name

    silu = torch.nn.functional.silu
    q, k = silu(normal((T, G, d), 101)), silu(normal((T, G, d), 102))
    q, k = q / q.norm(dim=-1, keepdim=True) * d ** -0.5, k / k.norm(dim=-1, keepdim=True)
    qkv = torch.cat([q.reshape(T, -1), k.reshape(T, -1), silu(normal((T, H * d), 103))], 1)
    step = torch.nn.functional.softplus(0.5 * normal((T, H), 104) + uniform((H,), 105, -7.0, -2.2))
    gates = torch.cat([torch.sigmoid(normal((T, H), 106)), torch.exp(-uniform((H,), 107, 1.0, 16.0) * step)], 1)
    want = delta_64(qkv, gates, torch.zeros(1, H * d * d), meta.tolist(), H, G, d, d)
    s1, s2 = torch.zeros(1, H * d * d).cuda(), torch.zeros(1, H * d * d).cuda()
    one = ops.delta_rule(qkv.cuda(), gates.cuda(), s1, meta, 1, H, G, d, d)
    no_larger((one, s1), (ops.delta_chunks(qkv.cuda(), gates.cuda(), s2, meta, 1, 0, T, H, G, d, d, out=torch.empty_like(one)), s2), want)

    proj, bonus = normal((T, 3 * H * d), 108).bfloat16(), 0.3 * normal((H * d,), 109)
    decay = torch.exp(-torch.exp(uniform((H * d,), 110, -6.0, 0.5) + 0.1 * normal((T, H * d), 111)))
    at = (0, H * d, 2 * H * d)
    want = linear_64(proj, at, 1.0, decay, bonus, torch.zeros(1, H * d * d), meta.tolist(), H, d, d)
    p, g, u, s1, s2 = proj.cuda(), decay.cuda(), bonus.cuda(), torch.zeros_like(s1), torch.zeros_like(s1)
    one = ops.linear_state(p, *at, 1.0, g, False, H, d, d, False, s1, meta, 1, bonus=u)
    no_larger((one, s1), (ops.linear_chunks(p, *at, 1.0, g, H, d, d, s2, meta, 1, 0, T, bonus=u, out=torch.empty_like(one)), s2), want)


def cut_rows(takes, pieces):
    """The bytes of a workspace for so many pieces, found through the library's own answer (`takes(bytes)`: one piece more than
    requests at least)."""
    lo, hi = 1, 1 << 28
    while lo < hi:
        lo, hi = (lo, (lo + hi) // 2) if takes((lo + hi) // 2) else ((lo + hi) // 2 + 1, hi)
    return lo // 6 * pieces   # (five requests)


@pytest.mark.parametrize("room", [1, 2, 3])
def test_rows_in_portions_where_the_workspace_is_small(room):
    """Room for 64, 128 or 192 rows at a time: portions end within requests, between them and at a remainder, and a request's
    state goes through memory on the way.  Bounds as for whole steps."""
    from simply_amd.kernels import lib as _lib, ops

    H, G, dk, dv, before, counts = 2, 1, 40, 24, 3, [1, 63, 64, 30, 141]
    lib, T = _lib.load(), 3 + sum(counts)
    meta = [(4 - i, before + sum(counts[:i]), n, 0) for i, n in enumerate(counts)]
    dev_meta = torch.tensor(meta, dtype=torch.int32).cuda()
    state = normal((5, H * dk * dv), 121)
    ptr, stream = ops._ptr, ops._stream

    def check(out, one, want, s2, s1, want_state):
        assert not out[:before].any()
        for got, ref, plain in ((out[before:], want[before:], one[before:]), (s2, want_state, s1)):
            err, base, top = ((x.double().cpu() - ref).abs().max() for x in (got, plain, torch.zeros_like(got)))
            assert err <= 3 * base and err <= 1e-5 * top, (float(err), float(base), float(top))

    C = 2 * G * dk + H * dv
    qkv = normal((T, C), 122)
    heads = qkv[:, :2 * G * dk].reshape(T, 2 * G, dk)
    qkv[:, :2 * G * dk] = (heads / heads.square().sum(-1, keepdim=True).sqrt()).reshape(T, -1)
    gates = torch.cat([uniform((T, H), 123), uniform((T, H), 124, 0.9, 1.0)], 1)
    want, want_state = delta_64(qkv, gates, state, meta, H, G, dk, dv)
    s1, s2, x, g, out = state.cuda(), state.cuda(), qkv.cuda(), gates.cuda(), torch.zeros(T, H * dv, device="cuda")
    one = ops.delta_rule(x, g, s1, dev_meta, 5, H, G, dk, dv)
    size = cut_rows(lambda b: lib.sa_delta_chunks_takes(C, G, H, dk, dv, state.stride(0), 5, b), 5 + room)
    ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
    _lib.call("sa_delta_chunks", ptr(x), C, G, dk, dv, ptr(g), H, ptr(s2), s2.stride(0), ptr(dev_meta), 5, before, T - before,
              max(counts), ptr(out), ptr(ws), size, stream())
    check(out, one, want, s2, s1, want_state)

    at = (0, H * dk, 2 * H * dk)
    proj, decay, bonus = normal((T, 2 * H * dk + H * dv), 125).bfloat16(), uniform((T, H * dk), 126, 0.5, 1.0), normal((H * dk,), 127)
    want, want_state = linear_64(proj, at, 1.0, decay, bonus, state, meta, H, dk, dv)
    s1, s2, p, g, u, out = state.cuda(), state.cuda(), proj.cuda(), decay.cuda(), bonus.cuda(), torch.zeros(T, H * dv, device="cuda")
    one = ops.linear_state(p, *at, 1.0, g, False, H, dk, dv, False, s1, dev_meta, 5, bonus=u)
    size = cut_rows(lambda b: lib.sa_linear_chunks_takes(H, dk, dv, at[0], at[1], p.stride(0), g.stride(0), state.stride(0), 5, b), 5 + room)
    ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
    _lib.call("sa_linear_chunks", ptr(p), p.stride(0), *at, 1.0, ptr(g), g.stride(0), 0, 0, 0.0, ptr(u), 0, H, dk, dv, ptr(s2),
              s2.stride(0), ptr(dev_meta), 5, before, T - before, max(counts), ptr(out), ptr(ws), size, stream())
    check(out, one, want, s2, s1, want_state)


@pytest.mark.parametrize("kind", ["logits", "redrawn"])
def test_errors_of_faster_decays(kind):
    """As above for decays of half-lives of some ten tokens, as logits give them and drawn anew for each token, where a key
    has been multiplied by as many decays as it is old: with these in 32 bits the errors were 1.1 to 1.2 (results) and 1.2 to
    1.4 times (state) the token-by-token kernel's."""
    from simply_amd.kernels import ops

    T, H, d = 150, 8, 128
    meta, at = torch.tensor([[0, 0, T, 0]], dtype=torch.int32).cuda(), (0, H * d, 2 * H * d)
    proj, bonus = normal((T, 3 * H * d), 121).bfloat16(), normal((H * d,), 122)
    decay = torch.sigmoid(normal((T, H * d), 123)) ** (1 / 16) if kind == "logits" else \
        torch.exp(-torch.exp(uniform((T, H * d), 123, -6.0, -1.0)))
    want = linear_64(proj, at, 1.0, decay, bonus, torch.zeros(1, H * d * d), meta.tolist(), H, d, d)
    p, g, u, s1, s2 = proj.cuda(), decay.cuda(), bonus.cuda(), torch.zeros(1, H * d * d).cuda(), torch.zeros(1, H * d * d).cuda()
    one = ops.linear_state(p, *at, 1.0, g, False, H, d, d, False, s1, meta, 1, bonus=u)
    out = ops.linear_chunks(p, *at, 1.0, g, H, d, d, s2, meta, 1, 0, T, bonus=u, out=torch.empty_like(one))
    for a, b, ref in ((one, out, want[0]), (s1, s2, want[1])):
        base, error = ((x.double().cpu() - ref).square().mean().sqrt() for x in (a, b))
        print(kind, float(base), float(error))
        assert error <= 1.1 * base


def special_values(run, T, H, dv, value_at, meta, token, bad):
    """`run(values)` -> (out, state).  A value of head 1, column 2 of `token` that is not finite changes that column of that
    head of its own request from `token` on, where nothing is finite any more, and no other bit."""
    (want, _), (got, state) = run(None), run((token, value_at + 1 * dv + 2, bad))
    _, first, count, _ = next(m for m in meta if m[1] <= token < m[1] + m[2])
    hit = torch.zeros(T, H, dv, dtype=torch.bool, device="cuda")
    hit[token:first + count, 1, 2] = True
    got, want = got.view(T, H, dv), want.view(T, H, dv)
    assert torch.isfinite(want).all() and not torch.isfinite(got[hit]).any()
    assert torch.equal(got[~hit], want[~hit])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("token", [3, 3 + 40, 3 + 47, 3 + 100 + 79, 3 + 100 + 129])
@pytest.mark.parametrize("bonus", [True, False])
def test_channel_decays_keep_special_values(bad, token, bonus):
    """A value that is not finite reaches its own and later tokens of its request alone, wherever in a piece it stands."""
    from simply_amd.kernels import ops

    H, dk, dv, meta = 2, 64, 24, [(0, 3, 100, 0), (1, 103, 130, 0)]
    T, at = 233, (0, 2 * 64, 4 * 64)
    proj = normal((T, 4 * 64 + H * dv), 81).bfloat16()
    gates, u = uniform((T, H * dk), 82, 0.5, 1.0).cuda(), normal((H * dk,), 83).cuda() if bonus else None

    def run(change):
        p, state, out = proj.clone(), normal((2, H * dk * dv), 84).cuda(), torch.zeros(T, H * dv, device="cuda")
        if change:
            p[change[0], change[1]] = change[2]
        ops.linear_chunks(p.cuda(), *at, 1.0, gates, H, dk, dv, state, torch.tensor(meta, dtype=torch.int32).cuda(), 2, 3, 130,
                          bonus=u, out=out)
        return out, state

    special_values(run, T, H, dv, at[2], meta, token, bad)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("token", [3, 3 + 40, 3 + 47, 3 + 100 + 79, 3 + 100 + 129])
def test_delta_rule_keeps_special_values(bad, token):
    """As above; and a key that is not finite leaves nothing finite behind itself in its head and changes nothing before."""
    from simply_amd.kernels import ops

    H, dk, dv, meta = 2, 64, 24, [(0, 3, 100, 0), (1, 103, 130, 0)]
    T, C = 233, 2 * H * 64 + H * 24
    qkv = normal((T, C), 91)
    heads = qkv[:, :2 * H * dk].reshape(T, 2 * H, dk)
    qkv[:, :2 * H * dk] = (heads / heads.square().sum(-1, keepdim=True).sqrt()).reshape(T, -1)
    gates = torch.cat([uniform((T, H), 92), uniform((T, H), 93, 0.9, 1.0)], 1).cuda()

    def run(change):
        x, state, out = qkv.clone(), normal((2, H * dk * dv), 94).cuda(), torch.zeros(T, H * dv, device="cuda")
        if change:
            x[change[0], change[1]] = change[2]
        ops.delta_chunks(x.cuda(), gates, state, torch.tensor(meta, dtype=torch.int32).cuda(), 2, 3, 130, H, H, dk, dv, out=out)
        return out, state

    special_values(run, T, H, dv, 2 * H * dk, meta, token, bad)
    (want, _), (got, _) = run(None), run((token, (H + 1) * dk + 5, bad))
    _, first, count, _ = next(m for m in meta if m[1] <= token < m[1] + m[2])
    hit = torch.zeros(T, H, dv, dtype=torch.bool, device="cuda")
    hit[token:first + count, 1] = True
    got, want = got.view(T, H, dv), want.view(T, H, dv)
    assert not torch.isfinite(got[hit]).any() and torch.equal(got[~hit], want[~hit])


@pytest.mark.parametrize("H,dk,dv,T", [(2, 128, 128, 768), (3, 40, 24, 1025), (1, 64, 130, 831), (2, 100, 3, 900)])
@pytest.mark.parametrize("bad", [None, float("inf"), float("nan")])
def test_outputs_behind_the_walk(H, dk, dv, T, bad):
    """A long request by itself, whose states are kept and whose outputs are made behind the walk, and the same request among so many
    that its outputs are made on the way: the same sums in the same order, so the same bits, also where a value is not finite."""
    from simply_amd.kernels import ops

    n = 128 // (H * -(-dv // 16)) + 1   # one more than half of the CUs have walkers for
    G, counts = H, [T] + [1] * n
    rows = sum(counts)
    meta = torch.tensor([[len(counts) - 1 - i, sum(counts[:i]), c, 0] for i, c in enumerate(counts)], dtype=torch.int32).cuda()
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(1.0), b.nan_to_num(1.0))

    def both(run, width):
        got = []
        for k in (1, len(counts)):
            state, out = normal((len(counts), H * dk * dv), 131).cuda(), torch.zeros(rows, width, device="cuda")
            run(state, k, out)
            got.append((out[:T], state[len(counts) - 1]))
        assert same(got[0][0], got[1][0]) and same(got[0][1], got[1][1]) and got[0][0][:100].isfinite().all()

    C = 2 * G * dk + H * dv
    C += -C % 4
    qkv = normal((rows, C), 132) * dk ** -0.5
    gates = torch.cat([uniform((rows, H), 133), uniform((rows, H), 134, 0.9, 1.0)], 1)
    proj = normal((rows, 2 * H * dk + H * dv), 135).bfloat16()
    proj = torch.cat([proj, torch.zeros(rows, -proj.shape[1] % 4, dtype=proj.dtype)], 1)
    if bad is not None:
        qkv[T - 70, 2 * G * dk + 1] = bad
        proj[T - 70, 2 * H * dk + 1] = bad
    x, g, p, decay, bonus = qkv.cuda(), gates.cuda(), proj.cuda(), uniform((rows, H * dk), 136, 0.5, 1.0).cuda(), normal((H * dk,), 137).cuda()
    of = lambda t, k: t[:T] if k == 1 else t
    both(lambda s, k, out: ops.delta_chunks(of(x, k), of(g, k), s, meta, k, 0, T, H, G, dk, dv, out=of(out, k)), H * dv)
    for u in (None, bonus):
        both(lambda s, k, out: ops.linear_chunks(of(p, k), 0, H * dk, 2 * H * dk, 1.0, of(decay, k), H, dk, dv, s, meta, k, 0, T, bonus=u,
                                                 out=of(out, k)), H * dv)


@pytest.mark.parametrize("H,G,dk,dv,counts", [(2, 1, 128, 128, [1, 65, 900, 0]), (3, 3, 40, 24, [768, 63, 0, 1030]), (1, 1, 64, 130, [832, 64, 800])])
def test_outputs_behind_the_walk_of_several_requests(H, G, dk, dv, counts):
    """Short, long and empty requests in slots of any order behind rows of others, few enough that the states are kept: among empty
    requests, so many that they are not, with a workspace just too small for the states, and with one just large enough: the same
    bits, and nothing written elsewhere.  The definition in 64 bits beside them, bounds as above."""
    from simply_amd.kernels import lib as _lib, ops

    before, S = 3, len(counts)
    lib, T, ptr, stream = _lib.load(), 3 + sum(counts), ops._ptr, ops._stream
    meta = [(3 * i % S if S % 3 else S - 1 - i, before + sum(counts[:i]), n, 0) for i, n in enumerate(counts)]
    assert sorted(m[0] for m in meta) == list(range(S))
    blocks, nt = -(-dv // 16), 4 if dk <= 64 else 8
    many = 128 // (H * blocks) + 1
    every = meta + [(S, T, 0, 0)] * many
    dev = torch.tensor(every, dtype=torch.int32).cuda()
    state = normal((S + 1, H * dk * dv), 141)
    pieces = sum(counts) // 64 + S

    def check(takes, launch, plain, exact):
        least = cut_rows(lambda b: takes(5, b), 1)   # a piece without its state
        kept = least + H * blocks * nt * 1024
        got = []
        for n, size in ((S, 256 << 20), (len(every), 256 << 20), (S, pieces * kept), (S, (pieces + 1) * kept)):
            s, out = state.cuda(), torch.full((T + 1, H * dv), 7.0, device="cuda")
            ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
            launch(s, n, out, ws)
            assert (out[:before] == 7).all() and (out[T:] == 7).all() and torch.equal(s[S].cpu(), state[S])
            got.append((out[before:T], s))
        for out, s in got[1:]:
            assert torch.equal(out, got[0][0]) and torch.equal(s, got[0][1])
        s1 = state.cuda()
        one = plain(s1)
        want, want_state = exact()
        for a, b, ref in ((got[0][0], one[before:], want[before:]), (got[0][1], s1, want_state)):
            err, base, top = ((x.double().cpu() - ref).abs().max() for x in (a, b, torch.zeros_like(a)))
            assert err <= 3 * base and err <= 1e-5 * top, (float(err), float(base), float(top))

    C = 2 * G * dk + H * dv
    C += -C % 4
    qkv = normal((T, C), 142)
    heads = qkv[:, :2 * G * dk].reshape(T, 2 * G, dk)
    qkv[:, :2 * G * dk] = (heads / heads.square().sum(-1, keepdim=True).sqrt()).reshape(T, -1)
    gates = torch.cat([uniform((T, H), 143), uniform((T, H), 144, 0.9, 1.0)], 1)
    x, g = qkv.cuda(), gates.cuda()
    check(lambda n, b: lib.sa_delta_chunks_takes(C, G, H, dk, dv, state.stride(0), n, b),
          lambda s, n, out, ws: _lib.call("sa_delta_chunks", ptr(x), C, G, dk, dv, ptr(g), H, ptr(s), s.stride(0), ptr(dev), n, before,
                                          T - before, max(counts), ptr(out), ptr(ws), ws.numel(), stream()),
          lambda s: ops.delta_rule(x, g, s, dev, S, H, G, dk, dv), lambda: delta_64(qkv, gates, state, meta, H, G, dk, dv))

    at = (0, H * dk, 2 * H * dk)
    proj, decay, bonus = normal((T, 2 * H * dk + H * dv), 145).bfloat16(), uniform((T, H * dk), 146, 0.5, 1.0), normal((H * dk,), 147)
    proj = torch.cat([proj, torch.zeros(T, -proj.shape[1] % 4, dtype=proj.dtype)], 1)
    p, d, u = proj.cuda(), decay.cuda(), bonus.cuda()
    check(lambda n, b: lib.sa_linear_chunks_takes(H, dk, dv, at[0], at[1], p.stride(0), d.stride(0), state.stride(0), n, b),
          lambda s, n, out, ws: _lib.call("sa_linear_chunks", ptr(p), p.stride(0), *at, 1.0, ptr(d), d.stride(0), 0, 0, 0.0, ptr(u), 0, H, dk,
                                          dv, ptr(s), s.stride(0), ptr(dev), n, before, T - before, max(counts), ptr(out), ptr(ws), ws.numel(),
                                          stream()),
          lambda s: ops.linear_state(p, *at, 1.0, d, False, H, dk, dv, False, s, dev, S, bonus=u),
          lambda: linear_64(proj, at, 1.0, decay, bonus, state, meta, H, dk, dv))
