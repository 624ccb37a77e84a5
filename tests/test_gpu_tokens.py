"""Kernels that take a decode step's tokens through several operations at once, against the separate kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def draw(shape, seed, std=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std


@pytest.mark.parametrize("counts,H,d,rank,vectors", [([1], 1, 64, 8, torch.float32), ([1] * 8, 16, 128, 64, torch.bfloat16),
                                                     ([2, 0, 1, 5], 3, 64, 128, torch.bfloat16), ([1, 1, 3], 2, 128, 40, torch.float32)])
def test_wkv_token(counts, H, d, rank, vectors):
    """The same decays (the same products); states and sums over keys differ by the order of sums alone.  A head's o is a sum of d
    products, off by d roundings of 2^-24 of their sizes at most; the norm and the gate hand that on, rounded to bfloat16."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles

    C, T, S = H * d, sum(counts), len(counts)
    proj = draw((T, 4 * C + rank + 8), 1).bfloat16().cuda()[:, :4 * C + rank]
    w = pack_tiles(draw((C, rank), 2, rank ** -0.5).bfloat16().cuda())
    base, bonus, norm = (draw((C,), 3 + i, 0.5).to(vectors).cuda() for i in range(3))
    state = draw((S + 2, C * d + 12), 6).cuda()
    first, meta = 0, []
    for i, n in enumerate(counts):
        meta.append([S + 1 - i, first, n, 7])
        first += n
    meta = torch.tensor(meta, dtype=torch.int32).cuda()
    columns = (0, C, 2 * C, 3 * C, 4 * C)
    assert ops.wkv_token_takes(proj, w, d, state, 4 * C)
    mine, theirs = state.clone(), state.clone()
    got = ops.wkv_token(proj, columns, w, base, bonus, norm, 1e-5, H, d, mine, meta, S)
    decay = ops.low_rank_decay(proj[:, 4 * C:], w, base)
    o = ops.linear_state(proj, 0, C, 2 * C, 1.0, decay, False, H, d, d, False, theirs, meta, S, bonus=bonus)
    want = ops.gated_heads(o, proj[:, 3 * C:4 * C], H, d, kind=ops.GATE_SILU, weight=norm, eps=1e-5, out_dtype=torch.float32)
    assert torch.allclose(mine, theirs, rtol=2.0 ** -22, atol=2.0 ** -22 * 5)   # (a product and a sum a token)
    assert torch.equal(mine[:, C * d:], state[:, C * d:]) and torch.equal(mine[0], state[0])
    # bfloat16: half a step of 2^-8; the sums' roundings lie far below
    assert ((got.float() - want).abs() <= 2.0 ** -8 * want.abs() + d * 2.0 ** -22).all()


@pytest.mark.parametrize("slots,H,R,dr,rot,P,weights", [
    (list(range(32, 64)), 16, 512, 64, 64, 16, torch.bfloat16), ([5, -1, 7, 40], 3, 64, 32, 32, 16, torch.float32),
    (list(range(3, 40)), 2, 96, 16, 8, 4, torch.bfloat16), (list(range(64, 96)) + list(range(7, 12)), 5, 1000, 24, 16, 32, torch.float32),
    ([17], 1, 8, 8, 8, 16, torch.bfloat16)])
def test_latent_rows(slots, H, R, dr, rot, P, weights):
    """Queries to the bit (the same products of the same angles); rows to a bfloat16 step: the sum of squares is taken in another
    order, which can round an entry the other way."""
    from simply_amd.kernels import ops

    T, unit = len(slots), R + dr
    q = draw((T, H * unit), 1).bfloat16().cuda()
    proj = draw((T, unit + 24), 2).bfloat16().cuda()
    rows, weight = proj[:, 8:8 + unit], draw((R,), 3).to(weights).cuda()
    positions = torch.arange(T, dtype=torch.int32).cuda() * 37
    freq = torch.rand(rot // 2, generator=torch.Generator().manual_seed(4)).cuda()
    slot = torch.tensor(slots, dtype=torch.int64).cuda()
    pages = 128 // P + 1
    mine = [torch.full((pages, 1, P, unit), 7.0).bfloat16().cuda(), torch.full((pages, 1, R, P), 7.0).bfloat16().cuda()]
    theirs = [p.clone() for p in mine]
    assert ops.latent_rows_takes(q, rows, weight, H, R, rot, mine[0])
    want = q.clone()
    ops.latent_rows(q, rows, positions, freq, rot, H, R, weight, 1e-5, slot, *mine, rot_mult=0.9)
    ops.norm_rope_cache_write(want, positions, freq, rot, H, 0, unit, 0, rot_mult=0.9, q_rot_at=R)
    ops.norm_rope_cache_write(rows, positions, freq, rot, 0, 1, unit, 0, rot_mult=0.9, eps=1e-5, k_weight=weight, k_norm_dims=R, k_rot_at=R,
                              slot_mapping=slot, k_pages=theirs[0], v_pages=theirs[1], key_values=R)
    assert torch.equal(q, want)
    for a, b in zip(mine, theirs):
        a, b = a.float(), b.float()
        assert ((a - b).abs() <= 2.0 ** -7 * b.abs()).all() and float((a != b).float().mean()) < 0.01


@pytest.mark.parametrize("T,H,dr,rot", [(1, 64, 64, 64), (1, 65, 64, 64), (3, 200, 64, 64), (17, 129, 16, 16), (2, 9, 512, 512), (5, 19, 264, 256)])
def test_latent_rows_of_many_heads(T, H, dr, rot):
    """Heads that more than one workgroup turns: eight times what its 1,024 threads hold of 16 tokens."""
    test_latent_rows(list(range(48, 48 + T)), H, 16, dr, rot, 16, torch.bfloat16)


@pytest.mark.parametrize("T,D,vectors,centered,add", [
    (1, 8, torch.bfloat16, True, "rows"), (3, 2048, torch.bfloat16, True, "row"), (8, 2048, torch.float32, False, "none"),
    (5, 2056, torch.bfloat16, True, "experts"), (64, 4096, torch.float32, False, "experts32"), (7, 1000, torch.bfloat16, False, "experts"),
    (2, 4096, torch.bfloat16, True, "none")])
def test_norm_and_token_shift(T, D, vectors, centered, add):
    """The same sums, norms, mixes and last rows as the norm's kernel and the token shift's, to the bit; requests in other slots, other
    rows and the columns behind the last rows stay as they are.  Rows that are not whole pieces of eight are left to those two."""
    from simply_amd.kernels import ops

    h = draw((T, D), 1).cuda()
    w, b = (draw((D,), 2 + i, 0.3).to(vectors).cuda() for i in range(2))
    mu = torch.rand((5, D), generator=torch.Generator().manual_seed(4)).to(vectors).cuda()
    state = draw((T + 2, D + 24), 5).cuda()
    meta = torch.tensor([[T + 1 - j, j, 1, 9] for j in range(T)], dtype=torch.int32).cuda()
    shared = draw((T, D), 6).to(torch.float32 if add == "experts32" else torch.bfloat16).cuda()
    y = {"rows": lambda: draw((T, D + 8), 7).bfloat16().cuda()[:, :D], "row": lambda: draw((1, D), 7).bfloat16().cuda().expand(T, -1),
         "none": lambda: None}.get(add, lambda: ops.ExpertSums(draw((T * 2, D), 8).cuda(), torch.rand((T, 2)).cuda(), shared, None, torch.bfloat16))()
    kw = dict(eps=1e-5, mult=0.7, bias=b if centered else None)
    mine, theirs, one, two = h.clone(), h.clone(), state.clone(), state.clone()
    got = ops.add_next_norm_shift(y, mine, w, plus_one=False, mu=mu, tails=one[:, 16:], seq_meta=meta, num_seqs=T, **kw)
    normed = ops.residual_add_next_norm(y, theirs, w, out_dtype=torch.bfloat16, **kw)
    want = ops.token_shift(normed, mu, two[:, 16:], meta, T, 1)
    assert torch.equal(got, want) and torch.equal(mine, theirs) and torch.equal(one, two)
    args = dict(plus_one=False, seq_meta=meta, num_seqs=T, **kw)
    assert ops.add_next_norm_shift(y, mine, w, mu=mu, tails=one[:, 15:], **args) is None      # not aligned
    assert ops.add_next_norm_shift(y, mine, w, mu=mu[:4], tails=one[:, 16:], **args) is None  # not five streams
    assert torch.equal(mine, theirs) and torch.equal(one, two)


@pytest.mark.parametrize("add", ["rows", "none", "experts", "gated experts"])
@pytest.mark.parametrize("T,D,centered,plus_one", [(5, 2048, False, True), (8, 2056, True, False), (3, 4096, False, True), (16, 1000, True, True)])
def test_norm_and_token_shift_of_requests_in_another_order(T, D, centered, plus_one, add):
    """Requests whose tokens stand elsewhere in the step than the requests do: sums, norms, mixes and last rows to the bit as the two
    kernels have them, with a gain of 1 + w, and with a shared feed-forward that a gate weights."""
    from simply_amd.kernels import ops

    h = draw((T, D), 1).cuda()
    w, b = (draw((D,), 2 + i, 0.3).bfloat16().cuda() for i in range(2))
    mu = torch.rand((5, D), generator=torch.Generator().manual_seed(4)).bfloat16().cuda()
    state = draw((T + 2, D + 24), 5).cuda()
    row = [(5 * j + 2) % T for j in range(T)] if T % 5 else [(3 * j + 2) % T for j in range(T)]
    meta = torch.tensor([[(j + 3) % (T + 2), row[j], 1, 9] for j in range(T)], dtype=torch.int32).cuda()
    assert sorted(row) == list(range(T)) and row != sorted(row)
    gate = torch.randn((T, 3), generator=torch.Generator().manual_seed(9)).cuda()[:, :1] if add == "gated experts" else None
    y = {"rows": lambda: draw((T, D), 7).bfloat16().cuda(), "none": lambda: None}.get(
        add, lambda: ops.ExpertSums(draw((T * 3, D), 8).cuda(), torch.rand((T, 3)).cuda(), draw((T, D), 6).bfloat16().cuda(), gate, torch.bfloat16))()
    kw = dict(eps=1e-5, mult=0.7, plus_one=plus_one, bias=b if centered else None)
    mine, theirs, one, two = h.clone(), h.clone(), state.clone(), state.clone()
    got = ops.add_next_norm_shift(y, mine, w, mu=mu, tails=one[:, 16:], seq_meta=meta, num_seqs=T, **kw)
    want = ops.token_shift(ops.residual_add_next_norm(y, theirs, w, out_dtype=torch.bfloat16, **kw), mu, two[:, 16:], meta, T, 1)
    assert torch.equal(got, want) and torch.equal(mine, theirs) and torch.equal(one, two)
    assert not torch.equal(one, state) and not any(torch.equal(got[0], got[i]) for i in range(1, T))


@pytest.mark.parametrize("widths, rows", [((1,), (1,)), ((512, 3), (4, 0)), ((300, 257, 1, 64, 7), (5, 8, 1, 2, 3))])
def test_rows_of_block_tables(widths, rows):
    """Rows of one to five block tables from one array: each in its place, all others as they were."""
    from simply_amd.kernels import lib, ops

    g = torch.Generator().manual_seed(sum(widths))
    tables = [torch.randint(-1, 1000, (8, w), generator=g, dtype=torch.int32) for w in widths]
    words, parts, want, at = [], [], [t.clone() for t in tables], 0
    for k, (t, n) in enumerate(zip(tables, rows)):
        places = torch.randperm(8, generator=g, dtype=torch.int32)[:n]
        new = torch.randint(-1, 1000, (n, t.shape[1]), generator=g, dtype=torch.int32)
        want[k][places.long()] = new
        words += [places, new.reshape(-1)]
        parts.append((t.cuda(), at, n))
        at += n * (1 + t.shape[1])
    words = torch.cat(words).cuda()
    ops.table_rows(words, parts)
    for (table, _, _), w in zip(parts, want):
        assert torch.equal(table.cpu(), w)
    with pytest.raises(lib.KernelError):
        ops.table_rows(words[:-1], parts[-1:])
