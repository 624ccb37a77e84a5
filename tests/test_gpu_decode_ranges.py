"""Decoding requests whose lengths differ widely: keys cut into ranges of about equal size, against 64 bits; more requests
than a wave has lanes, requests of several tokens, of one key and without tokens, windows, sinks and slopes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,K,hd,page,window,q_len,extra,lens", [
    (8, 4, 256, 16, None, 1, "", [1, 17, 32, 33, 5000]),
    (16, 8, 256, 16, 700, 1, "", [3, 2000, 700, 701, 40, 1500]),
    (4, 4, 128, 32, None, 3, "", [3, 1600, 64, 95]),
    (8, 2, 128, 16, None, 1, "sinks", [1 + (i * 37) % 90 for i in range(150)] + [3000, 1, 2600]),
    (6, 2, 64, 48, 1900, 2, "slopes", [2000, 5, 0, 1700, 0, 300] * 12),
    (16, 1, 64, 16, None, 1, "", [4097, 1]),
    (1, 1, 64, 16, None, 1, "understated", [140000, 40]),   # more tiles than ranges that are added up, of the least size
])
def test_decode_uneven(H, K, hd, page, window, q_len, extra, lens):
    """Probabilities are rounded to bfloat16 before the values and the result once more, 2^-8 each; 2^-11 of the terms more
    for the 32-bit scores, exponentials and the merging of the ranges."""
    from simply_amd.kernels import ops

    g = torch.Generator().manual_seed(11)
    G = H // K
    blocks = [-(-n // page) for n in lens]
    order = torch.randperm(sum(blocks), generator=g) + 1
    keys, values = torch.randn(sum(blocks) + 1, page, K, hd, generator=g).bfloat16(), torch.randn(sum(blocks) + 1, page, K, hd, generator=g).bfloat16()
    table, at, meta, row = torch.zeros(len(lens), max(blocks), dtype=torch.int32), 0, [], 0
    sinks = torch.randn(H, generator=g) if extra == "sinks" else None
    slopes = torch.rand(H, generator=g) * 0.1 if extra == "slopes" else None
    T = sum(min(q_len, n) for n in lens)
    q = (torch.randn(T, H, hd, generator=g) * hd ** -0.5).bfloat16()
    want, room = torch.zeros(T, H, hd, dtype=torch.float64), torch.zeros(T, H, hd, dtype=torch.float64)
    for i, n in enumerate(lens):
        new = min(q_len, n)
        meta.append((i, row, new, n - new))
        table[i, :blocks[i]] = order[at:at + blocks[i]]
        k, v = (t[table[i, :blocks[i]].long()].reshape(-1, K, hd)[:n].double() for t in (keys, values))
        at += blocks[i]
        for t in range(new):
            pos = n - new + t
            lo = max(0, pos - window + 1) if window else 0
            x = torch.einsum("hd,nhd->hn", q[row + t].double(), k[lo:pos + 1].repeat_interleave(G, 1))
            if slopes is not None:
                x = x - slopes.double()[:, None] * (pos - torch.arange(lo, pos + 1))
            if sinks is not None:
                x = torch.cat([x, sinks.double()[:, None]], 1)
            p = torch.softmax(x, dim=1)[:, :pos + 1 - lo]
            want[row + t] = torch.einsum("hn,nhd->hd", p, v[lo:pos + 1].repeat_interleave(G, 1))
            room[row + t] = torch.einsum("hn,nhd->hd", p, v[lo:pos + 1].repeat_interleave(G, 1).abs())
        row += new
    # pages hold keys in blocks of 16 keys by 32 entries, [entry / 8][key][entry % 8], and values by entry
    kp = keys.permute(0, 2, 1, 3).reshape(-1, K, page // 16, 16, hd // 32, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(-1, K, page, hd)
    vp = values.permute(0, 2, 3, 1)
    dev = lambda t: None if t is None else t.contiguous().cuda()
    kp, vp, table, meta, qd, sinks, slopes = map(dev, (kp, vp, table, torch.tensor(meta, dtype=torch.int32), q.reshape(T, -1), sinks, slopes))
    results = []
    for _ in range(2):
        out = torch.full((T, H * hd), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.paged_attention_decode(qd, kp, vp, table, meta, 0, len(lens), H, window=window, soft_cap=None, max_kv_len=1600 if extra == "understated" else max(lens),
                                   max_q_len=q_len, out=out, num_splits=-1, sinks=sinks, slopes=slopes)
        results.append(out.double().cpu().reshape(T, H, hd))
    assert torch.equal(*results)
    error = (results[0] - want).abs()
    assert (error <= (2.0 ** -8 + 2.0 ** -11) * room + 2.0 ** -8 * want.abs()).all(), (error / room).max()


def test_recorded_steps_follow_the_lengths(tmp_path, monkeypatch):
    """A recorded step that cuts keys into ranges of equal size reads the lengths when it is replayed: 20 decode steps across
    2,560 keys, from where on the longest request has a sixth range (its 81st tile of 32 keys), then requests of like lengths,
    which have a recording of their own, then the first ones' again.  The same bits as without recordings."""
    import tiny
    from simply_amd.config import EngineConfig
    from simply_amd.engine import Executor, StepEntry
    from simply_amd.engine.loading import load_model

    d = dict(tiny.TINY_D, max_position_embeddings=4096, layer_types=["full_attention", "sliding_attention", "full_attention"])
    folder = tiny.write_config_model(d, str(tmp_path / "m"), seed=9, dtype=torch.bfloat16, std=0.15)

    def decode(graphs):
        model, _ = load_model(folder, torch.bfloat16, "cuda:0")
        ex = Executor(model, EngineConfig(activation_dtype="bfloat16", batch_size=7, max_seq_len=4096, max_num_issue_tokens=2048,
                                          total_num_pages=1300, device="cuda:0", use_graphs=graphs))
        out = []
        for lens, steps in (([2550] + [20] * 6, 20), ([2550] * 7, 3), ([2555] + [20] * 6, 3)):
            for i, n in enumerate(lens):
                ex.add_request(i)
                t = tiny.random_tokens(n, d["vocab_size"], i)
                for a in range(0, n, 2048):
                    ex.step([StepEntry(i, t[a:a + 2048])])
            for k in range(steps):
                out.append(ex.step([StepEntry(i, [7 * k + i], [0]) for i in range(7)]).clone())
            for i in range(7):
                ex.finish_request(i)
        return torch.stack(out), ex

    from simply_amd.kernels import ops

    asked, plain = [], ops.paged_attention_decode
    monkeypatch.setattr(ops, "paged_attention_decode", lambda *a, **kw: (asked.append(kw.get("num_splits")), plain(*a, **kw))[1])
    want, _ = decode(False)
    assert -1 in asked and 0 in asked
    got, ex = decode(True)
    assert torch.equal(got, want) and torch.isfinite(want).all()
    assert len(ex._graphs) == 2 and {k[-1] for k in ex._graphs} == {(-1, 0), (0, 0)}, list(ex._graphs)


@pytest.mark.parametrize("H,K,hd,S,keys", [(8, 4, 256, 4, 128), (32, 16, 128, 1, 128), (32, 16, 128, 1, 160), (32, 16, 128, 8, 256),
                                           (16, 8, 128, 2, 224), (8, 4, 64, 4, 256)])
def test_few_keys_errors_no_larger_than_in_ranges(H, K, hd, S, keys):
    """Relative errors against attention in 32 bits, mean of twelve drawings: with the number of ranges that is chosen no larger than
    with a range for every 64 keys.  (Drawing by drawing the two share nearly all roundings: the means are alike to 0.0001 where the
    waves' tiles are, and 0.004 to 0.012 apart where a wave has two tiles; 0.002 lies between.)"""
    from simply_amd.kernels import ops

    P, means = 16, [0.0, 0.0]
    per = -(-keys // P)
    table = torch.arange(S * per, dtype=torch.int32, device="cuda").view(S, per)
    meta = torch.tensor([[i, i, 1, keys - 1] for i in range(S)], dtype=torch.int32, device="cuda")
    kw = dict(window=None, soft_cap=50.0, max_kv_len=keys, max_q_len=1)
    for seed in range(12):
        g = torch.Generator().manual_seed(100 * keys + seed)
        k, v = torch.randn(S * per, K, P, hd, generator=g).bfloat16().cuda(), torch.randn(S * per, K, hd, P, generator=g).bfloat16().cuda()
        q = (torch.randn(S, H * hd, generator=g) * (0.05, 0.1, 0.3)[seed % 3]).bfloat16().cuda()
        want = ops.paged_attention_f32(q.float(), k.float(), v.float(), table, meta, 0, S, H, out=torch.empty(S, H * hd, device="cuda"), **kw).double()
        for i, n in enumerate((0, max(1, min(256 // (S * K), (keys + 63) // 64)))):
            got = ops.paged_attention_decode(q, k, v, table, meta, 0, S, H, num_splits=n, out=torch.empty_like(q), **kw)
            means[i] += float((got.double() - want).norm() / want.norm()) / 12
    assert 1e-4 < means[0] <= 1.002 * means[1] < 1e-2, means
