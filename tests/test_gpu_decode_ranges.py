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
