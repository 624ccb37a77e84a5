"""Attention of prompts whose heads share a key vector, in groups of units over the matrix cores, against 64 bits: sizes of
keys and values, heads that fill no unit, requests that fill no group, windows, portions behind earlier keys, pages of
other sizes; what lies beside the keys is never a number."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,K,hd,hv,page,window,cases", [
    (16, 1, 576, 512, 16, None, [(0, 323), (37, 65), (500, 5)]),
    (12, 1, 576, 512, 32, 100, [(0, 150), (333, 131)]),
    (32, 1, 544, 512, 16, None, [(2, 130)]),
    (8, 1, 512, 512, 48, 31, [(0, 401), (64, 260)]),
    (4, 1, 320, 256, 16, None, [(0, 1027)]),
    (32, 2, 288, 256, 16, 64, [(77, 129), (0, 1)]),
    (5, 1, 256, 256, 16, None, [(1000, 130)]),
    (16, 1, 192, 128, 16, None, [(0, 257), (1, 255)]),
    (10, 2, 160, 128, 80, 33, [(15, 500)]),
    (16, 16, 128, 128, 16, None, [(0, 200)]),
])
def test_groups(H, K, hd, hv, page, window, cases):
    """Probabilities are rounded to bfloat16 before the values and the result once more: half a spacing each, which is 2^-8
    of a number just above a power of two (7 bits behind the leading one), of every term p |v| and of the result; 2^-12 of
    the terms more for the 32-bit scores and exponentials."""
    from simply_amd.kernels import lib as _lib, ops

    g = torch.Generator().manual_seed(7)
    G, gs = H // K, ops.attention_group_size()
    per = 16 // ops.attention_maps_heads_per_unit(H, K)
    blocks = [-(-(s + n) // page) for s, n in cases]
    order = torch.randperm(sum(blocks), generator=g) + 1
    table = torch.zeros(len(cases), max(blocks) + 1, dtype=torch.int32)
    k_pages = torch.full((sum(blocks) + 1, K, page, hd), float("nan"))
    v_pages = torch.full((sum(blocks) + 1, K, hv, page), float("nan"))
    T = sum(n for _, n in cases) + 3
    q = torch.randn(T, H, hd, generator=g).bfloat16()
    want, room, units, at, first = torch.zeros(T, H, hv, dtype=torch.float64), torch.zeros(T, H, hv, dtype=torch.float64), [], 0, 3
    scale = hd ** -0.5
    for i, (s, n) in enumerate(cases):
        keys, values = torch.randn(s + n, K, hd, generator=g).bfloat16(), torch.randn(s + n, K, hv, generator=g).bfloat16()
        low = max(0, s - window + 1) if window else 0
        for b in range(low // page, blocks[i]):   # (blocks that no row sees any more have no page)
            p = table[i, b] = order[at + b]
            lo, hi = max(b * page, low), min((b + 1) * page, s + n)
            # pages hold keys in blocks of 16 keys by 32 entries, [entry / 8][key][entry % 8], and values by entry
            rows = torch.full((page, K, hd), float("nan"), dtype=torch.bfloat16)
            rows[lo - b * page:hi - b * page] = keys[lo:hi]
            k_pages[p] = rows.permute(1, 0, 2).reshape(K, page // 16, 16, hd // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).reshape(K, page, hd)
            v_pages[p][:, :, lo - b * page:hi - b * page] = values[lo:hi].permute(1, 2, 0).float()
        at += blocks[i]
        pos = torch.arange(s, s + n)[:, None]
        seen = torch.arange(s + n)[None] <= pos
        if window:
            seen &= torch.arange(s + n)[None] > pos - window
        for h in range(H):
            x = q[first:first + n, h].double() @ keys[:, h // G].double().T * scale
            p = torch.softmax(x.masked_fill(~seen, float("-inf")), dim=1)
            want[first:first + n, h] = p @ values[:, h // G].double()
            room[first:first + n, h] = p @ values[:, h // G].double().abs()
        count = -(-(-(-n // per)) // gs) * gs
        units += [(i, first + min(u * per, n), min(n - min(u * per, n), per), s + min(u * per, n)) for u in range(count)]
        first += n
    units = torch.tensor(units, dtype=torch.int32)
    k_pages, v_pages, table, units, qd = (t.cuda() for t in (k_pages.bfloat16(), v_pages.bfloat16(), table, units, q.reshape(T, -1)))
    most = max(s + n for s, n in cases)
    lib = _lib.load()
    assert lib.sa_paged_attention_groups_takes(H, K, hd, hv, page, qd.stride(0), qd.data_ptr())
    assert lib.sa_paged_attention_groups_pays(len(units), H, K, window or 0, most, per)
    out = torch.full((T, H * hv), 7.0, dtype=torch.bfloat16, device="cuda")
    run = lambda: ops.paged_attention_maps_units(qd, k_pages, v_pages, table, units, 0, len(units), H, scale=scale, window=window,
                                                 max_kv_len=most, max_q_len=per, grouped=len(units), out=out)
    got = run().double().cpu().reshape(T, H, hv)
    assert (got[:3] == 7.0).all()   # rows of no unit
    error = (got - want).abs()[3:]
    assert (error <= (2.0 ** -8 + 2.0 ** -12) * room[3:] + 2.0 ** -8 * want[3:].abs()).all(), (error / room[3:]).max()
    again = run().double().cpu().reshape(T, H, hv)
    assert torch.equal(again, got)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("H,hd,hv,window,at", [(16, 576, 512, None, 41), (16, 192, 128, None, 701), (16, 288, 256, 50, 63),
                                               (8, 160, 128, 33, 96), (4, 128, 128, None, 100)])
def test_groups_keep_special_values(H, hd, hv, window, at, bad):
    """A value that is not finite reaches the rows that see its key (rows of a unit together) and changes no bit of others."""
    from simply_amd.kernels import lib as _lib, ops

    g, T, page = torch.Generator().manual_seed(17), 703, 16
    gs, per = ops.attention_group_size(), 16 // ops.attention_maps_heads_per_unit(H, 1)
    pages = -(-T // page)
    table = torch.arange(pages, dtype=torch.int32)[None].cuda()
    k_pages = torch.randn(pages, 1, page, hd, generator=g).bfloat16().cuda()
    v_pages = torch.randn(pages, 1, hv, page, generator=g).bfloat16().cuda()
    q = torch.randn(T, H * hd, generator=g).bfloat16().cuda()
    count = -(-(-(-T // per)) // gs) * gs
    units = torch.tensor([(0, min(u * per, T), min(T - min(u * per, T), per), min(u * per, T)) for u in range(count)],
                         dtype=torch.int32).cuda()
    assert _lib.load().sa_paged_attention_groups_pays(count, H, 1, window or 0, T, per)
    run = lambda: ops.paged_attention_maps_units(q, k_pages, v_pages, table, units, 0, count, H, scale=hd ** -0.5, window=window,
                                                 max_kv_len=T, max_q_len=per, grouped=count).reshape(T, H, hv)
    want = run()
    entry = hv - 19
    v_pages[at // page, 0, entry, at % page] = bad
    got = run()
    row = torch.arange(T, device="cuda")
    sees = (row >= at) & ((row - at) < (window or T))
    of_unit = ((row // per * per + per - 1).clamp(max=T - 1) >= at) & (row // per * per - at < (window or T))
    assert not torch.isfinite(got[sees][:, :, entry]).any()
    same = torch.ones(T, H, hv, dtype=torch.bool, device="cuda")
    same[of_unit, :, entry] = False
    assert torch.isfinite(want).all() and torch.equal(got[same], want[same])
