"""Which requests of a step the recurrences with decays per channel take in pieces: every row once, and the results of the
recurrence over all of them.  With the kernels' plain references."""
import pytest
import torch

from simply_amd.engine.context import StepContext


@pytest.mark.parametrize("lens,pieces", [
    ([1], 0), ([127], 0), ([128], 1), ([1, 63, 127], 0), ([1, 63, 64, 128], 2), ([79] * 8, 0), ([64] * 7 + [80], 8),
    ([63] + [64] * 6 + [80], 0), ([1, 1, 200, 130], 2), ([5] * 9 + [127], 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_channel_decays(monkeypatch, cpu_ops, lens, pieces, dtype):
    from simply_amd.kernels import ops
    from simply_amd.parts.linear_state import channel_decay_state

    lens, H, dk, dv = sorted(lens), 2, 4, 3
    T, cu = sum(lens), [sum(lens[:i]) for i in range(len(lens) + 1)]
    meta = torch.tensor([(i, cu[i], n, 0) for i, n in enumerate(lens)], dtype=torch.int32)
    ctx = StepContext(dtype=dtype, num_tokens=T, positions=None, token_seq=None, seq_meta=meta, groups={},
                      request_ids=list(range(len(lens))), seq_slots=list(range(len(lens))), seq_starts=[0] * len(lens),
                      q_lens=lens, cu_q_lens=cu)
    gen = torch.Generator().manual_seed(T)
    proj = torch.randn(T, H * (2 * dk + dv) + 2, generator=gen).to(dtype)
    gates, state = torch.rand(T, H * dk, generator=gen), torch.randn(len(lens), H * dk * dv, generator=gen)
    columns, seen, plain = (0, H * dk, 2 * H * dk), [], ops.linear_chunks

    def chunks(*args, **kw):
        seen.append(args[11])
        return plain(*args, **kw)

    monkeypatch.setattr(ops, "linear_chunks", chunks)
    s1, s2 = state.clone(), state.clone()
    want = ops.linear_state(proj, *columns, 0.5, gates, False, H, dk, dv, False, s1, meta, len(lens))
    got = channel_decay_state(proj, columns, 0.5, gates, H, dk, dv, s2, ctx)
    assert seen == ([pieces] if pieces and dtype == torch.bfloat16 else [])
    assert torch.equal(got, want) and torch.equal(s1, s2)
