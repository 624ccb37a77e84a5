"""When a decode step's keys are cut into ranges of equal size, and which steps share a recording.  Host functions: no GPU is
needed, only the built library."""
import pytest
import torch

import tiny
from simply_amd.config import EngineConfig
from simply_amd.engine import StepEntry
from simply_amd.engine.context import StepContext
from simply_amd.engine.loading import load_model
from simply_amd.kernels import build


@pytest.fixture(autouse=True)
def _library():
    if build.find_library() is None:
        pytest.skip("the kernel library has not been built here")


def context(lens):
    return StepContext(dtype=torch.bfloat16, num_tokens=len(lens), positions=None, token_seq=None, seq_meta=None, groups={},
                       request_ids=list(range(len(lens))), seq_slots=list(range(len(lens))), seq_starts=[n - 1 for n in lens],
                       q_lens=[1] * len(lens), cu_q_lens=list(range(len(lens) + 1)))


@pytest.mark.parametrize("lens,window,heads,want", [
    ([8191] + [129] * 63, None, 8, -1),          # more than 128 (request, key head): 16 key heads' worth
    ([8000] * 16 + [80] * 48, None, 8, 0),       # 132
    ([8000] * 16 + [1] * 48, None, 8, -1),       # 128.05
    ([4000] * 33, None, 4, 0),
    ([4000] + [300] * 7, None, 4, -1),           # fewer: 1.5 of 8 requests
    ([4000] * 2 + [1600] + [20] * 5, None, 4, -1),   # 2.43 of 8, below 2.5
    ([4000] * 2 + [2400] + [20] * 5, None, 4, 0),    # 2.63
    ([1505, 10], None, 4, 0),                    # 1.007 of 2
    ([1473] + [10] * 6, None, 4, -1), ([1472] + [10] * 6, None, 4, 0),       # 1,473 keys are 48 tiles and the one they may begin in
    ([8000] + [10] * 6, 700, 4, 0), ([8000] + [10] * 6, 1500, 4, -1), ([8000] + [1500] * 6, 1500, 4, 0),
    ([9000], None, 4, 0)])
def test_rule(lens, window, heads, want):
    ctx = context(lens)
    assert ctx.decode_splits(window, len(lens), heads) == want
    assert ctx.splits_asked == {(window or 0, heads)}


def test_a_recording_s_bound_decides_what_its_kernels_can_do():
    ctx = context([1100] + [10] * 6)
    assert ctx.decode_splits(None, 7, 4) == 0
    ctx = context([1100] + [10] * 6)
    ctx.kv_bound = 2048   # (planned for so many keys, the launch has two ways)
    assert ctx.decode_splits(None, 7, 4) == -1


def recorded(tmp_path, monkeypatch, cpu_ops, asks, batches):
    """The keys under which `Executor._replay` records steps with requests of these lengths, of layers that ask as `asks`."""
    from simply_amd.engine import executor as E

    model, _ = load_model(tiny.write_model("A", str(tmp_path / "A"), std=0.3), torch.float32, "cpu")
    ex = E.Executor(model, EngineConfig(activation_dtype="float32", page_size=16, batch_size=4, max_seq_len=4096,
                                        max_num_issue_tokens=4096, total_num_pages=1024, windowed_num_pages=1024, device="cpu"))
    recordings = []

    class Recording:
        def replay(self):
            recordings[-1] += 1

    def forward(tokens, ctx, views, rows, logits_out=None):
        for window, heads in asks:
            ctx.decode_splits(window, ctx.num_seqs, heads)
        return logits_out

    def record(run):
        run()
        recordings.append(0)
        return Recording()

    monkeypatch.setattr(ex.model, "forward", forward)
    monkeypatch.setattr(ex, "_record", record)
    for lens in batches:
        for i, n in enumerate(lens):
            ex.add_request(i)
            ex.adopt(i, n - 1)
            ex.cache.reserve(i, 0, n - 1)
        T, _, ctx, rows, wants, _ = ex._prepare([StepEntry(i, [1], [0]) for i in range(len(lens))])
        ex._replay(T, ctx, rows)
        for i in range(len(lens)):
            ex.finish_request(i)
    return list(ex._graphs), recordings


LONG, ALIKE = [4000, 20, 20, 20], [4000, 3900, 3000, 4000]


@pytest.mark.parametrize("asks,batches,keys", [
    ([], [LONG, ALIKE, LONG], 1),                                # a 32-bit run, or latent attention alone: no such choice
    ([(None, 2), (8, 2)], [[900, 20, 20, 20], [900, 800, 900, 900], [900, 20, 20, 20]], 1),   # launches with but one way
    ([(8, 2)], [LONG, ALIKE], 1),
    ([(None, 2), (8, 2)], [LONG, ALIKE, LONG, ALIKE], 2)])
def test_recordings(tmp_path, monkeypatch, cpu_ops, asks, batches, keys):
    got, replays = recorded(tmp_path, monkeypatch, cpu_ops, asks, batches)
    assert len(got) == len(replays) == keys, got
    assert sum(replays) == len(batches) - keys
