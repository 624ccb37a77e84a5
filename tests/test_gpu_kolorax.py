"""Kolorax on the GPU: every kernel against the plain implementation's function for its mechanism, the mixers and
feed-forwards as parts, and the engine (whole prompts, token-by-token decoding, portions down to two tokens, unequal
requests together in a tight pool, long decoding, recorded decode steps, greedy generation through the scheduler, trace
replay as a child process) against the plain implementation, in 32-bit and in bfloat16."""
import pytest
import torch

import kolorax_cases as cases
import kolorax_mechanisms as mech
import plain_kolorax as plain
from simply_amd.engine import StepEntry
from simply_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(autouse=True)
def _lib(gpu_lib):
    return gpu_lib


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("body", [mech.layer_norm_after_a_sum, mech.token_shift, mech.low_rank_decay, mech.recurrence_with_bonus,
                                  mech.head_norm_and_gate, mech.clamped_products, mech.clamped_experts,
                                  mech.queries_with_a_gate_per_entry])
def test_kernel(body, dtype):
    body(ops, DEV, dtype)


def test_router():
    mech.router_of_groups(ops, DEV)


def test_products():
    mech.products_of_several_inputs(ops, DEV)
    mech.wide_products_in_32_bit(ops, DEV)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("body", [mech.layer_norm_part, mech.pass_input_part, mech.wkv_part, mech.latent_part, mech.routed_part])
def test_part(body, dtype):
    body(DEV, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_parts_at_other_sizes(dtype):
    mech.wkv_part(DEV, dtype, sizes=(24, 1, 4, 9), length=9, cuts=([9], [2, 2, 2, 2, 1], [1] * 9))   # a rank above the heads
    mech.latent_part(DEV, dtype, sizes=(24, 2, 4, 6, 5, 8), dims=4, length=12, cuts=([12], [5, 2, 5], [1] * 12))
    mech.routed_part(DEV, dtype, experts=4, top=4, groups=(1, 1), shared=None, T=9)
    mech.routed_part(DEV, dtype, experts=4, top=2, groups=(2, 1), ff=64, shared=64, width=64, T=200)


def test_parts_at_aligned_sizes():
    """Sizes in multiples of 32 and 64 in pages of 16 keys, bfloat16, 300 tokens: whatever fast kernels the parts choose at
    such sizes, whole, decoding behind a long portion, and in portions of 17."""
    cuts = ([300], [268] + [1] * 32, [17] * 17 + [11])
    mech.wkv_part(DEV, torch.bfloat16, sizes=(128, 4, 64, 32), length=300, cuts=cuts, std=0.1)
    mech.wkv_part(DEV, torch.bfloat16, sizes=(256, 2, 128, 64), length=300, cuts=cuts, std=0.08)
    mech.latent_part(DEV, torch.bfloat16, sizes=(128, 4, 64, 32, 64, 96), page_size=16, length=300, cuts=cuts, std=0.1)
    mech.latent_part(DEV, torch.bfloat16, sizes=(128, 16, 64, 64, 32, 192), page_size=16, length=300, cuts=cuts, std=0.08)


@pytest.mark.parametrize("dtype", DTYPES)
def test_far_keys(dtype):
    mech.far_keys(DEV, dtype)
    mech.far_keys(DEV, dtype, page_size=4, T=130)


def test_far_keys_on_the_matrix_cores():
    mech.far_keys(DEV, torch.bfloat16, sizes=(64, 4, 32, 32, 32, 96), std=0.1, T=500)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["mixed", "units", "no_loop", "only_wkv", "aligned"])
def test_cuts_match_plain(tmp_path, name, dtype):
    cases.cuts_match_plain(tmp_path, DEV, name, dtype, length=45 if name != "aligned" else 70)


def test_mistakes_would_show(tmp_path):
    cases.mistakes_would_show(tmp_path, DEV)


@pytest.mark.parametrize("name, dtype", [("mixed", "float32"), ("aligned", "bfloat16")])
def test_layers_match_plain(tmp_path, name, dtype):
    cases.layers_match_plain(tmp_path, DEV, name, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["mixed", "only_wkv", "aligned"])
def test_batches_match_alone(tmp_path, name, dtype):
    cases.batches_match_alone(tmp_path, DEV, name, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_portions_and_pages_of_sixteen(tmp_path, dtype):
    cases.cuts_match_plain(tmp_path, DEV, "aligned", dtype, length=171, page_size=16)
    cases.batches_match_alone(tmp_path / "b", DEV, "aligned", dtype, page_size=16)


@pytest.mark.parametrize("length", [150, 301])
def test_prompts_with_the_choices_that_they_made(tmp_path, monkeypatch, length):
    """A router that is close moves a token to another expert, and its logits far more than the rounding of everything else,
    which would hide a mistake of that size.  So the plain implementation takes the engine's own choices, and so does a run of
    the kernels' plain references with bfloat16 rounding, which says how far off roundings alone are: the engine's median row
    is off by at most 1.5 times that run's, its worst row by twice that run's.  And the choices are the plain implementation's
    own but for a few (one in twenty), each between scores within the same distance of one another."""
    import torch_ops

    d = cases.write_model("aligned", str(tmp_path / "m"), dtype=torch.bfloat16)
    w, cfg = cases.plain_weights(d, "bfloat16")
    tokens = cases.random_tokens(length, cfg["vocab"], 7)
    taken, routed = [], ops.routed_experts

    def run(device):
        ex = cases.make_executor(d, device, "bfloat16", page_size=16, num_pages=64, max_len=320)
        ex.add_request("r")
        return ex.step([StepEntry("r", tokens, list(range(length)))])

    with monkeypatch.context() as mp:
        mp.setattr(ops, "routed_experts", lambda x, experts, *a, **kw: (taken.append(experts.cpu()), routed(x, experts, *a, **kw))[1])
        got = run(DEV)
    with monkeypatch.context() as mp:
        left = list(taken)

        def route_choice(logits, top, scale, **kw):
            experts = left.pop(0)
            s = torch.softmax(logits.float(), -1).gather(1, experts.long())
            return experts, s / (s.sum(-1, keepdim=True) + 1e-20) * scale

        for name in torch_ops.STAND_INS:
            mp.setattr(ops, name, getattr(torch_ops, name))
        mp.setattr(ops, "route_choice", route_choice)
        rounded = run("cpu")
        assert not left
    rows, free, others = [r for e in taken for r in e.tolist()], plain.choose, []

    def choose(z, router):
        chosen, s = rows.pop(0), torch.softmax(z, -1)
        own = [e for e, _ in free(z, router)]
        if set(own) != set(chosen):
            best = lambda es: max(float(s[e]) for e in es)   # (of what one choice has and the other lacks)
            others.append(best(set(own) - set(chosen)) / best(set(chosen) - set(own)) - 1.0)
        total = sum(s[e] for e in chosen) + 1e-20
        return [(e, s[e] / total) for e in chosen]

    choices = len(rows)
    monkeypatch.setattr(plain, "choose", choose)
    want = plain.forward(w, cfg, tokens)
    assert not rows
    off, alone = cases.rel_rows(got, want), cases.rel_rows(rounded, want)
    print(length, *(float(f(x)) for x in (off, alone) for f in (torch.median, torch.max)), choices, len(others), max(others, default=0.0))
    assert off.median() <= 1.5 * alone.median() and off.max() <= 2.0 * alone.max()
    assert len(others) <= choices // 20 and all(m <= 2.0 * float(alone.max()) for m in others), (len(others), max(others))


@pytest.mark.parametrize("seed", range(12))
def test_drawn_configurations(tmp_path, seed):
    cases.drawn_configuration_runs(tmp_path, DEV, seed)


@pytest.mark.parametrize("seed", [1, 4, 7, 10])
def test_drawn_configurations_bfloat16(tmp_path, seed):
    cases.drawn_configuration_runs(tmp_path, DEV, seed, "bfloat16")


@pytest.mark.parametrize("name, dtype", [("mixed", "float32"), ("aligned", "bfloat16")])
def test_long_decoding(tmp_path, name, dtype):
    cases.long_decoding(tmp_path, DEV, name, dtype, steps=150, page_size=16)


@pytest.mark.parametrize("name, dtype, page_size", [("mixed", "float32", 4), ("mixed", "bfloat16", 4), ("aligned", "bfloat16", 16)])
def test_recorded_decode_steps(tmp_path, name, dtype, page_size):
    """Decode-only steps are recorded in a HIP graph and replayed: three requests decode together for 40 steps, and each
    step's logits are those of the same step run eagerly by a second engine (states advance exactly once)."""
    d = cases.write_model(name, str(tmp_path / "m"))
    V = plain.load(d)[1]["vocab"]
    prompts = {r: cases.random_tokens(n, V, 70 + n) for r, n in (("a", 9), ("b", 3), ("c", 14))}
    follow = {r: cases.random_tokens(40, V, 90 + len(p)) for r, p in prompts.items()}
    engines = [cases.make_executor(d, DEV, dtype, page_size=page_size, num_pages=64, batch=4, max_len=64, graphs=g)
               for g in (True, False)]
    for ex in engines:
        for r, p in prompts.items():
            ex.add_request(r)
        ex.step([StepEntry(r, p, []) for r, p in prompts.items()])
    for k in range(40):
        outs = [ex.step([StepEntry(r, [follow[r][k]], [0]) for r in prompts]).clone() for ex in engines]
        torch.testing.assert_close(outs[0], outs[1], rtol=0, atol=0)


def test_greedy_generation(tmp_path):
    cases.greedy_generation(tmp_path, DEV, "mixed", "float32")


def test_greedy_generation_bfloat16_runs(tmp_path):
    """The serving path as it is used: bfloat16, recorded decode steps, several steps in a row on the device."""
    from simply_amd.engine.llm import LMInterface
    from simply_amd.sampling import SamplingParams

    d = cases.write_model("aligned", str(tmp_path / "m"), dtype=torch.bfloat16)
    lm = LMInterface(d, activation_dtype="bfloat16", batch_size=4, max_seq_len=128, device=DEV)
    prompts = [cases.random_tokens(n, 256, n) for n in (5, 33, 17, 2, 60)]
    outs = lm.generate(prompts, sampling_params=SamplingParams(temperature=0.0, max_decode_steps=24))
    again = lm.generate(prompts, sampling_params=SamplingParams(temperature=0.0, max_decode_steps=24))
    assert all(len(o.output_token_ids) == 24 for o in outs)
    assert [o.output_token_ids for o in outs] == [o.output_token_ids for o in again]


def test_trace_replay_child_process(tmp_path):
    """bin/trace_run as a user starts it: a folder whose config.json leaves the decays' ranks to the tensors, steps on
    standard input, logits in files; two live requests."""
    import json
    import os
    import subprocess

    import numpy as np

    d = cases.write_model("mixed", str(tmp_path / "m"), dtype=torch.bfloat16)
    path = os.path.join(d, "config.json")
    raw = json.load(open(path))
    for l in raw["layers"]:
        l["mixer"].pop("rank", None)
    json.dump(raw, open(path, "w"))
    w, cfg = plain.load(d)
    tx, ty = cases.random_tokens(30, cfg["vocab"], 5), cases.random_tokens(12, cfg["vocab"], 6)
    wx, wy = plain.forward(w, cfg, tx), plain.forward(w, cfg, ty)
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": tx[:17], "want": [0, 16]}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": tx[17:19], "want": []}, {"id": "y", "tokens": ty[:11], "want": [10]}],
              "end": []},
             {"step": 2, "entries": [{"id": "y", "tokens": ty[11:], "want": [0]}, {"id": "x", "tokens": tx[19:], "want": [10]}],
              "end": ["x", "y"]}]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = tmp_path / "out"
    r = subprocess.run([os.path.join(root, "bin", "trace_run"), "--model", d, "--dtype", "float32", "--out", str(out),
                        "--max-tokens", "128"], input="\n".join(json.dumps(s) for s in steps) + "\n", text=True,
                       capture_output=True, timeout=600)
    assert r.returncode == 0, r.stderr
    assert [l for l in r.stdout.splitlines() if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    got = [torch.from_numpy(np.fromfile(out / f"{i}.f32", dtype="<f4").reshape(n, -1)) for i, n in ((0, 2), (1, 1), (2, 2))]
    for g, want in zip(got, (wx[[0, 16]], wy[[10]], torch.stack([wy[11], wx[29]]))):
        assert float(cases.rel_rows(g, want).max()) <= cases.BOUND_F32
