"""The measured cases: what users of the engine have it do, through its public entry points.

Three families of models stand for the engine's parts: Gemma 2 at the sizes of `bench.py` (2B, 9B, 27B layers; dense
attention over pages, behind a window in every other layer), Zenuzen (the gated delta rule, attention with a sink) and
Kolorax (the token-shift recurrence, latent attention, routed experts).  Weights and tokens are drawn from the seed;
keys and states that a pass starts from come from running real prompts.

A pass is one of
  generate  `LMInterface.generate` on a model folder: prompts in, greedy tokens out; then `LMInterface.score_tokens` of
            each prompt with its answer
  decode    `Executor.step` with one token for each request behind the tokens that it holds, logits out
  prompt    a request admitted, its prompt run in portions, logits behind its last token out, the request finished
  mixed     `Executor.step` with a portion of one prompt beside decoding requests, all their logits out
  turn      requests admitted, their prompts run, then a number of given tokens one by one, logits of each out

`exact` computes the same in 64 bits with plain torch on the same weights.
"""
from __future__ import annotations

import json
import math
import os
import tempfile

import torch

from simply_amd import LMInterface, SamplingParams
from simply_amd.config import EngineConfig, config_from_dict
from simply_amd.engine import Executor, StepEntry
from simply_amd.models import DecoderModel

DEVICE = "cuda:0"

GEMMA = {
    "tiny": dict(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, head_dim=16, intermediate_size=128,
                 vocab_size=256, sliding_window=8, query_pre_attn_scalar=16, num_hidden_layers=2),
    "2b": dict(hidden_size=2304, num_attention_heads=8, num_key_value_heads=4, head_dim=256, intermediate_size=9216,
               vocab_size=256000, sliding_window=4096, query_pre_attn_scalar=256, num_hidden_layers=26),
    "9b": dict(hidden_size=3584, num_attention_heads=16, num_key_value_heads=8, head_dim=256, intermediate_size=14336,
               vocab_size=256000, sliding_window=4096, query_pre_attn_scalar=256, num_hidden_layers=42),
    "27b": dict(hidden_size=4608, num_attention_heads=32, num_key_value_heads=16, head_dim=128, intermediate_size=36864,
                vocab_size=256000, sliding_window=4096, query_pre_attn_scalar=144, num_hidden_layers=46),
}
LAYERED = {
    "small": dict(width=1024, heads=8, kv_heads=2, dim=128, ff=4096, vocab=32768),
    "medium": dict(width=2048, heads=16, kv_heads=4, dim=128, ff=8192, vocab=32768),
    "large": dict(width=4096, heads=32, kv_heads=8, dim=128, ff=14336, vocab=32768),
}
TOKEN_BUDGET = 2048     # tokens of a step at most, the engine's default
EXPERTS, CHOSEN, RANK, LATENT, ROT = 16, 2, 64, 512, 64


def listed():
    return [
        # a test-sized model answering three short prompts, the answers scored: the smallest calls, launches and host work
        dict(name="tiny_generate", do="generate", arch="gemma2", size="tiny", layers=2, dtype="float32", batch=3,
             short=5, long=17, new=8),
        # one user's conversation, the next token of a short context
        dict(name="decode_1_at_511", do="decode", arch="gemma2", size="2b", layers=26, dtype="bfloat16", batch=1,
             short=511, long=511),
        # the headline: eight users with long contexts
        dict(name="decode_8_at_8192", do="decode", arch="gemma2", size="2b", layers=26, dtype="bfloat16", batch=8,
             short=8192, long=8192),
        # a full server: many users, contexts of every length, layers of the 9B size
        dict(name="decode_64_ragged", do="decode", arch="gemma2", size="9b", layers=6, dtype="bfloat16", batch=64,
             short=129, long=8191),
        # a prompt in one step
        dict(name="prompt_2048", do="prompt", arch="gemma2", size="2b", layers=26, dtype="bfloat16", tokens=2048,
             portion=2048),
        # a long document whose length nobody rounded, in steps of the engine's token budget
        dict(name="prompt_8191_portions", do="prompt", arch="gemma2", size="2b", layers=26, dtype="bfloat16", tokens=8191,
             portion=2048),
        # continuous batching: the portion of a new prompt beside decoding users, layers of the 27B size
        dict(name="mixed_31_and_1025", do="mixed", arch="gemma2", size="27b", layers=4, dtype="bfloat16", batch=31,
             short=129, long=4095, tokens=1025, before=1024),
        # the 32-bit path, by which logits are checked: a prompt, and decoding
        dict(name="float32_prompt_509", do="prompt", arch="gemma2", size="2b", layers=6, dtype="float32", tokens=509,
             portion=2048),
        dict(name="float32_decode_4", do="decode", arch="gemma2", size="2b", layers=6, dtype="float32", batch=4,
             short=257, long=1023),
        # the two other families on a prompt, and answering short prompts
        dict(name="zenuzen_prompt_2048", do="prompt", arch="zenuzen", size="medium", layers=8, dtype="bfloat16",
             tokens=2048, portion=2048),
        dict(name="kolorax_prompt_2047", do="prompt", arch="kolorax", size="medium", layers=8, dtype="bfloat16",
             tokens=2047, portion=2048),
        dict(name="kolorax_turn_8", do="turn", arch="kolorax", size="medium", layers=8, dtype="bfloat16", batch=8,
             short=33, long=201, new=16),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    largest = max(_seconds(c) for c in listed())
    while True:
        case = _draw(rng)
        if _seconds(case) <= largest:
            return case


def _draw(rng):
    kind = rng.choice(["generate", "decode", "decode", "decode", "prompt", "prompt", "mixed", "f32_prompt", "f32_decode",
                       "other_prompt", "other_prompt", "other_turn", "other_turn"])
    if kind == "generate":
        short = _log_uniform(rng, 1, 24)
        return dict(do="generate", arch="gemma2", size="tiny", layers=2, dtype="float32", batch=rng.randint(1, 4),
                    short=short, long=rng.randint(short, 48), new=rng.randint(4, 16))
    if kind in ("decode", "mixed"):
        size = rng.choice(["2b", "9b", "27b"])
        layers = rng.randint(4, 26) if size == "2b" else rng.randint(2, 6) if size == "9b" else rng.randint(2, 4)
        short, long = sorted((_log_uniform(rng, 16, 8192), _log_uniform(rng, 16, 8192)))
        case = dict(do=kind, arch="gemma2", size=size, layers=layers, dtype="bfloat16", batch=_log_uniform(rng, 1, 64),
                    short=short, long=long)
        while sum(_lengths(case)) > 130000:
            case["batch"] = max(1, case["batch"] // 2)
        if kind == "mixed":
            # (the portion is run again and again: it ends before the window moves)
            case["batch"] = min(case["batch"], 31)
            case["tokens"], case["before"] = _log_uniform(rng, 16, 2000), rng.choice([0, _log_uniform(rng, 16, 2048)])
        return case
    if kind == "prompt":
        size = rng.choice(["2b", "9b", "27b"])
        layers = rng.randint(4, 26) if size == "2b" else rng.randint(2, 6) if size == "9b" else rng.randint(2, 4)
        return dict(do="prompt", arch="gemma2", size=size, layers=layers, dtype="bfloat16",
                    tokens=_log_uniform(rng, 16, 8192), portion=rng.choice([512, 1024, 2048]))
    if kind == "f32_prompt":
        return dict(do="prompt", arch="gemma2", size="2b", layers=rng.randint(2, 6), dtype="float32",
                    tokens=_log_uniform(rng, 16, 1024), portion=rng.choice([256, 2048]))
    if kind == "f32_decode":
        short, long = sorted((_log_uniform(rng, 16, 2048), _log_uniform(rng, 16, 2048)))
        return dict(do="decode", arch="gemma2", size="2b", layers=rng.randint(2, 6), dtype="float32",
                    batch=_log_uniform(rng, 1, 16), short=short, long=long)
    arch, size = rng.choice(["zenuzen", "kolorax"]), rng.choice(["small", "medium", "large"])
    layers = rng.randint(4, 8) if size != "large" else 4
    if kind == "other_prompt":
        return dict(do="prompt", arch=arch, size=size, layers=layers, dtype="bfloat16",
                    tokens=_log_uniform(rng, 16, 4096), portion=rng.choice([512, 2048]))
    short, long = sorted((_log_uniform(rng, 8, 512), _log_uniform(rng, 8, 512)))
    return dict(do="turn", arch=arch, size=size, layers=layers, dtype="bfloat16", batch=_log_uniform(rng, 1, 16),
                short=short, long=long, new=rng.randint(4, 24))


def _lengths(case):
    """Tokens that each of the requests holds: spread evenly over their logarithm, odd in between.  (A decode pass is
    run at the same position again and again; with a length that is not 14 modulo the page size of 16 the last key
    behind the window of 4,096 does not end its page, so that the engine still holds it then.)"""
    n, lo, hi = case["batch"], case["short"], case["long"]
    if lo == hi:
        return [lo + (lo % 16 == 14)] * n
    return [min(hi | 1, int(round(lo * (hi / lo) ** (i / max(n - 1, 1)))) | 1) for i in range(n)]


def _config(case):
    """The model's config.json."""
    if case["arch"] == "gemma2":
        return dict(GEMMA[case["size"]], architectures=["Gemma2ForCausalLM"], num_hidden_layers=case["layers"],
                    rms_norm_eps=1e-6, rope_theta=10000.0, attn_logit_softcapping=50.0, final_logit_softcapping=30.0,
                    tie_word_embeddings=True, max_position_embeddings=8448, hidden_activation="gelu_pytorch_tanh",
                    torch_dtype=case["dtype"])
    s = LAYERED[case["size"]]
    H, d = s["heads"], s["dim"]
    layers = []
    for i in range(case["layers"]):
        if case["arch"] == "zenuzen":
            mlp = {"kind": "dense", "ff": s["ff"]}
            if i % 4 == 3:
                layers.append({"type": "attention", "mlp": mlp, "mixer": {
                    "heads": H, "kv_heads": s["kv_heads"], "dim": d, "vdim": d, "scale": d ** -0.5, "v_mix": True,
                    "rot": {"dims": d // 2, "base": 1000000.0}}})
            else:
                layers.append({"type": "delta", "mlp": mlp, "mixer": {
                    "heads": H, "kv_heads": H // 2, "dim": d, "vdim": d, "conv": 4}})
        else:
            ff = s["ff"] // 4
            mlp = {"kind": "moe", "expert": {"ff": ff, "limit": 7.0}, "shared": {"ff": ff, "limit": 7.0},
                   "router": {"experts": EXPERTS, "top": CHOSEN, "groups": {"count": 4, "keep": 2}}}
            if i % 4 == 3:
                layers.append({"type": "latent_attention", "mlp": mlp, "mixer": {
                    "heads": H, "dim": d, "rot_dim": ROT, "vdim": d, "kv_rank": LATENT, "scale": (d + ROT) ** -0.5,
                    "rot": {"dims": ROT, "base": 50000.0}}})
            else:
                layers.append({"type": "wkv", "mlp": mlp, "mixer": {"heads": H, "dim": d, "rank": RANK}})
    c = {"vocab": s["vocab"], "width": s["width"], "residual_mult": 0.7, "norm": {"eps": 1e-5}, "layers": layers}
    if case["arch"] == "zenuzen":
        return dict(c, architecture="Zenuzen")
    c = dict(c, architecture="Kolorax", embedding={"scale": 1.0})
    if case["layers"] >= 4:
        c["loop"] = {"start": 2, "stop": 4, "times": 2}
    return c


# --------------------------------------------------------------------------- inputs


class _Weights:
    """Draws the weights of a model by name, on the GPU, in the activation dtype."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)
        self.dtype, self.w = dtype, {}

    def matrix(self, name, rows, cols, std=0.02):
        self.w[name] = torch.empty(rows, cols, dtype=self.dtype, device=DEVICE).normal_(0.0, std, generator=self.gen)

    def vector(self, name, shape, std=0.1, mean=0.0):
        v = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(mean, std, generator=self.gen)
        self.w[name] = v.to(self.dtype)

    def uniform(self, name, shape, lo, hi, through=lambda v: v):
        v = torch.empty(shape, dtype=torch.float32, device=DEVICE).uniform_(lo, hi, generator=self.gen)
        self.w[name] = through(v).to(self.dtype)


def _weights(case, cfg, seed):
    """Every tensor of the model folder.  Matrices and norm scales as the engine's random-weights mode draws them;
    where a recurrence's memory hangs on a vector, values as trained models of the kind have them.  Zenuzen and Kolorax
    have no norm of their own behind the embedding, so its rows are of unit size; Kolorax, whose sublayers add to the
    stream as they are, has the matrices that write to it scaled down with the depth, as such models are initialised."""
    d = _Weights(seed, getattr(torch, case["dtype"]))
    if case["arch"] == "gemma2":
        D, H, K, hd, F = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                          "intermediate_size"))
        # the tiny model's larger weights give continuations that are not one token
        std = 0.02 if case["size"] != "tiny" else 0.2
        d.matrix("model.embed_tokens.weight", cfg["vocab_size"], D, std)
        for i in range(case["layers"]):
            p = f"model.layers.{i}."
            for name, rows, cols in (("self_attn.q_proj", H * hd, D), ("self_attn.k_proj", K * hd, D),
                                     ("self_attn.v_proj", K * hd, D), ("self_attn.o_proj", D, H * hd),
                                     ("mlp.gate_proj", F, D), ("mlp.up_proj", F, D), ("mlp.down_proj", D, F)):
                d.matrix(p + name + ".weight", rows, cols, std)
            for name in ("input", "post_attention", "pre_feedforward", "post_feedforward"):
                d.vector(p + name + "_layernorm.weight", D)
        d.vector("model.norm.weight", D)
        return d.w
    D, H, dim, V = cfg["width"], LAYERED[case["size"]]["heads"], LAYERED[case["size"]]["dim"], cfg["vocab"]
    d.matrix("embed", V, D, 1.0)
    one = dict(std=0.1, mean=1.0)
    last = 0.02 if case["arch"] == "zenuzen" else 0.02 / math.sqrt(2 * case["layers"])
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        if layer["type"] == "attention":
            G = m["kv_heads"]
            for name, rows, cols in (("q", H * dim, D), ("k", G * dim, D), ("v", G * dim, D), ("g", H * dim, D),
                                     ("o", D, H * dim)):
                d.matrix(p + name, rows, cols)
            d.vector(p + "sink", H, 1.0)
            d.vector(p + "vmix", (), 0.1, 0.5)
        elif layer["type"] == "delta":
            G = m["kv_heads"]
            for name, rows in (("q", G * dim), ("k", G * dim), ("v", H * dim)):
                d.matrix(p + name, rows, D)
                d.matrix(p + name + ".conv", rows, m["conv"], 0.5)
            for name, rows, cols in (("a", H, D), ("b", H, D), ("g", H * dim, D), ("o", D, H * dim)):
                d.matrix(p + name, rows, cols)
            # half-lives from a few tokens to thousands: rates in [1, 16], steps in [0.001, 0.1] before the softplus
            d.uniform(p + "A_log", H, 1.0, 16.0, torch.log)
            d.uniform(p + "dt_bias", H, math.log(1e-3), math.log(1e-1), lambda v: torch.log(torch.expm1(torch.exp(v))))
            d.vector(p + "norm", dim, **one)
        elif layer["type"] == "wkv":
            for s in "rkvgw":
                d.uniform(p + "mu." + s, D, 0.0, 1.0)
            for name, rows, cols in (("r", H * dim, D), ("k", H * dim, D), ("v", H * dim, D), ("g", H * dim, D),
                                     ("w1", RANK, D), ("w2", H * dim, RANK)):
                d.matrix(p + name, rows, cols)
            d.matrix(p + "o", D, H * dim, last)
            d.uniform(p + "w0", H * dim, -6.0, 0.5)     # decays from 0.998 to 0.19 a token
            d.vector(p + "u", (H, dim), 0.3)
            d.vector(p + "norm", H * dim, **one)
        else:
            for name, rows, cols in (("q", H * (dim + ROT), D), ("dkv", LATENT + ROT, D), ("uk", H * dim, LATENT),
                                     ("uv", H * dim, LATENT), ("g", H * dim, D)):
                d.matrix(p + name, rows, cols)
            d.matrix(p + "o", D, H * dim, last)
            d.vector(p + "dkv.norm", LATENT, **one)
        p, mlp = f"l{i}.mlp.", layer["mlp"]
        if mlp["kind"] == "dense":
            d.matrix(p + "up", mlp["ff"], D)
            d.matrix(p + "down", D, mlp["ff"])
        else:
            d.matrix(p + "router", EXPERTS, D)
            for e in [f"e{j}." for j in range(EXPERTS)] + ["shared."]:
                ff = mlp["expert"]["ff"]
                d.matrix(p + e + "gate", ff, D)
                d.matrix(p + e + "up", ff, D)
                d.matrix(p + e + "down", D, ff, last)
        for name in ("norm1", "norm2"):
            d.vector(f"l{i}.{name}", D, **one)
            if case["arch"] == "kolorax":
                d.vector(f"l{i}.{name}.b", D)
    if cfg.get("loop"):
        d.matrix("loop.in", D, 2 * D)
        d.vector("loop.step", (cfg["loop"]["times"], D))
    d.vector("final.norm", D, **one)
    if case["arch"] == "kolorax":
        d.vector("final.norm.b", D)
    d.matrix("head", V, D)
    return d.w


def _tokens(case, cfg, seed):
    """For each request of the case its tokens: what it holds before the pass and what the pass brings."""
    gen = torch.Generator()
    gen.manual_seed(seed + 1000003)
    vocab = cfg.get("vocab_size", cfg.get("vocab"))
    new = {"generate": 0, "decode": 1, "prompt": 0, "mixed": 1, "turn": case.get("new", 0)}[case["do"]]
    lengths = [case["tokens"]] if case["do"] == "prompt" else [n + new for n in _lengths(case)]
    if case["do"] == "mixed":
        lengths.append(case["before"] + case["tokens"])
    return [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in lengths]


def _portions(tokens, at_most):
    return [tokens[i:i + at_most] for i in range(0, len(tokens), at_most)]


def prepare(case, seed):
    cfg = _config(case)
    weights, tokens = _weights(case, cfg, seed), _tokens(case, cfg, seed)
    if case["do"] == "generate":
        from safetensors.torch import save_file

        with tempfile.TemporaryDirectory() as folder:
            save_file({k: v.cpu().contiguous() for k, v in weights.items()}, os.path.join(folder, "model.safetensors"),
                      metadata={"format": "pt"})
            with open(os.path.join(folder, "config.json"), "w") as f:
                json.dump(cfg, f)
            lm = LMInterface(folder, activation_dtype=case["dtype"], batch_size=case["batch"],
                             max_seq_len=case["long"] + case["new"] + 2)
        params = SamplingParams(temperature=0.0, max_decode_steps=case["new"], ignore_eos=True)
        return dict(case=case, lm=lm, tokens=tokens, params=params)
    model = DecoderModel(config_from_dict(cfg).model_spec())
    model.load_tensors(weights)
    del weights
    longest = max(len(t) for t in tokens)
    pages = sum(-(-len(t) // 16) + 1 for t in tokens) + 8
    ex = Executor(model, EngineConfig(activation_dtype=case["dtype"], batch_size=len(tokens), max_seq_len=longest + 16,
                                      max_num_issue_tokens=case.get("portion", TOKEN_BUDGET), total_num_pages=pages,
                                      intermediate_steps=1))
    state = dict(case=case, ex=ex, tokens=tokens)
    if case["do"] in ("decode", "mixed"):
        # what the requests hold, run as the engine runs it: portions of several requests fill a step's budget
        held = [t[:-1] for t in tokens[:case["batch"]]]
        if case["do"] == "mixed":
            held.append(tokens[-1][:case["before"]])
        for i in range(len(tokens)):
            ex.add_request(i)
        _run_prompts(ex, held)
        state["starts"] = [len(t) for t in held]
    return state


def _run_prompts(ex, prompts, wanted=False):
    """The requests' prompts, a step's token budget at a time; logits behind their last tokens, if wanted."""
    done, logits, budget = [0] * len(prompts), [None] * len(prompts), ex.config.issue_budget
    while any(d < len(p) for d, p in zip(done, prompts)):
        entries, room = [], budget
        for i, p in enumerate(prompts):
            n = min(len(p) - done[i], room)
            if n > 0:
                last = done[i] + n == len(p)
                entries.append(StepEntry(i, p[done[i]:done[i] + n], [n - 1] if wanted and last else []))
                done[i] += n
                room -= n
        out = ex.step(entries)
        ends = [e.request_id for e in entries if e.want]
        for row, i in enumerate(ends):
            logits[i] = out[row]
    return logits


def run(state):
    case = state["case"]
    if case["do"] == "generate":
        outs = state["lm"].generate(state["tokens"], sampling_params=state["params"])
        scores = [state["lm"].score_tokens(o.input_token_ids + o.output_token_ids) for o in outs]
        return {"tokens": torch.tensor([o.output_token_ids for o in outs]), "scores": torch.tensor(sum(scores, []))}
    ex, tokens = state["ex"], state["tokens"]
    if case["do"] == "prompt":
        ex.add_request(0)
        for part in _portions(tokens[0], case["portion"])[:-1]:
            ex.step([StepEntry(0, part)])
        part = _portions(tokens[0], case["portion"])[-1]
        logits = ex.step([StepEntry(0, part, [len(part) - 1])])
        ex.finish_request(0)
        return logits
    if case["do"] in ("decode", "mixed"):
        entries = [StepEntry(i, t[s:], [len(t) - s - 1], s) for i, (t, s) in enumerate(zip(tokens, state["starts"]))]
        return ex.step(entries)
    new = case["new"]
    for i in range(len(tokens)):
        ex.add_request(i)
    out = [torch.stack(_run_prompts(ex, [t[:-new] for t in tokens], wanted=True))]
    for k in range(new):
        # (the steps' logits share a buffer: who keeps them copies them)
        out.append(ex.step([StepEntry(i, [t[len(t) - new + k]], [0]) for i, t in enumerate(tokens)]).clone())
    for i in range(len(tokens)):
        ex.finish_request(i)
    return torch.stack(out)


# --------------------------------------------------------------------------- what a pass cannot do without


def _steps(case):
    """The steps of a pass: per step a list of (tokens, tokens held before, logits wanted)."""
    if case["do"] == "generate":
        L = _lengths(case)
        return [[(n, 0, 1) for n in L]] + [[(1, n + k, 1) for n in L] for k in range(case["new"] - 1)]
    if case["do"] == "decode":
        return [[(1, n, 1) for n in _lengths(case)]]
    if case["do"] == "mixed":
        return [[(1, n, 1) for n in _lengths(case)] + [(case["tokens"], case["before"], 1)]]
    if case["do"] == "prompt":
        T, P = case["tokens"], case["portion"]
        return [[(min(P, T - a), a, int(a + P >= T))] for a in range(0, T, P)]
    L = _lengths(case)
    total, steps, at = sum(L), [], 0
    for _ in range(-(-total // TOKEN_BUDGET)):
        step, room, before = [], TOKEN_BUDGET, 0
        for n in L:
            begin, end = max(before, at), min(before + n, at + room)
            if end > begin:
                step.append((end - begin, begin - before, int(end == before + n)))
            before += n
        steps.append(step)
        at += room
    return steps + [[(1, n + k, 1) for n in L] for k in range(case["new"])]


def _seen(start, n, window):
    """Keys that n tokens behind `start` others look at, all together, and the keys that one of them needs at all."""
    pairs = sum(min(start + j + 1, window) for j in range(n)) if window else n * start + n * (n + 1) // 2
    return pairs, start + n if window is None else min(start + n, window + n - 1)


def work(case):
    cfg, e = _config(case), 2 if case["dtype"] == "bfloat16" else 4
    D, V = cfg.get("hidden_size", cfg.get("width")), cfg.get("vocab_size", cfg.get("vocab"))
    order = list(range(case["layers"]))
    if cfg.get("loop"):
        order = [0, 1, 2, 3, 2, 3] + order[4:]
    nbytes = flops = 0
    for step in _steps(case):
        T, R = sum(s[0] for s in step), sum(s[2] for s in step)
        nbytes += T * D * e + R * V * 4 + (V * D * e if R else 0)
        flops += 2 * R * V * D
        for run_at, i in enumerate(order):
            if case["arch"] == "gemma2":
                H, K, hd, F = (cfg[k] for k in ("num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size"))
                params, touched = D * (2 * H + 2 * K) * hd + 3 * D * F, 0
                kv, qk, window = 2 * K * hd, 4 * H * hd, cfg["sliding_window"] if i % 2 == 0 else None
                state = rec = 0
            else:
                s, layer = LAYERED[case["size"]], cfg["layers"][i]
                H, d = s["heads"], s["dim"]
                kv = qk = state = rec = 0
                window, touched = None, 0
                if layer["type"] == "attention":
                    params = D * d * (3 * H + 2 * s["kv_heads"])
                    kv, qk = 2 * s["kv_heads"] * d, 4 * H * d
                elif layer["type"] == "delta":
                    params = D * d * (H // 2 * 2 + 3 * H) + 2 * D * H
                    state, rec = 2 * 4 * H * d * d, 8 * H * d * d
                elif layer["type"] == "wkv":
                    params = 5 * D * H * d + 2 * RANK * D
                    state, rec = 2 * 4 * H * d * d, 6 * H * d * d
                else:
                    params = D * H * (d + ROT) + D * (LATENT + ROT) + 2 * LATENT * H * d + 2 * D * H * d
                    kv, qk = LATENT + ROT, 2 * H * (2 * d + ROT)
                if layer["mlp"]["kind"] == "dense":
                    params += 2 * D * layer["mlp"]["ff"]
                else:
                    one = 3 * D * layer["mlp"]["expert"]["ff"]
                    params += EXPERTS * D + one
                    touched = one * EXPERTS * (1.0 - (1.0 - CHOSEN / EXPERTS) ** T)
                    flops += 2 * T * CHOSEN * one
            nbytes += (params + touched) * e
            flops += 2 * T * params + T * rec
            for n, start, _ in step:
                pairs, keys = _seen(start, n, window)
                nbytes += (keys + n) * kv * e + state
                flops += pairs * qk
        if cfg.get("loop"):
            nbytes += 2 * D * D * e
            flops += cfg["loop"]["times"] * 4 * T * D * D
    return {"bytes": int(nbytes), "flops": int(flops)}


def _seconds(case):
    w = work(case)
    return w["bytes"] / 6e12 + w["flops"] / (1e15 if case["dtype"] == "bfloat16" else 1e14)


def tolerance(case):
    """About four times what the engine shows against `exact`."""
    if case["do"] == "generate":
        return {"rel": 2e-6, "differ": 0.02}    # (greedy tokens differ only where two logits meet in the last bits)
    if case["dtype"] == "float32":
        return {"rel": 2e-5}                    # 4e-6 to 5e-6
    if case["arch"] == "gemma2":
        return {"rel": 4e-2}                    # 0.007 to 0.0095
    if case["arch"] == "zenuzen":
        return {"rel": 3e-2}                    # 0.0065 to 0.0077
    # 0.003 to 0.004 for a prompt's last token, but 0.03 where rounding moves that token to another expert in one layer
    # (0.3 of the root mean square on the worst of a turn's logits, 0.01 to 0.013 over all of them)
    return {"rel": 1e-1}


# --------------------------------------------------------------------------- the same in 64 bits


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, dims, base):
    """x [T, heads, size]: the first `dims` entries in pairs (i, i + dims / 2)."""
    half = dims // 2
    freq = float(base) ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims)
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None, None] * freq
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., dims:]], -1)


def _attend(q, k, v, scale, cap=None, window=None, sink=None):
    """q [T, H, dk], k [T, G, dk], v [T, G, dv]: causal, head h reads key head h // (H / G)."""
    T, H, _ = q.shape
    rep = H // k.shape[1]
    out = torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=q.device)
    pos = torch.arange(T, device=q.device)
    for a in range(0, T, 2048):     # rows in blocks, keys up to the block's end
        b = min(T, a + 2048)
        low = max(0, a - window + 1) if window else 0
        diff = pos[a:b, None] - pos[None, low:b]
        hidden = diff < 0
        if window:
            hidden = hidden | (diff >= window)
        for h in range(H):
            s = q[a:b, h] @ k[low:b, h // rep].T * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(hidden, float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink[h].expand(b - a, 1)], 1)
            out[a:b, h] = torch.softmax(s, -1)[:, :b - low] @ v[low:b, h // rep]
    return out


class _Exact:
    """A model in 64 bits; whole sequences."""

    def __init__(self, case, seed):
        self.case, self.cfg = case, _config(case)
        self.w = _weights(case, self.cfg, seed)

    def __getitem__(self, name):
        return self.w[name].double()

    def times(self, x, name):
        return x @ self[name].T

    def sequences(self, sequences, places):
        """Logits at `places` (one list per sequence) of each sequence, layer by layer."""
        with torch.no_grad():
            x = [self.embed(torch.tensor(t, device=DEVICE)) for t in sequences]
            sizes = [len(t) for t in sequences]
            x = torch.cat(x)
            x = self.layers(x, sizes)
            first, rows = 0, []
            for n, at in zip(sizes, places):
                rows += [first + p for p in at]
                first += n
            return self.head(x[torch.tensor(rows, device=DEVICE)])

    def each(self, sizes, fn, *tensors):
        """fn on every sequence's rows."""
        return torch.cat([fn(*part) for part in zip(*(t.split(sizes) for t in tensors))])

    # Gemma 2
    def embed(self, t):
        if self.case["arch"] == "gemma2":
            table = self.w["model.embed_tokens.weight"]
            return table[t].double() * math.sqrt(self.cfg["hidden_size"])
        return self.w["embed"][t].double()

    def head(self, x):
        if self.case["arch"] == "gemma2":
            z = self.times(_rms(x, 1e-6) * (1 + self["model.norm.weight"]), "model.embed_tokens.weight")
            return 30.0 * torch.tanh(z / 30.0)
        return self.times(self.normed(x, "final.norm"), "head")

    def normed(self, x, name):
        if self.case["arch"] == "zenuzen":
            return _rms(x, 1e-5) * self[name]
        return _rms(x - x.mean(-1, keepdim=True), 1e-5) * self[name] + self[name + ".b"]

    def layers(self, x, sizes):
        if self.case["arch"] == "gemma2":
            for i in range(self.case["layers"]):
                x = self.gemma_layer(x, sizes, i)
            return x
        loop, first_values, x0 = self.cfg.get("loop"), {}, x
        order = [(i, None) for i in range(self.case["layers"])]
        if loop:
            turn = [[(2, t), (3, None)] for t in range(loop["times"])]
            order = order[:2] + sum(turn, []) + order[4:]
        for i, begins in order:
            if begins is not None:
                x = self.times(torch.cat([x, x0], -1), "loop.in") + self["loop.step"][begins]
            layer, p = self.cfg["layers"][i], f"l{i}."
            if self.case["arch"] == "zenuzen":
                mixer = self.sink_attention if layer["type"] == "attention" else self.delta
                x = x + 0.7 * self.normed(mixer(x, sizes, p + "mix.", layer["mixer"], first_values), p + "norm1")
                x = x + 0.7 * self.normed(self.times(torch.relu(self.times(x, p + "mlp.up")) ** 2, p + "mlp.down"), p + "norm2")
            else:
                mixer = self.wkv if layer["type"] == "wkv" else self.latent
                x = x + 0.7 * mixer(self.normed(x, p + "norm1"), sizes, p + "mix.", layer["mixer"])
                x = x + 0.7 * self.experts(self.normed(x, p + "norm2"), p + "mlp.")
        return x

    def gemma_layer(self, x, sizes, i):
        c, p = self.cfg, f"model.layers.{i}."
        H, K, hd = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        norm = lambda y, name: _rms(y, 1e-6) * (1 + self[p + name + "_layernorm.weight"])
        y = norm(x, "input")
        q, k, v = (self.times(y, p + f"self_attn.{s}_proj.weight").view(-1, n, hd) for s, n in (("q", H), ("k", K), ("v", K)))
        window = c["sliding_window"] if i % 2 == 0 else None
        scale = c["query_pre_attn_scalar"] ** -0.5
        o = self.each(sizes, lambda q, k, v: _attend(_rotate(q, hd, 10000.0), _rotate(k, hd, 10000.0), v, scale, 50.0, window),
                      q, k, v)
        x = x + norm(self.times(o.reshape(-1, H * hd), p + "self_attn.o_proj.weight"), "post_attention")
        y = norm(x, "pre_feedforward")
        gate, up = self.times(y, p + "mlp.gate_proj.weight"), self.times(y, p + "mlp.up_proj.weight")
        y = self.times(torch.nn.functional.gelu(gate, approximate="tanh") * up, p + "mlp.down_proj.weight")
        return x + norm(y, "post_feedforward")

    # Zenuzen
    def sink_attention(self, x, sizes, p, m, first_values):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.times(x, p + s).view(-1, n, d) for s, n in (("q", H), ("k", G), ("v", G)))
        if "v" in first_values:
            lam = self[p + "vmix"]
            v = (1 - lam) * v + lam * first_values["v"]
        else:
            first_values["v"] = v
        turned = lambda z: _rms(_rotate(z, m["rot"]["dims"], m["rot"]["base"]), 1e-5)
        o = self.each(sizes, lambda q, k, v: _attend(turned(q), turned(k), v, m["scale"], sink=self[p + "sink"]), q, k, v)
        return self.times(o.reshape(-1, H * d) * torch.sigmoid(self.times(x, p + "g")), p + "o")

    def delta(self, x, sizes, p, m, _):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]

        def short(name):
            def conv(y):
                taps = self[p + name + ".conv"]
                n = taps.shape[1]
                y = torch.nn.functional.pad(y, (0, 0, n - 1, 0))
                return sum(y[j:y.shape[0] - n + 1 + j] * taps[:, j] for j in range(n))
            return torch.nn.functional.silu(self.each(sizes, conv, self.times(x, p + name)))

        unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
        q, k, v = unit(short("q").view(-1, G, d)) * d ** -0.5, unit(short("k").view(-1, G, d)), short("v").view(-1, H, d)
        q, k = (z.repeat_interleave(H // G, 1) for z in (q, k))
        beta = torch.sigmoid(self.times(x, p + "b"))
        step = torch.nn.functional.softplus(self.times(x, p + "a") + self[p + "dt_bias"])
        decay = torch.exp(-torch.exp(self[p + "A_log"]) * step)

        def rule(q, k, v, beta, decay):
            S, out = torch.zeros(H, d, d, dtype=q.dtype, device=q.device), torch.empty_like(v)
            for t in range(q.shape[0]):
                S.mul_(decay[t][:, None, None])
                u = beta[t][:, None] * (v[t] - (k[t][:, :, None] * S).sum(1))
                S.addcmul_(k[t][:, :, None], u[:, None, :])
                out[t] = (q[t][:, :, None] * S).sum(1)
            return out

        o = _rms(self.each(sizes, rule, q, k, v, beta, decay), 1e-5) * self[p + "norm"]
        gate = torch.nn.functional.silu(self.times(x, p + "g"))
        return self.times(o.reshape(-1, H * d) * gate, p + "o")

    # Kolorax
    def wkv(self, h, sizes, p, m):
        H, d = m["heads"], m["dim"]
        before = self.each(sizes, lambda y: torch.cat([torch.zeros_like(y[:1]), y[:-1]]), h)
        mix = {s: h + (before - h) * self[p + "mu." + s] for s in "rkvgw"}
        r, k, v = (self.times(mix[s], p + s).view(-1, H, d) for s in "rkv")
        a = torch.exp(-torch.exp(self.times(torch.tanh(self.times(mix["w"], p + "w1")), p + "w2") + self[p + "w0"]))
        u = self[p + "u"]

        def rule(r, k, v, a):
            S, out = torch.zeros(H, d, d, dtype=r.dtype, device=r.device), torch.empty_like(v)
            for t in range(r.shape[0]):
                # (the bonus term of a token's own key and value, then the state behind it)
                out[t] = (r[t][:, :, None] * S).sum(1) + (r[t] * u * k[t]).sum(-1, keepdim=True) * v[t]
                S.mul_(a[t][:, :, None]).addcmul_(k[t][:, :, None], v[t][:, None, :])
            return out

        o = _rms(self.each(sizes, rule, r, k, v, a.view(-1, H, d)), 1e-5).reshape(-1, H * d)
        return self.times(o * self[p + "norm"] * torch.nn.functional.silu(self.times(mix["g"], p + "g")), p + "o")

    def latent(self, h, sizes, p, m):
        H, d = m["heads"], m["dim"]
        q, down = self.times(h, p + "q").view(-1, H, d + ROT), self.times(h, p + "dkv")
        c = _rms(down[:, :LATENT], 1e-5) * self[p + "dkv.norm"]
        ku, v = self.times(c, p + "uk").view(-1, H, d), self.times(c, p + "uv").view(-1, H, d)
        base = m["rot"]["base"]

        def attend(q, kr, ku, v):
            q = torch.cat([q[..., :d], _rotate(q[..., d:], ROT, base)], -1)
            kr = _rotate(kr[:, None], ROT, base).expand(-1, H, -1)
            return _attend(q, torch.cat([ku, kr], -1), v, m["scale"])

        o = self.each(sizes, attend, q, down[:, LATENT:], ku, v).reshape(-1, H * d)
        return self.times(o * torch.sigmoid(self.times(h, p + "g")), p + "o")

    def expert(self, h, p):
        g, u = self.times(h, p + "gate").clamp(max=7.0), self.times(h, p + "up").clamp(-7.0, 7.0)
        return self.times(g * torch.sigmoid(1.702 * g) * (u + 1), p + "down")

    def experts(self, h, p):
        s = torch.softmax(self.times(h, p + "router"), -1)
        best = s.view(-1, 4, EXPERTS // 4).amax(-1).topk(2, -1).indices
        allowed = torch.zeros(h.shape[0], 4, dtype=torch.bool, device=h.device).scatter_(1, best, True)
        weight, chosen = s.masked_fill(~allowed.repeat_interleave(EXPERTS // 4, 1), -1.0).topk(CHOSEN, -1)
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20)
        y = self.expert(h, p + "shared.")
        for e in range(EXPERTS):
            at, which = (chosen == e).nonzero(as_tuple=True)
            if at.numel():
                y.index_add_(0, at, self.expert(h[at], f"{p}e{e}.") * weight[at, which][:, None])
        return y


def exact(case, seed):
    model = _Exact(case, seed)
    tokens = _tokens(case, model.cfg, seed)
    if case["do"] == "generate":
        out_tokens, scores = [], []
        for t in tokens:
            t = list(t)
            for _ in range(case["new"]):
                t.append(int(model.sequences([t], [[len(t) - 1]])[0].argmax()))
            out_tokens.append(t[-case["new"]:])
            z = torch.log_softmax(model.sequences([t], [list(range(len(t) - 1))]), -1)
            scores.append(z.gather(1, torch.tensor(t[1:], device=DEVICE)[:, None])[:, 0])
        return {"tokens": torch.tensor(out_tokens), "scores": torch.cat(scores)}
    if case["do"] == "turn":
        n = case["new"] + 1
        z = model.sequences(tokens, [list(range(len(t) - n, len(t))) for t in tokens])
        return z.view(len(tokens), n, -1).transpose(0, 1).contiguous()
    return model.sequences(tokens, [[len(t) - 1] for t in tokens])
