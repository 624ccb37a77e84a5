"""The norm in front of a time-mixing part in a step with one token of every request: who gets it, and who the norm by itself.  The
kernel's entry is replaced; what it computes is tested on the GPU."""
import types

import torch

from simply_amd.kernels import ops
from simply_amd.parts.block import PreNormBlock
from simply_amd.parts.norm import LayerNorm, RMSNorm
from simply_amd.parts.wkv import WKV, ShiftedNorm


def step(requests=3, width=32):
    mixer = WKV(width, 2, 16, 8, 1e-5)
    mixer.mu = torch.rand(5, width)
    ctx = types.SimpleNamespace(dtype=torch.bfloat16, max_q_len=1, num_tokens=requests, num_seqs=requests,
                                positions=types.SimpleNamespace(is_cuda=True), seq_meta=torch.zeros(requests, 4, dtype=torch.int32))
    cache = types.SimpleNamespace(write=True, state=torch.zeros(requests, mixer.state_words + width))
    return mixer, ctx, cache


def made(norm_class, width=32):
    norm = norm_class(width, 1e-6)
    norm.scale = torch.ones(width, dtype=torch.bfloat16)
    return norm


def test_a_norm_that_adds_what_it_norms_takes_the_next_norm_by_itself(monkeypatch):
    """A block whose sums run in its own norms' kernel, in front of one that offers its norm with the token shift: one launch."""
    mixer, ctx, cache = step()
    before, behind = made(RMSNorm), made(RMSNorm)
    offered = mixer.norm_of_step(behind, ctx, cache)
    assert isinstance(offered, ShiftedNorm)
    calls = []
    monkeypatch.setattr(ops, "add_rmsnorm", lambda y, residual, **kw: calls.append(kw) or "normed")
    monkeypatch.setattr(ops, "rmsnorm", lambda *args: calls.append("apart"))
    y = torch.zeros(3, 32, dtype=torch.bfloat16)
    assert before.add_into(torch.zeros(3, 32), y, offered, torch.bfloat16) == "normed"
    assert len(calls) == 1 and calls[0]["next_weight"] is behind.scale and calls[0]["next_eps"] == behind.eps


class OtherForward(RMSNorm):
    def forward(self, x, out_dtype):
        return x


class OtherSum(RMSNorm):
    def after_sum(self, residual, y, mult, out_dtype):
        return residual


class OtherMixer(WKV):
    def forward(self, x, ctx, cache):
        return x


def patched(part, **methods):
    for name, method in methods.items():
        setattr(part, name, method)
    return part


def test_norms_and_mixers_with_methods_of_their_own_get_what_they_got_before():
    mixer, ctx, cache = step()
    for norm_class in (RMSNorm, LayerNorm):
        assert isinstance(mixer.norm_of_step(made(norm_class), ctx, cache), ShiftedNorm)
    other = lambda *args: None
    for norm in (made(OtherForward), made(OtherSum), patched(made(RMSNorm), after_sum=other), patched(made(LayerNorm), forward=other)):
        assert mixer.norm_of_step(norm, ctx, cache) is norm
    norm = made(RMSNorm)
    another = OtherMixer(32, 2, 16, 8, 1e-5)
    assert another.norm_of_step(norm, ctx, cache) is norm
    assert patched(mixer, forward=other).norm_of_step(norm, ctx, cache) is norm
    block = PreNormBlock(step()[0], None, {"pre_mixer": norm})
    assert isinstance(block.norm_of_step(ctx, cache), ShiftedNorm)
    assert patched(block, forward=other).norm_of_step(ctx, cache) is norm
