"""Time mixing with a token shift, data-dependent decays and a bonus for the current token.

Every one of the five streams r, k, v, g, w reads a mix of the token's input h and the one before it, h' (zeros before a
sequence's first token), h + (h' - h) * mu_s.  r, k, v (heads x size) and the gate are projections of their mixes; the
decay per head and key channel is a = exp(-exp(W_2 tanh(W_1 mix_w) + w_0)).  Per head, with S [size, size] from zero,

    o_t = (S_(t-1) + diag(u) k_t v_t^T)^T r_t,      S_t = diag(a_t) S_(t-1) + k_t v_t^T

and each head's o is divided by its root mean square, multiplied by a weight (one entry per head and channel) and by
silu(gate), then projected.  A request's state is S and its last h, one float32 row of a state slot; mixes, decays, S and
the norm are 32-bit, the projections read and give the activation type."""
from __future__ import annotations

import torch

from ..kernels import ops
from ..registry import MIXERS
from .base import MixedRows, Mixer, Norm, ParamSpec, StateNeed, as_product_weight, is_method, knows_expert_sums
from .linear_state import channel_decay_state
from .norm import LayerNorm, RMSNorm


class ShiftedNorm(Norm):
    """The norm in front of the mixer, together with the mixer's token shift: for a step with one token of every request."""

    fuses_sum = True

    def __init__(self, norm, mixer, ctx, cache):
        self.norm, self.mixer, self.ctx, self.cache = norm, mixer, ctx, cache

    @property
    def by_itself(self):
        return self.norm

    def forward(self, x, out_dtype):
        return self.norm.forward(x, out_dtype)

    @knows_expert_sums
    def after_sum(self, residual, y, mult, out_dtype):
        n, m = self.norm, self.mixer
        rows = None
        if out_dtype == torch.bfloat16:
            rows = ops.add_next_norm_shift(y, residual, n.scale, eps=n.eps, plus_one=getattr(n, "scale_plus_one", False), mult=mult,
                                           bias=getattr(n, "bias", None), mu=m.mu, tails=self.cache.state[:, m.state_words:],
                                           seq_meta=self.ctx.seq_meta, num_seqs=self.ctx.num_seqs)
        return MixedRows(rows) if rows is not None else n.after_sum(residual, y, mult, out_dtype)


@MIXERS.register("wkv")
class WKV(Mixer):
    STREAMS = ("r", "k", "v", "g", "w")

    def __init__(self, hidden_size: int, num_heads: int, head_dim: int, decay_rank: int, norm_eps: float):
        self.hidden_size, self.num_heads, self.head_dim = int(hidden_size), int(num_heads), int(head_dim)
        self.decay_rank, self.norm_eps = int(decay_rank), float(norm_eps)
        self.state_words = self.num_heads * self.head_dim * self.head_dim
        self.mu = self.in_proj = self.decay_out = self.decay_base = self.bonus = self.norm = self.o_proj = None

    def param_specs(self):
        D, H, d, R = self.hidden_size, self.num_heads, self.head_dim, self.decay_rank
        vec = dict(role="vector", init="norm")
        specs = {"mu_" + s: ParamSpec((D,), **vec) for s in self.STREAMS}
        specs.update({s + "_proj": ParamSpec((H * d, D)) for s in "rkvg"})
        specs.update(decay_in=ParamSpec((R, D)), decay_out=ParamSpec((H * d, R)), decay_base=ParamSpec((H * d,), **vec),
                     bonus=ParamSpec((H, d), **vec), norm=ParamSpec((H * d,), **vec), o_proj=ParamSpec((D, H * d)))
        return specs

    def load(self, tensors):
        t = tensors
        self.mu = torch.stack([t["mu_" + s].to(t["mu_r"].dtype) for s in self.STREAMS]).contiguous()
        # r, k, v, the gate and the decay's first factor: products whose blocks of outputs read blocks of the mixes, run
        # as one where the decay's rank is not larger than the heads
        rkvg = [t[s + "_proj"] for s in "rkvg"]
        self.decay_in = None if self.decay_rank <= rkvg[0].shape[0] else as_product_weight(t["decay_in"])
        self.in_proj = ops.SectionedWeight(rkvg + ([t["decay_in"]] if self.decay_in is None else []))
        self.decay_out = as_product_weight(t["decay_out"])
        self.decay_base, self.norm = t["decay_base"].contiguous(), t["norm"].contiguous()
        self.bonus = t["bonus"].reshape(-1).contiguous()
        self.o_proj = as_product_weight(t["o_proj"])

    def cache_need(self):
        return StateNeed((self.state_words + self.hidden_size,), torch.float32)   # S, then the last token's h

    def norm_of_step(self, norm, ctx, cache):
        """`norm`, or in a step with one token of every request that norm with the token shift in its kernel.  (A norm or a mixer
        whose methods are others than the ones here is left alone, be it by its class or by what a program put in their place.)"""
        known = norm.fuses_sum and is_method(norm.after_sum, RMSNorm.after_sum, LayerNorm.after_sum) \
            and is_method(norm.forward, RMSNorm.forward, LayerNorm.forward)
        if known and is_method(self.forward, WKV.forward) and cache.write and ctx.dtype == torch.bfloat16 and ctx.max_q_len == 1 \
                and ctx.num_tokens == ctx.num_seqs and ctx.positions.is_cuda:
            return ShiftedNorm(norm, self, ctx, cache)
        return norm

    def forward(self, x, ctx, cache):
        if not cache.write:
            raise RuntimeError("wkv: a recurrent state cannot be read through another entry's cache")
        D, H, d = self.hidden_size, self.num_heads, self.head_dim
        C = H * d
        if isinstance(x, MixedRows):
            mixes = x.rows
        else:
            mixes = ops.token_shift(x, self.mu, cache.state[:, self.state_words:], ctx.seq_meta, ctx.num_seqs, ctx.max_q_len)
        if self.decay_in is None:
            proj = ops.gemm_sections(mixes, self.in_proj)                             # [T, r | k | v | gate | decay's factor]
            low = proj[:, 4 * C:]
            if ctx.max_q_len == 1 and ops.wkv_token_takes(proj, self.decay_out, d, cache.state, 4 * C):
                z = ops.wkv_token(proj, (0, C, 2 * C, 3 * C, 4 * C), self.decay_out, self.decay_base, self.bonus, self.norm,
                                  self.norm_eps, H, d, cache.state, ctx.seq_meta, ctx.num_seqs)
                return ops.gemm(z, self.o_proj)
        else:
            proj, low = ops.gemm_sections(mixes[:, :4 * D], self.in_proj), ops.gemm(mixes[:, 4 * D:], self.decay_in)
        decay = ops.low_rank_decay(low, self.decay_out, self.decay_base)
        o = channel_decay_state(proj, (0, C, 2 * C), 1.0, decay, H, d, d, cache.state, ctx, bonus=self.bonus)
        z = ops.gated_heads(o, proj[:, 3 * C:4 * C], H, d, kind=ops.GATE_SILU, weight=self.norm, eps=self.norm_eps,
                            out_dtype=ctx.dtype)
        return ops.gemm(z, self.o_proj)
