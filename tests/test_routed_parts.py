"""Which way a feed-forward of routed experts goes, and what a block hands on from it: the decisions alone, on the CPU."""
import types

import pytest
import torch

from simply_amd.kernels import ops
from simply_amd.parts.base import FeedForward, Mixer, knows_expert_sums
from simply_amd.parts.block import PreNormBlock
from simply_amd.parts.ffn import GatedDense, RoutedExperts
from simply_amd.parts.norm import LayerNorm, RMSNorm


class Routed(Exception):
    """The router's launch was asked for."""


@pytest.fixture
def few(monkeypatch):
    """A step of few tokens, whose router's launch says what it was asked for."""

    def route_few(*args, dense=None, **kw):
        raise Routed("beside" if dense is not None else "apart")

    monkeypatch.setattr(ops, "route_few_takes", lambda *a: True)
    monkeypatch.setattr(ops, "route_few_pays", lambda *a: True)
    monkeypatch.setattr(ops, "few_rows_experts", lambda *a: True)
    monkeypatch.setattr(ops, "route_few", route_few)


@pytest.mark.parametrize("size,way", [(None, "apart"), (16, "beside"), (ops.SHARED_BESIDE_MAX, "beside"), (ops.SHARED_BESIDE_MAX + 1, "apart"),
                                      (16384, "apart")])
@pytest.mark.parametrize("gated", [True, False])
def test_a_wide_shared_feed_forward_has_launches_of_its_own(few, size, way, gated):
    part = RoutedExperts(32, 4, 2, 16, shared_size=size, shared_gate=False, gated=gated)
    with pytest.raises(Routed, match=way):
        part.forward(torch.zeros(2, 32))


def test_a_shared_feed_forward_of_another_kind_is_called(few, monkeypatch):
    """One in the place of the part's own, one whose forward() is overridden, one that a program has patched."""

    class Own(GatedDense):
        def forward(self, x, ctx=None, defer_sum=False):
            return super().forward(x, ctx)

    class Other(FeedForward):
        def forward(self, x, ctx):
            return x

    patched = GatedDense(32, 16)
    patched.forward = lambda x, ctx: x
    for shared in (Own(32, 16), Other(), patched):
        part = RoutedExperts(32, 4, 2, 16, shared_size=16, shared_gate=False)
        part.shared = shared
        with pytest.raises(Routed, match="apart"):
            part.forward(torch.zeros(2, 32))


class Plain(RoutedExperts):
    """One that overrides forward() as it was before anything was left to the next norm."""

    def __init__(self):
        super().__init__(32, 4, 2, 16)

    def forward(self, x, ctx):
        return x + 1


class Deferring(RoutedExperts):
    def __init__(self):
        super().__init__(32, 4, 2, 16)

    @knows_expert_sums
    def forward(self, x, ctx, defer_experts=False):
        return "sums" if defer_experts else x + 1


class Adds(RMSNorm):
    @knows_expert_sums
    def after_sum(self, residual, y, mult, out_dtype):
        return y


class AddsTensors(RMSNorm):
    def after_sum(self, residual, y, mult, out_dtype):
        assert isinstance(y, torch.Tensor)
        return y


class OwnSum(PreNormBlock):
    def _add(self, h, y, norm, dtype):
        assert isinstance(y, torch.Tensor)
        return y


class Same(Mixer):
    def forward(self, x, ctx, cache):
        return x


def run(block, part, norm):
    norms = {n: norm(32, 1e-6) for n in ("pre_mixer", "pre_ffn")}
    x = torch.zeros(2, 32)
    return block(Same(), part, norms).forward(x, types.SimpleNamespace(dtype=torch.float32), None, x, norm(32, 1e-6))[1]


def test_experts_sums_are_handed_on_where_all_know_of_them():
    assert run(PreNormBlock, Deferring(), Adds) == "sums"
    for block, part, norm in ((PreNormBlock, Plain(), Adds), (PreNormBlock, Deferring(), AddsTensors), (OwnSum, Deferring(), Adds),
                              (OwnSum, Plain(), AddsTensors)):
        assert torch.equal(run(block, part, norm), torch.ones(2, 32))
    patched = Deferring()   # a program's own function in the place of a part's forward
    patched.forward = lambda x, ctx: x + 1
    assert torch.equal(run(PreNormBlock, patched, Adds), torch.ones(2, 32))
    # the parts here do
    for method in (RoutedExperts.forward, RMSNorm.after_sum, LayerNorm.after_sum, PreNormBlock._add):
        assert method.knows_expert_sums
