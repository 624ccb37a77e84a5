"""Which way a feed-forward of routed experts goes, and what a block hands on from it: the decisions alone, on the CPU."""
import pytest
import torch

from simply_amd.kernels import ops
from simply_amd.parts.ffn import RoutedExperts


class Routed(Exception):
    """The router's launch was asked for."""


@pytest.fixture
def few(monkeypatch):
    """A step of few tokens, whose router's launch says what it was asked for."""

    def route_few(*args, dense=None, **kw):
        raise Routed("beside" if dense is not None else "apart")

    monkeypatch.setattr(ops, "route_few_takes", lambda *a: True)
    monkeypatch.setattr(ops, "few_rows_experts", lambda *a: True)
    monkeypatch.setattr(ops, "route_few", route_few)


@pytest.mark.parametrize("size,way", [(None, "apart"), (16, "beside"), (ops.SHARED_BESIDE_MAX, "beside"), (ops.SHARED_BESIDE_MAX + 1, "apart"),
                                      (16384, "apart")])
@pytest.mark.parametrize("gated", [True, False])
def test_a_wide_shared_feed_forward_has_launches_of_its_own(few, size, way, gated):
    part = RoutedExperts(32, 4, 2, 16, shared_size=size, shared_gate=False, gated=gated)
    with pytest.raises(Routed, match=way):
        part.forward(torch.zeros(2, 32))
