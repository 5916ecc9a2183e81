"""``plain_linear``: which projections another launch may take the place of, and
FeedForward's call of the others as modules (CPU)."""

from __future__ import annotations

import pytest
import torch

from sophia_amd import decoder, ops
from sophia_amd.config import ModelArgs
from sophia_amd.kda import RuntimeLinear, plain_linear


def _own_hook(m):
    handle = m.register_forward_hook(lambda *a: None)
    return handle.remove


def _global(register):
    def change(m):
        return register(lambda *a: None).remove
    return change


def _forward(m):
    m.forward = lambda x: torch.zeros(x.size(0), m.out_features, dtype=x.dtype)
    return lambda: m.__dict__.pop("forward")


G = torch.nn.modules.module
CHANGES = {"own hook": _own_hook, "forward of its own": _forward,
           "global forward hook": _global(G.register_module_forward_hook),
           "global pre-hook": _global(G.register_module_forward_pre_hook),
           "global backward hook": _global(G.register_module_full_backward_hook),
           "global backward pre-hook": _global(G.register_module_full_backward_pre_hook)}


@pytest.mark.parametrize("name", CHANGES)
def test_plain_linear_sees(name):
    m = RuntimeLinear(32, 16)
    assert plain_linear(m)
    undo = CHANGES[name](m)
    try:
        assert not plain_linear(m)
    finally:
        undo()
    assert plain_linear(m)


def test_plain_linear_takes_no_other_module():
    assert not plain_linear(RuntimeLinear(32, 16, bias=True)) and not plain_linear(torch.nn.Linear(32, 16, bias=False))
    assert not plain_linear(type("Own", (RuntimeLinear,), {})(32, 16))


def test_feed_forward_calls_a_changed_projection(monkeypatch):
    """The projection's own forward, and a global hook, are reached."""
    monkeypatch.setattr(ops, "situ_glu", lambda y, gate, up: y[:, :8])
    m = decoder.FeedForward(ModelArgs(dim=16, ffn_hidden=8))
    x = torch.randn(3, 16)
    seen = []
    handle = G.register_module_forward_hook(lambda mod, args, out: seen.append(mod))
    try:
        m(x)
    finally:
        handle.remove()
    assert seen == [m.gate_up_proj, m.down_proj, m]
    undo = _forward(m.gate_up_proj)
    assert bool((m(x) == 0).all())
    undo()
    assert not bool((m(x) == 0).all())
