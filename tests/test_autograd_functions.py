"""The autograd functions that only move gradients, on the CPU."""

from __future__ import annotations

import torch

from sophia_amd import ops


def test_unbind_heads_second_derivative():
    """Gradients that are parts of one row and have a history (create_graph):
    the derivative reaches dq, dk and dv alike, as through x.unbind(2)."""
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(2, 5, 3, 2, 128, generator=gen, dtype=torch.float64, requires_grad=True)
    buf = torch.randn(2, 5, 3, 2, 128, generator=gen, dtype=torch.float64, requires_grad=True)
    weight = torch.randn(2, 5, 3, 2, 128, generator=gen, dtype=torch.float64)
    for unbind in (ops.UnbindHeads.apply, lambda t: t.unbind(2)):
        dx, = torch.autograd.grad(unbind(x), x, buf.unbind(2), create_graph=True)
        assert torch.equal(dx, buf)
        d_buf, = torch.autograd.grad((dx * weight).sum(), buf)
        assert torch.equal(d_buf, weight)
