"""torch.compile's tracing of the training path, on the CPU: Dynamo and the fake
kernels need no GPU.  A backend that keeps the graph and stops there shows
whether forward and backward trace without a break (the values are compared on
the GPU, test_gpu_compile.py)."""

from __future__ import annotations

import pytest
import torch

from sophia_amd import ops


class _Traced(Exception):
    pass


def _trace(fn, *args):
    """Graphs that torch.compile(fullgraph=True) hands to its backend for fn."""
    graphs = []

    def backend(gm, example_inputs):
        graphs.append(gm)

        def stop(*_):
            raise _Traced
        return stop

    torch._dynamo.reset()
    with pytest.raises(_Traced):
        torch.compile(fn, backend=backend, fullgraph=True)(*args)
    return graphs


@pytest.mark.parametrize("fused", [True, False])
def test_chunk_kda_with_gradients_traces_to_one_graph(fused):
    """q, k, v as views of one fused row (the mixer's) and as tensors of their own."""
    x = torch.randn(1, 70, 3, 2, 128).to(torch.bfloat16).requires_grad_(True)
    g = torch.randn(1, 70, 2, 128, requires_grad=True)
    beta = torch.randn(1, 70, 2, requires_grad=True)
    a_log, bias = torch.randn(2, requires_grad=True), torch.randn(256, requires_grad=True)

    def core(x, g, beta):
        q, k, v = x.unbind(2) if fused else (t.clone() for t in x.unbind(2))
        o, _ = ops.chunk_kda(q, k, v, g, beta, A_log=a_log, dt_bias=bias, use_gate_in_kernel=True,
                             use_beta_sigmoid_in_kernel=True, use_qk_l2norm_in_kernel=True)
        return o

    assert len(_trace(core, x, g, beta)) == 1


def test_mixer_with_gradients_traces_to_one_graph(monkeypatch):
    from sophia_amd import kda
    from sophia_amd.config import ModelArgs
    monkeypatch.setattr(kda, "_require_gpu", lambda x: None)
    torch.manual_seed(0)
    mixer = kda.SophiaKDA(ModelArgs(dim=256, num_heads=2, use_cache=False)).train()
    x = torch.randn(2, 70, 256, requires_grad=True)
    assert len(_trace(mixer, x)) == 1
