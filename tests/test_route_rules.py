"""The rules that take a call to a kernel of its own, on the CPU: forms that the
kernel refuses must stay on the general path."""

from __future__ import annotations

import pytest
import torch

from sophia_amd import ops
from sophia_amd.kda import RuntimeLinear


def _at_offset(t, elements):
    """t as a contiguous view `elements` into a flat buffer (parameters of one
    flat buffer lie like this)."""
    flat = torch.zeros(t.numel() + elements + 8, dtype=t.dtype)
    flat = flat[(-flat.data_ptr() // t.element_size()) % 8:]   # 16-byte aligned
    view = flat[elements:elements + t.numel()].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("which", ["x", "k_up", "v_up"])
def test_head_linear_rule_looks_at_alignment(which):
    """The per-head kernel needs 16-byte aligned rows and weights."""
    x = torch.randn(5, 2, 128).to(torch.bfloat16)
    w = {"k_up": torch.randn(256, 32).to(torch.bfloat16), "v_up": torch.randn(256, 32).to(torch.bfloat16)}
    with torch.no_grad():
        for offset in (0, 8, 1, 4):
            args = {"x": x, **w}
            args[which] = _at_offset(args[which], offset)
            assert ops.head_linear_takes(args["x"], args["k_up"], args["v_up"]) == (offset % 8 == 0), offset


def test_head_linear_rule_forms():
    """Other types, strides, widths, and calls that ask for more than values."""
    x, w = torch.randn(5, 2, 128).to(torch.bfloat16), torch.randn(256, 32).to(torch.bfloat16)
    with torch.no_grad():
        assert ops.head_linear_takes(x, w, w)
        wide = torch.zeros(5, 264, dtype=torch.bfloat16)
        assert ops.head_linear_takes(wide[:, :256].view(5, 2, 128), w)
        assert not ops.head_linear_takes(torch.zeros(5, 260, dtype=torch.bfloat16)[:, :256].view(5, 2, 128), w)
        assert not ops.head_linear_takes(x.float(), w, w) and not ops.head_linear_takes(x, w.float(), w)
        assert not ops.head_linear_takes(x, w.t().contiguous().t())
        assert not ops.head_linear_takes(x, torch.zeros(256, 48, dtype=torch.bfloat16))
        assert not ops.head_linear_takes(x[:, :, :48], torch.zeros(96, 32, dtype=torch.bfloat16))
    assert not ops.head_linear_takes(x, w.clone().requires_grad_(True))


def test_linear_of_other_tensors():
    """Proxies of a symbolic trace, nested and sparse tensors reach F.linear."""
    torch.manual_seed(0)
    m = RuntimeLinear(64, 32)
    x = torch.randn(3, 64)
    want = torch.nn.functional.linear(x, m.weight)
    assert torch.equal(torch.fx.symbolic_trace(m)(x), want)
    nested = m(torch.nested.nested_tensor([x[:2], x[1:]]))
    assert torch.allclose(nested[0], want[:2], atol=1e-5) and torch.allclose(nested[1], want[1:], atol=1e-5)
    for form in (x.to_sparse(), x.to_sparse_csr()):
        assert torch.allclose(ops.linear(form, m.weight), want, atol=1e-5)
    half = x.to(torch.bfloat16)
    for other in (half.to_sparse(), torch.nested.nested_tensor([half]), half[0]):
        assert ops._few_rows(other, m.weight.detach().to(torch.bfloat16)) is None
    assert ops._few_rows(half, m.weight.detach().to(torch.bfloat16).to_sparse()) is None


@pytest.mark.parametrize("bias", [False, True])
def test_runtime_linear_scripts(bias):
    m = RuntimeLinear(64, 32, bias=bias)
    x = torch.randn(3, 64)
    assert torch.equal(torch.jit.script(m)(x), torch.nn.functional.linear(x, m.weight, m.bias))


def test_row_linear_rule_leaves_what_the_library_does_faster():
    """Shapes measured slower on the few-row kernel than in the library, beside
    ones measured faster (rows, outputs, k)."""
    slower = [(1, 10256, 4096), (8, 12288, 2048), (8, 16384, 3968), (1, 65536, 2048), (8, 8192, 6144), (9, 512, 6144),
              (16, 4112, 3072), (16, 1536, 4608), (17, 4112, 3968), (24, 4096, 2560), (32, 512, 3072),
              (32, 8192, 3968), (32, 6144, 1280), (17, 8192, 8192)]
    faster = [(1, 8384, 1536), (8, 10240, 4096), (8, 1536, 3968), (9, 8192, 2048), (16, 7936, 1536), (16, 4096, 4096),
              (17, 2048, 384), (32, 1536, 2048), (32, 1536, 3968), (24, 4096, 3200), (32, 4096, 1536)]
    assert [c for c in slower if ops.row_linear_gains(*c)] == []
    assert [c for c in faster if not ops.row_linear_gains(*c)] == []
    assert ops.row_linear_gains(32, 7936, 1536, glu=True) and not ops.row_linear_gains(17, 8192, 3968, glu=True)


@pytest.mark.parametrize("form", [ops.row_linear, lambda x, w: ops.row_linear_situ_glu(x, w, 4.0, 25.0)])
def test_row_linear_refuses_operands_that_do_not_fit(form):
    """Called directly: a weight of another k (the kernel would read past it),
    other strides and dimensions, and host tensors raise before any launch."""
    x, w = torch.zeros(4, 96, dtype=torch.bfloat16), torch.zeros(32, 96, dtype=torch.bfloat16)
    for other in (w[:, :64].contiguous(), torch.zeros(32, dtype=torch.bfloat16), w.view(2, 16, 96)):
        with pytest.raises(RuntimeError, match="share k"):
            form(x, other)
    with pytest.raises(RuntimeError, match="share k"):
        form(x.view(2, 2, 96), w)
    with pytest.raises(RuntimeError, match="contiguous"):
        form(x, w.t().contiguous().t())
    with pytest.raises(RuntimeError, match="dense"):
        form(x.t().contiguous().t(), w)
    with pytest.raises(RuntimeError, match="GPU"):
        form(x, w)
