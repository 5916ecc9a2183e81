"""The few-row projection kernels (sophia_row_linear, sophia_row_linear_situ_glu)
and the rule that takes a call to them, against float64 on the same bf16 inputs.

Tolerance: the sums are fp32 over bf16 products (exact in fp32) and rounded to
bf16 once, 2^-9 of each value; the fp32 sum of k terms adds at most
k 2^-24 sum |x w|, far below it here.  max|y - ref| <= 2^-8 max|ref|; the
activation's own rounding (fp32, a few ulp) is covered by the same bound."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


def _data(rows, n, k, seed=0):
    g = torch.Generator().manual_seed(seed + rows + n + k)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16)
    return x, w


def _close(y, ref):
    return float((y.double().cpu() - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())


# one k-step; k short of, at and past one batch of steps per wavefront with 4,
# 8 and 16 wavefronts, and past one batch of 16; one and two tiles per
# work-group, an odd tile left over; half tiles (to 8 rows) by one, two and five,
# an odd number of k-steps
@pytest.mark.parametrize("n,k", [(16, 32), (48, 96), (2048, 128), (32, 1024), (32, 1056), (1536, 2048), (16, 2080),
                                 (1536, 3968), (16, 8192), (16 * 257, 64), (16 * 511, 1536), (16 * 524, 96),
                                 (16 * 513, 3616), (2048, 384)])
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32])
def test_row_linear_matches_float64(rows, n, k):
    from sophia_amd import ops
    dev = _dev()
    x, w = _data(rows, n, k)
    wide = torch.full((rows, k + 24), 9.0, dtype=torch.bfloat16)
    wide[:, 8:8 + k] = x
    y = ops.row_linear(wide.to(dev)[:, 8:8 + k], w.to(dev))
    assert y.shape == (rows, n) and _close(y, x.double() @ w.double().t())


@pytest.mark.parametrize("hidden,k", [(8, 32), (24, 160), (3968, 1536), (8 * 259, 64), (8 * 519, 96)])
@pytest.mark.parametrize("rows,cap", [(1, 4.0), (8, 3.0), (16, 3.0), (19, 4.0), (32, 4.0)])
def test_row_linear_situ_glu_matches_float64(rows, cap, hidden, k):
    from sophia_amd import ops
    dev = _dev()
    x, w = _data(rows, 2 * hidden, k)
    h = ops.row_linear_situ_glu(x.to(dev), w.to(dev), cap, 25.0)
    g, u = (x.double() @ w.double().t()).chunk(2, -1)
    ref = cap * torch.tanh(g / cap) * torch.sigmoid(g) * 25.0 * torch.tanh(u / 25.0)
    assert h.shape == (rows, hidden) and _close(h, ref)


def test_linear_rule_and_general_path_agree():
    """Every form of x and weight that F.linear takes gives its result, whether
    the rule takes it to the kernel or not; the ones it must not take (a gradient
    to record, autocast, other types, odd strides) are left to F.linear."""
    from sophia_amd import ops
    dev = _dev()
    x, w = (t.to(dev) for t in _data(12, 64, 96))
    big = torch.zeros(12, 101, dtype=torch.bfloat16, device=dev)
    big[:, :96] = x
    forms = {"rows": x, "leading dims": x.view(3, 2, 2, 96), "one row of many": x[:1], "row slice": x[2:9],
             "odd row stride": big[:, :96], "expanded": x[:1].expand(12, 96), "transposed": x.t().contiguous().t(),
             "leading dims, transposed": x.view(3, 4, 96).transpose(0, 1), "too many rows": x.repeat(4, 1),
             "no rows": x[:0], "every second": x[::2]}
    with torch.no_grad():
        for name, form in forms.items():
            y, ref = ops.linear(form, w), form.double() @ w.double().t()
            assert y.shape == ref.shape and y.dtype == torch.bfloat16, name
            if ref.numel():
                assert _close(y, ref.cpu()), name
        assert ops._few_rows(x, w) is not None and ops._few_rows(big[:, :96], w) is None
        assert ops._few_rows(x[:1].expand(12, 96), w) is None and ops._few_rows(x.float(), w) is None
        assert torch.equal(ops.linear(x.float(), w.float()), F.linear(x.float(), w.float()))
        wt = w.t().contiguous().t()
        assert ops._few_rows(x, wt) is None and _close(ops.linear(x, wt), (x.double() @ w.double().t()).cpu())
        with torch.autocast("cuda", dtype=torch.float16):
            assert ops.linear(x, w).dtype == torch.float16
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x.clone(), torch.ones_like(x))
            assert ops._few_rows(dual, w) is None
        empty = ops.linear(x, w[:0])
        assert empty.shape == (12, 0) and empty.dtype == torch.bfloat16
    wg = w.clone().requires_grad_(True)
    y = ops.linear(x, wg)
    y.float().sum().backward()
    assert wg.grad is not None
    seen = []

    def under_vmap(r):
        seen.append(ops._few_rows(r, w))
        return r

    torch.vmap(under_vmap)(x.view(3, 4, 96))
    assert seen == [None]


def test_linear_of_another_device_stays_with_the_library(monkeypatch):
    """Tensors of a device that is not the current one: F.linear changes to it, a
    launch of the kernel would go to the current device."""
    from sophia_amd import ops
    dev = _dev()
    x, w = (t.to(dev) for t in _data(12, 64, 96))
    with torch.no_grad():
        assert ops._few_rows(x, w) is not None
        monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
        assert ops._few_rows(x, w) is None


@pytest.mark.parametrize("rows", [5, 40])
def test_feed_forward_few_rows_and_graph(rows):
    """FeedForward with the one-launch projection and activation (5 rows) and
    without (40), against float64; captured, each replay equals the eager call."""
    from sophia_amd.config import ModelArgs
    from sophia_amd.decoder import FeedForward
    dev = _dev()
    torch.manual_seed(rows)
    with torch.device(dev):
        m = FeedForward(ModelArgs(dim=256, ffn_hidden=264)).to(torch.bfloat16)
    x = torch.randn(rows, 256, device=dev, dtype=torch.bfloat16)
    with torch.no_grad():
        y = m(x)
        g, u = (x.double() @ m.gate_up_proj.weight.double().t()).chunk(2, -1)
        h = 4.0 * torch.tanh(g / 4.0) * torch.sigmoid(g) * 25.0 * torch.tanh(u / 25.0)
        ref = h @ m.down_proj.weight.double().t()
        # h and (40 rows) the projection are rounded to bf16 before down_proj
        assert float((y.double() - ref).norm()) <= 8e-3 * float(ref.norm())
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = m(x)
        for seed in range(3):
            x.copy_(torch.randn(rows, 256, generator=torch.Generator().manual_seed(seed)))
            graph.replay()
            assert torch.equal(out, m(x))


@pytest.mark.parametrize("rows,heads,n,k", [(1, 1, 16, 32), (8, 16, 128, 128), (240, 16, 128, 128), (17, 3, 144, 96),
                                            (5, 2, 32, 320)])
def test_head_linear_matches_float64(rows, heads, n, k):
    """Rows and outputs that end inside a tile, more than one work-group of
    outputs, k past one batch of steps; x a slice of a wider row, the output a
    view of one (nothing written beside it)."""
    from sophia_amd import ops
    dev = _dev()
    g = torch.Generator().manual_seed(rows)
    wide = torch.randn(rows, heads, k + 8, generator=g).to(torch.bfloat16)
    w = (torch.randn(heads, n, k, generator=g) * k ** -0.5).to(torch.bfloat16)
    big = torch.full((rows + 2, heads, n + 4), 3.0, dtype=torch.bfloat16, device=dev)
    y = ops.head_linear(wide.to(dev)[:, :, 8:], w.to(dev), out=big[1:-1, :, :n])
    ref = torch.einsum("rhk,hnk->rhn", wide[:, :, 8:].double(), w.double())
    assert _close(y, ref) and _close(ops.head_linear(wide.to(dev)[:, :, 8:], w.to(dev)), ref)
    assert bool((big[0] == 3).all() and (big[-1] == 3).all() and (big[1:-1, :, n:] == 3).all())
    gate = torch.randn(rows, heads * n + 4, generator=g).to(torch.bfloat16).to(dev)[:, 4:].unflatten(1, (heads, n))
    gated = ops.head_linear(wide.to(dev)[:, :, 8:], w.to(dev), gate=gate)
    plain = ops.head_linear(wide.to(dev)[:, :, 8:], w.to(dev))
    assert _close(gated, plain.double().cpu() * torch.sigmoid(gate.double().cpu()))
    with pytest.raises(RuntimeError):
        ops.head_linear(wide.to(dev)[:, :, 8:].float(), w.to(dev))
    with pytest.raises(RuntimeError):
        ops.head_linear(wide.to(dev)[:, :, 8:], w.to(dev), gate=gate.float())


@pytest.mark.parametrize("rows,heads,n,k", [(1, 1, 16, 32), (8, 16, 128, 128), (17, 3, 144, 96), (5, 2, 32, 320),
                                            (33, 2, 272, 256)])
def test_head_linear_of_rows_first_weights_equals_the_transposed_copy(rows, heads, n, k):
    """weight_kn takes w [heads, k, n] as it lies: bit for bit head_linear of its
    transposed copy (the same operands in the same steps), with outputs and rows
    that end inside a tile, k short of, at and past the rows held in LDS."""
    from sophia_amd import ops
    dev = _dev()
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, heads, k + 8, generator=g).to(torch.bfloat16).to(dev)[:, :, 8:]
    w = (torch.randn(heads, k, n, generator=g) * k ** -0.5).to(torch.bfloat16).to(dev)
    big = torch.full((rows + 2, heads, n + 4), 3.0, dtype=torch.bfloat16, device=dev)
    y = ops.head_linear(x, w, out=big[1:-1, :, :n], weight_kn=True)
    assert torch.equal(y, ops.head_linear(x, w.transpose(1, 2).contiguous()))
    assert bool((big[0] == 3).all() and (big[-1] == 3).all() and (big[1:-1, :, n:] == 3).all())
    with pytest.raises(RuntimeError):
        ops.head_linear(x, w.transpose(1, 2).contiguous() if n != k else w[:, 1:], weight_kn=True)
