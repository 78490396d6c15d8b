"""Calls that keep torch's operators where a kernel stands in for them on plain GPU tensors:
tracing, vmap, forward mode, dispatch modes and tensors whose memory is not their value.  The CPU
tests put the device aside (``plain`` in the place of ``plain_cuda``); with a kernel taken they would
fail on the pointer of a traced tensor, or trace nothing."""
import pytest
import torch

from flydsl_amd import _tensors, moe, quant
from flydsl_amd.moe import moe_sorting
from flydsl_amd.quant import blockscale_quant


def _operands(dev="cpu"):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(5, 256, generator=g).to(dev)
    ids = torch.stack([torch.randperm(8, generator=g)[:2] for _ in range(5)]).to(dev)
    return x, ids, torch.rand(5, 2, generator=g).to(dev)


def _both(x, ids, w):
    return (*blockscale_quant(x, 1, 128), *moe_sorting(ids, w, 8, 16))


def _same(got, want):
    for a, b in zip(got, want, strict=True):
        assert a.dtype == b.dtype and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _one_graph(f, *args):
    """f's results under torch.compile, which has to trace all of it into one graph."""
    sizes = []

    def backend(gm, _):
        sizes.append(sum(n.op in ("call_function", "call_method") for n in gm.graph.nodes))
        return gm.forward

    torch._dynamo.reset()
    out = torch.compile(f, fullgraph=True, backend=backend)(*args)
    assert len(sizes) == 1 and sizes[0] > 10
    return out


@pytest.fixture
def any_device(monkeypatch):
    for m in (moe, quant):
        monkeypatch.setattr(m, "plain_cuda", _tensors.plain)
    return monkeypatch


def test_compile_traces_the_operators(any_device):
    ops = _operands()
    got = _one_graph(_both, *ops)
    for m in (moe, quant):
        any_device.setattr(m, "plain_cuda", _tensors.plain_cuda)   # CPU tensors: the operators
    _same(got, _both(*ops))


@pytest.mark.gpu
def test_compile_on_the_gpu():
    ops = _operands("cuda")
    _same(_one_graph(_both, *ops), _both(*ops))


def test_plain():
    x = torch.randn(4, 4)
    assert _tensors.plain(x, x)
    assert not _tensors.plain(torch._neg_view(x))
    assert not _tensors.plain(x.to_sparse())
    assert not _tensors.plain(torch.nn.Parameter(x))
    leaf = x.clone().requires_grad_()
    assert not _tensors.plain(leaf)
    with torch.no_grad():
        assert _tensors.plain(leaf)
    with torch.device("cpu"):               # a function mode
        assert not _tensors.plain(x)
    with torch.autograd.forward_ad.dual_level():
        assert not _tensors.plain(x)
    seen = []
    torch.func.vmap(lambda r: seen.append(_tensors.plain(r)) or r)(x)
    assert seen == [False]
