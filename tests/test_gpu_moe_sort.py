"""moe_sorting on the GPU (the counting-sort kernel of csrc/moe_sort.hip) against the operator form
that CPU tensors take, which tests/test_oracle.py checks against the oracle: every buffer bit for bit."""
import pytest
import torch

from flydsl_amd import moe

pytestmark = pytest.mark.gpu


def _routing(M, topk, E, seed, skew=0.0, stray=0.0):
    g = torch.Generator().manual_seed(seed)
    score = torch.randn(M, E, generator=g) + skew * torch.randn(1, E, generator=g)
    top, ids = torch.topk(score, topk, dim=1)
    if stray:   # ids of no expert, negative ones among them
        out = torch.rand(M, topk, generator=g) < stray
        ids = torch.where(out, torch.randint(-3, E + 5, (M, topk), generator=g), ids)
    return ids, torch.softmax(top, dim=1)


def _same(got, want):
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and tuple(g.shape) == tuple(w.shape) and g.is_contiguous()
        assert torch.equal(g.cpu(), w)


# M, topk, E, block: one route; a wave and one more; one launch's largest routing and the first of
# two launches; chunks of one route; the most experts of the kernel, and one more (operators)
CASES = [(1, 1, 1, 16), (1, 8, 256, 32), (8, 8, 256, 32), (13, 5, 7, 1), (65, 1, 3, 64), (129, 2, 8, 32), (333, 9, 17, 64),
         (1023, 1, 128, 16), (1024, 8, 128, 64), (1025, 8, 128, 64), (4097, 4, 16, 64), (8192, 8, 256, 16), (31, 6, 512, 16),
         (5000, 8, 512, 32), (40, 2, 513, 16)]


@pytest.mark.parametrize("M,topk,E,block", CASES)
@pytest.mark.parametrize("form", ["plain", "skewed", "stray", "masked"])
def test_sorting_equals_operators(gpu, M, topk, E, block, form):
    ids, w = _routing(M, topk, E, M + E, skew=3.0 if form == "skewed" else 0.0, stray=0.3 if form == "stray" else 0.0)
    mask = None
    if form == "masked":
        mask = (torch.rand(E, generator=torch.Generator().manual_seed(E)) < 0.6).to(torch.int32)
    for ids_t, w_t in ((ids.to(torch.int32), w), (ids, w.to(torch.bfloat16))):
        want = moe.moe_sorting(ids_t, w_t, E, block, mask)
        got = moe.moe_sorting(ids_t.to(gpu), w_t.to(gpu), E, block, None if mask is None else mask.to(gpu))
        _same(got, want)


def test_every_route_to_one_expert_and_none_kept(gpu):
    for M, topk in ((64, 2), (9000, 2)):
        ids = torch.full((M, topk), 5, dtype=torch.int32)
        w = torch.rand(M, topk)
        for mask in (None, torch.tensor([0, 1, 0, 1, 0, 1, 0]), torch.tensor([1, 1, 1, 1, 1, 0, 1])):
            want = moe.moe_sorting(ids, w, 7, 32, mask)
            _same(moe.moe_sorting(ids.to(gpu), w.to(gpu), 7, 32, None if mask is None else mask.to(gpu)), want)


def test_strided_inputs(gpu):
    ids, w = _routing(70, 4, 16, 3)
    want = moe.moe_sorting(ids, w, 16, 16)
    wide_i, wide_w = torch.zeros(70, 8, dtype=torch.int64), torch.zeros(70, 8)
    wide_i[:, ::2], wide_w[:, ::2] = ids, w
    _same(moe.moe_sorting(wide_i.to(gpu)[:, ::2], wide_w.to(gpu)[:, ::2], 16, 16), want)
    _same(moe.moe_sorting(ids.t().contiguous().to(gpu).t(), w.t().contiguous().to(gpu).t(), 16, 16), want)
    one_i, one_w = wide_i[:, :2].to(gpu)[:, :1], wide_w[:, :2].to(gpu)[:, :1]   # [M, 1] with row stride 8
    _same(moe.moe_sorting(one_i, one_w, 16, 16), moe.moe_sorting(one_i.cpu(), one_w.cpu(), 16, 16))


def test_gradients_reach_the_weights(gpu):
    """Weights under autograd keep the operators, whose output carries the graph."""
    ids, w = _routing(9, 2, 4, 1)
    w = w.to(gpu).requires_grad_()
    sw = moe.moe_sorting(ids.to(gpu), w, 4, 16)[1]
    sw.sum().backward()
    assert torch.equal(w.grad, torch.ones_like(w))


@pytest.mark.parametrize("M", [16, 4096])
def test_under_graph_capture(gpu, M):
    """Captured once, replayed on new routings with eager work between the replays."""
    ids, w = _routing(M, 8, 64, 0)
    ids_d, w_d = ids.to(torch.int32).to(gpu), w.to(gpu)
    moe.moe_sorting(ids_d, w_d, 64, 32)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = moe.moe_sorting(ids_d, w_d, 64, 32)
    for seed in (1, 2, 3):
        ids, w = _routing(M, 8, 64, seed, skew=1.0)
        ids_d.copy_(ids)
        w_d.copy_(w)
        g.replay()
        torch.cuda.synchronize()
        _same(out, moe.moe_sorting(ids.to(torch.int32), w, 64, 32))
