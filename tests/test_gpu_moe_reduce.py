"""Reduce-mode stage 2 in one library call against its two steps on rows zeroed first (per-route GEMM,
then the reduction; both are checked against the oracle in tests/test_gpu_moe.py): equal bit for bit,
with routes that no expert takes, whether the rows are zeroed or the routes marked."""
import pytest
import torch

from flydsl_amd import workloads
from flydsl_amd.kernels.moe_gemm_2stage import (MoeGemm2Mode, compile_moe_gemm2, compile_moe_gemm2_ex,
                                                compile_moe_reduction)
from flydsl_amd.moe import moe_sorting

pytestmark = pytest.mark.gpu
_DT = {"f16": torch.float16, "bf16": torch.bfloat16}


def _problem(tokens, topk, dim, inter, experts, tile_m, kept, gpu):
    p = workloads.moe_problem(workloads.moe_custom(tokens, dim, inter, experts, topk, tile_m, 64, 128, seed=tokens), gpu)
    mask = torch.zeros(experts, dtype=torch.int32, device=gpu)
    mask[:kept] = 1
    ids, w, eids, post = moe_sorting(p["topk_ids"], p["topk_weights"], experts, tile_m, mask)
    return p, (ids, eids, w, post[:1].contiguous()), eids.numel()


def _args(p, meta, tokens, dim, inter, blocks):
    return (p["a2"].view(-1), p["w2_shuf"].view(-1), p["sa2"], p["sw2"], *meta, tokens, dim, inter, blocks)


# tokens, topk, model_dim, tile_m: rows below and above the 16 MB from which routes are marked; one,
# two and three groups of eight slots
CASES = [(40, 8, 1024, 16), (1023, 8, 1024, 32), (1025, 8, 1024, 32), (600, 9, 2048, 64), (300, 17, 2048, 16), (1100, 2, 4096, 64)]


@pytest.mark.parametrize("tokens,topk,dim,tile_m", CASES)
@pytest.mark.parametrize("out_dtype", ["f16", "bf16"])
@pytest.mark.parametrize("kept", [0, 11, 24])
def test_one_call_equals_two_steps(gpu, tokens, topk, dim, tile_m, out_dtype, kept):
    experts, inter = 24, 256
    p, meta, blocks = _problem(tokens, topk, dim, inter, experts, tile_m, kept, gpu)
    kw = dict(model_dim=dim, inter_dim=inter, experts=experts, topk=topk, tile_m=tile_m, tile_n=128, tile_k=128,
              doweight_stage2=True, in_dtype="fp8", out_dtype=out_dtype)
    args = _args(p, meta, tokens, dim, inter, blocks)
    rows = torch.zeros(tokens * topk * dim, dtype=_DT[out_dtype], device=gpu)
    want = torch.empty(tokens * dim, dtype=_DT[out_dtype], device=gpu)
    stream = torch.cuda.current_stream()
    compile_moe_gemm2(**kw, accumulate=False)(rows, *args, stream)
    compile_moe_reduction(topk=topk, model_dim=dim, dtype_str=out_dtype)(rows, want, None, tokens, stream)
    # memory that the allocator hands out next holds NaNs: rows that are neither written nor zeroed show
    n = rows.numel()
    del rows
    junk = torch.full((2 * n + 65536,), float("nan"), dtype=_DT[out_dtype], device=gpu)
    del junk
    got = torch.empty_like(want)
    compile_moe_gemm2_ex(**kw, mode=MoeGemm2Mode.REDUCE)(got, *args, stream=stream)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("topk", [1, 2, 7, 8, 9, 15, 16, 17, 25])
def test_reduction_groups_and_remainders(gpu, dt, topk):
    """Every form of the reduction, bit for bit: fp32 sums in slot order, one rounding, masked slots
    not read (they hold NaN)."""
    tokens, dim = 67, 264
    dtype = torch.float32 if dt == "f32" else _DT[dt]
    g = torch.Generator().manual_seed(topk)
    x = torch.randn(tokens, topk, dim, generator=g).to(dtype)
    mask = (torch.rand(tokens, topk, generator=g) < 0.7).to(torch.int8)
    mask[3] = 0
    for use_mask in (False, True):
        want = torch.zeros(tokens, dim)
        for s in range(topk):
            want = torch.where((mask[:, s:s + 1] != 0) if use_mask else torch.tensor(True), want + x[:, s].float(), want)
        xs = x.clone()
        if use_mask:
            xs[mask == 0] = float("nan")
        y = torch.empty(tokens, dim, dtype=dtype, device=gpu)
        compile_moe_reduction(topk=topk, model_dim=dim, dtype_str=dt, use_mask=use_mask)(
            xs.to(gpu).view(-1), y.view(-1), mask.to(gpu).view(-1) if use_mask else None, tokens)
        assert torch.equal(y.cpu(), want.to(dtype))


def test_other_stream(gpu):
    """Called for another stream than the current one: everything runs there."""
    tokens, topk, dim = 1025, 8, 1024
    p, meta, blocks = _problem(tokens, topk, dim, 256, 24, 32, 11, gpu)
    s2 = compile_moe_gemm2_ex(model_dim=dim, inter_dim=256, experts=24, topk=topk, tile_m=32, tile_n=128, tile_k=128,
                              doweight_stage2=True, in_dtype="fp8", out_dtype="f16", mode=MoeGemm2Mode.REDUCE)
    args = _args(p, meta, tokens, dim, 256, blocks)
    want, got = (torch.empty(tokens * dim, dtype=torch.float16, device=gpu) for _ in range(2))
    s2(want, *args)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    s2(got, *args, stream=side)
    side.synchronize()
    assert torch.equal(got, want)
    got.zero_()
    torch.cuda.synchronize()
    s2(got, *args, stream=side.cuda_stream)
    side.synchronize()
    assert torch.equal(got, want)


def _stage2(topk, dim, **kw):
    return compile_moe_gemm2_ex(model_dim=dim, inter_dim=256, experts=24, topk=topk, tile_m=32, tile_n=128, tile_k=128,
                                doweight_stage2=True, in_dtype="fp8", out_dtype="f16", mode=MoeGemm2Mode.REDUCE, **kw)


def _busy(big):
    """Some twenty milliseconds of work on the current stream: far more than one layer takes."""
    for _ in range(60):
        big[1].copy_(big[0])


@pytest.mark.parametrize("as_handle", [False, True])
def test_other_stream_with_work_queued_on_the_current_one(gpu, as_handle):
    """While the current stream still has work to do on a block that was handed back to the allocator,
    a call for another stream neither takes that block for its rows nor reads a mask that the
    current stream has yet to copy."""
    tokens, topk, dim = 1025, 8, 1024
    p, meta, blocks = _problem(tokens, topk, dim, 256, 24, 32, 11, gpu)
    args = _args(p, meta, tokens, dim, 256, blocks)
    want, want_m, got = (torch.empty(tokens * dim, dtype=torch.float16, device=gpu) for _ in range(3))
    mask = (torch.rand(topk, tokens, device=gpu) < 0.5).to(torch.int8).t()     # not contiguous
    kept = p["topk_ids"] < 11
    mask &= kept                                                               # routes that have a row
    plain, masked = _stage2(topk, dim), _stage2(topk, dim, valid_mask=mask)
    plain(want, *args)
    masked(want_m, *args, valid_mask=mask)
    # a block of every size class that the rows (and the mask behind them) can come from
    nbytes = [(tokens * topk * dim * 2 + 255) // 256 * 256 + m for m in (0, (tokens * topk + 255) // 256 * 256)]
    after = [torch.empty(n, dtype=torch.uint8, device=gpu) for n in nbytes]
    big = torch.zeros(2, 2 ** 30, dtype=torch.uint8, device=gpu)
    side = torch.cuda.Stream()
    stream = side.cuda_stream if as_handle else side
    torch.cuda.synchronize()
    for fn, kw, ref in ((plain, {}, want), (masked, dict(valid_mask=mask), want_m)):
        fn(got, *args, stream=stream, **kw)     # (memory of the side stream's own, so that nothing waits below)
        torch.cuda.synchronize()
        got.zero_()
        torch.cuda.synchronize()
        held = [torch.full((n,), 7, dtype=torch.uint8, device=gpu) for n in nbytes]
        _busy(big)
        for a, h in zip(after, held):
            a.copy_(h)
        del held, h
        fn(got, *args, stream=stream, **kw)
        side.synchronize()
        assert not torch.cuda.current_stream().query()      # the side call overtook the queued work
        assert torch.equal(got, ref)
        torch.cuda.synchronize()
        assert all(bool((a == 7).all()) for a in after)
