"""MoE stages on the tiles between decode and large experts, against the oracle at the bar of
tests/test_gpu_moe.py: stage 1 of W4A16 and blockscale on the stream kernel (every number of K steps
around its register sets, partly filled runs), and stage 2 on runs of 32 and 64 rows."""
import numpy as np
import pytest
import torch

from flydsl_amd import workloads as W
from flydsl_amd.kernels.moe_gemm_2stage import MoeGemm2Mode, compile_moe_gemm2_ex
from tests import helpers as H
from tests import test_gpu_moe as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [-1, 32])
@pytest.mark.parametrize("tile_m", [16, 32, 64])
@pytest.mark.parametrize("tokens", [1, 43, 190])
def test_w4a16_stage1_stream(gpu, group, tile_m, tokens):
    """K of 1 to 7 steps of 256 elements, and of no whole step (the LDS-staged kernel)."""
    for K in (256, 512, 768, 1024, 1280, 1792, 320):
        w = W.moe_custom(tokens, K, 128, 5, 2, tile_m, 64, 64, "int4_bf16", seed=K + tokens)
        p = W.moe_problem(w, gpu, group_size=group, with_stage2_input=False)
        out = M.run_stage1(p, gpu, "bf16" if K % 512 else "f16", doweight=K % 512 == 0)
        M.check_stage1(p, out, K % 512 == 0, what=f"W4A16 g{group} tm{tile_m} t{tokens} K{K}")


@pytest.mark.parametrize("group", [-1, 32])
@pytest.mark.parametrize("tokens,tile", [(512, (1, 128)), (160, (1, 64))])
def test_w4a16_stage1_lds_tiles(gpu, group, tokens, tile):
    """Stage 1 of W4A16 where model_dim is no whole number of 256-element steps: single-block tiles of
    128 columns from about three workgroups per CU, else of 64."""
    w = W.moe_custom(tokens, 576, 1024, 64, 4, 32, 256, 64, "int4_bf16", seed=tokens)
    assert M._chosen_tile(1, w, "int4_bf16") == tile
    p = W.moe_problem(w, gpu, group_size=group, with_stage2_input=False)
    # (group scales: against the oracle's truncation, and against the exact dequantization, an
    # approximate bound, on the smaller routing)
    M.check_stage1(p, M.run_stage1(p, gpu, "bf16", doweight=True), True, what=f"W4A16 g{group} LDS tiles t{tokens}",
                   exact=tokens == 160)


@pytest.mark.parametrize("tile_m", [16, 32, 64])
@pytest.mark.parametrize("tokens", [251, 700])
def test_blockscale_stage1_stream(gpu, tile_m, tokens):
    """inter_dim 4096, so that there are workgroups for the whole chip; a sample of tokens."""
    rows = np.unique(np.r_[np.arange(0, tokens, 13), tokens - 1])
    for K in (128, 256, 384, 512, 640, 896):
        w = W.moe_custom(tokens, K, 4096, 5, 2, tile_m, 64, 128, "fp8_block", seed=K + tokens)
        assert M._chosen_tile(1, w, "fp8", 1) == (128 // tile_m, 64)
        p = W.moe_problem(w, gpu, with_stage2_input=False)
        out = M.run_bs_stage1(p, gpu, "bf16" if K % 256 else "f16", doweight=K % 256 == 0)
        assert torch.isfinite(out.float()).all()
        M._check(out, M.ref_bs1(p, K % 256 == 0, rows), rows, what=f"blockscale tm{tile_m} t{tokens} K{K}")


def _reduce(p, gpu, kind, out_dtype, group=-1):
    w = p["workload"]
    fn = compile_moe_gemm2_ex(model_dim=w.model_dim, inter_dim=w.inter_dim, experts=w.experts, topk=w.topk,
                              tile_m=w.tile_m, tile_n=w.tile_n2, tile_k=M._tile_k(kind), doweight_stage2=True, in_dtype=kind,
                              out_dtype=out_dtype, mode=MoeGemm2Mode.REDUCE, group_size=group)
    out = torch.full((w.tokens, w.model_dim), float("nan"), dtype=M.OUT_T[out_dtype], device=gpu)
    empty = torch.empty(0, dtype=torch.float32, device=gpu)
    fn(out, H.dev_flat(p["a2"], gpu), H.dev_flat(p["w2_shuf"], gpu), empty if p["sa2"] is None else p["sa2"],
       empty if p["sw2"] is None else p["sw2"], p["sorted_ids"], p["sorted_expert_ids"], p["sorted_weights"],
       p["num_valid_ids"], w.tokens, w.model_dim, w.inter_dim, p["blocks"])
    return out


# kind, inter_dim, tokens (top-2 of 5 experts: 40, 60 and 160 routes per expert), on whatever tile they take
STAGE2 = [("fp8", 256, 100), ("fp8", 256, 400), ("bf16", 128, 100), ("bf16", 256, 400), ("int4", 256, 100), ("fp8", 1024, 100),
          ("fp8", 1152, 400), ("int8", 1024, 150), ("int4", 1024, 400), ("fp16", 512, 150), ("bf16", 576, 400),
          ("int4_bf16", 512, 150), ("int4_bf16", 1024, 400)]


@pytest.mark.parametrize("kind,inter,tokens", STAGE2)
@pytest.mark.parametrize("tile_m", [16, 32, 64])
@pytest.mark.parametrize("model_dim", [256, 384])
def test_stage2_mid(gpu, kind, inter, tokens, tile_m, model_dim):
    w = W.moe_custom(tokens, model_dim, inter, 5, 2, tile_m, 64, 128, kind, seed=inter + tokens + tile_m)
    p = W.moe_problem(w, gpu)
    what = f"stage2 {kind} tm{tile_m} t{tokens} {model_dim}x{inter}"
    for out_dtype in ("f16", "f32", "bf16"):
        out = M.run_stage2(p, gpu, out_dtype, doweight=True)
        M.check_stage2(p, out, True, what=f"{what} atomics {out_dtype}",
                       atol_rms=M.BF16_ATOMIC_ATOL if out_dtype == "bf16" else 1e-2)
    M.check_stage2(p, _reduce(p, gpu, kind, "bf16"), True, what=f"{what} rows", route_round="bf16")


# The tiles of the routings in between, each reached on purpose: kind, group, tokens, model_dim, inter_dim, experts,
# top-k, tile_m, tile_n, tile with atomics (None: the query does not cover group scales)
TILES = [("fp8", -1, 100, 256, 256, 5, 2, 16, 128, (2, 64)), ("int4", -1, 100, 256, 256, 5, 2, 16, 128, (2, 64)),
         ("fp8", -1, 400, 256, 256, 5, 2, 16, 128, (4, 128)), ("bf16", -1, 150, 256, 512, 5, 2, 16, 128, (4, 128)),
         ("int8", -1, 400, 256, 1024, 5, 2, 16, 128, (4, 128)), ("int4", -1, 400, 256, 1024, 5, 2, 16, 128, (4, 128)),
         ("fp16", -1, 300, 256, 1024, 5, 2, 16, 128, (4, 128)), ("bf16", -1, 400, 256, 1024, 5, 2, 16, 128, (16, 256)),
         ("fp8", -1, 100, 256, 4096, 5, 2, 16, 128, (4, 128)), ("fp8", -1, 180, 1152, 1024, 5, 2, 16, 128, (4, 128)),
         ("int4_bf16", -1, 150, 256, 1024, 5, 2, 16, 128, (4, 128)), ("int4_bf16", -1, 500, 384, 512, 5, 2, 16, 128, (4, 128)),
         ("fp8", -1, 100, 256, 4096, 5, 2, 32, 128, (2, 128)), ("int4", -1, 100, 384, 4096, 5, 2, 32, 128, (2, 128)),
         ("bf16", -1, 1100, 256, 1024, 12, 4, 32, 128, (2, 128)), ("int4_bf16", -1, 150, 256, 4096, 5, 2, 32, 128, (2, 128)),
         ("fp8", -1, 280, 256, 4096, 5, 2, 64, 128, (1, 128)), ("int8", -1, 1100, 256, 1024, 12, 4, 64, 128, (1, 128)),
         # group scales at 60 and 200 routes per expert
         ("int4_bf16", 32, 150, 256, 512, 5, 2, 16, 128, None), ("int4_bf16", 32, 500, 256, 1024, 5, 2, 16, 128, None),
         ("int4_bf16", 32, 150, 256, 4096, 5, 2, 32, 128, None), ("int4_bf16", 32, 1200, 256, 512, 12, 4, 32, 128, None),
         ("int4_bf16", 32, 150, 256, 1024, 5, 2, 64, 128, None), ("int4_bf16", 32, 600, 384, 1024, 12, 4, 64, 128, None),
         ("int4_bf16", 32, 1100, 256, 1024, 12, 4, 64, 128, None)]


@pytest.mark.parametrize("case", TILES, ids=lambda c: "-".join(str(v) for v in c[:9]))
def test_stage2_mid_tiles(gpu, case):
    kind, group, tokens, model_dim, inter, experts, topk, tile_m, tile_n, tile = case
    w = W.moe_custom(tokens, model_dim, inter, experts, topk, tile_m, 64, tile_n, kind, seed=inter + tokens + tile_m)
    if tile is not None:
        assert M._chosen_tile(2, w, kind) == tile
    p = W.moe_problem(w, gpu, group_size=group)
    p["group_size"] = group
    rows = np.unique(np.r_[np.arange(0, tokens, 7), tokens - 1])
    for out_dtype in ("f16", "f32", "bf16"):
        out = M.run_stage2(p, gpu, out_dtype, doweight=True)
        assert torch.isfinite(out.float()).all()
        M.check_stage2(p, out, True, rows, rows, what=f"{case} atomics {out_dtype}",
                       atol_rms=M.BF16_ATOMIC_ATOL if out_dtype == "bf16" else 1e-2)
    out = _reduce(p, gpu, kind, "bf16", group)
    assert torch.isfinite(out.float()).all()
    M.check_stage2(p, out, True, rows, rows, what=f"{case} rows", route_round="bf16")


@pytest.mark.parametrize("tile_m", [16, 32, 64])
@pytest.mark.parametrize("tokens", [150, 240])
def test_blockscale_stage2_mid(gpu, tile_m, tokens):
    w = W.moe_custom(tokens, 384, 1024, 5, 2, tile_m, 128, 128, "fp8_block", seed=tokens + tile_m)
    p = W.moe_problem(w, gpu)
    for out_dtype, mode in (("f16", "atomic"), ("f32", "atomic"), ("f16", "reduce")):
        out = M.run_bs_stage2(p, gpu, out_dtype, doweight=True, mode=mode)
        M._check(out, M.ref_bs2(p, True), what=f"blockscale stage2 tm{tile_m} t{tokens} {mode} {out_dtype}")


def test_under_graph_capture(gpu):
    """Both stages of W4A16 and blockscale captured once and replayed, each replay equal to the eager
    run (stage 1 and the fp32 rows have one order; stage 2 through the reduce mode)."""
    for kind in ("int4_bf16", "fp8_block"):
        w = W.moe_custom(200, 512, 4096, 5, 2, 16, 64, 128, kind, seed=3)
        assert M._chosen_tile(1, w, "fp8" if kind == "fp8_block" else kind, kind == "fp8_block")[0] > 1   # the stream kernel
        p = W.moe_problem(w, gpu)
        run = (lambda: (M.run_bs_stage1(p, gpu), M.run_bs_stage2(p, gpu, mode="reduce"))) if kind == "fp8_block" else \
            (lambda: (M.run_stage1(p, gpu, "bf16"), _reduce(p, gpu, kind, "bf16")))
        eager = [t.clone() for t in run()]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            run()
        torch.cuda.current_stream().wait_stream(side)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            outs = run()
        for _ in range(3):
            for t in outs:
                t.zero_()
            g.replay()
            torch.cuda.synchronize()
            for got, want in zip(outs, eager):
                assert torch.equal(got, want)
            run()
