"""MoE stage 1 of W4A16 and blockscale on the stream kernel, against the oracle at the bar of
tests/test_gpu_moe.py: every number of K steps around its register sets, partly filled runs."""
import pytest
import torch

from flydsl_amd import workloads as W
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


@pytest.mark.parametrize("tile_m", [16, 32, 64])
@pytest.mark.parametrize("tokens", [67, 190, 700])
def test_blockscale_stage1_stream(gpu, tile_m, tokens):
    for K in (128, 256, 384, 512, 640, 896):
        w = W.moe_custom(tokens, K, 256, 5, 2, tile_m, 64, 128, "fp8_block", seed=K + tokens)
        p = W.moe_problem(w, gpu, with_stage2_input=False)
        out = M.run_bs_stage1(p, gpu, "bf16" if K % 256 else "f16", doweight=K % 256 == 0)
        M._check(out, M.ref_bs1(p, K % 256 == 0), what=f"blockscale tm{tile_m} t{tokens} K{K}")


def test_under_graph_capture(gpu):
    """Captured once and replayed, each replay equal to the eager run."""
    for kind in ("int4_bf16", "fp8_block"):
        w = W.moe_custom(200, 512, 1024, 5, 2, 16, 64, 128, kind, seed=3)
        p = W.moe_problem(w, gpu)
        run = (lambda: (M.run_bs_stage1(p, gpu),)) if kind == "fp8_block" else (lambda: (M.run_stage1(p, gpu, "bf16"),))
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
