"""Row and block quantization at the edges of their kernels: every lanes-per-row form and its first
longer row, both workgroup sizes, row counts that fill no workgroup, and rows whose quotients take the
reciprocal form, the division (scales outside 2^-90 .. 2^90) and the scrubbing of NaN and infinity.
Codes and scales bit for bit against the oracle (rows) and torch's operators on the GPU (blocks)."""
import numpy as np
import pytest
import torch

from flydsl_amd.kernels.quant import build_quant_module, per_token_quant
from flydsl_amd.quant import FP8, blockscale_quant
from oracle import quant as oq

pytestmark = pytest.mark.gpu


def _rows(N, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(29, N, generator=g) * torch.exp(3 * torch.randn(29, 1, generator=g))
    x[1] = 0.0
    x[2] = -0.0
    x[3, ::2] = -0.0
    x[4] *= 1e-30          # bf16 / fp32: scales below 2^-90, or zero in fp16
    x[5] *= 1e-38
    x[6, N // 2] = float("inf")
    x[7, N - 1] = float("nan")
    x[8, 0], x[8, N // 3] = -float("inf"), float("nan")
    if dtype != torch.float16:
        x[9] *= 1e30
    x[10] = torch.round(x[10])
    return x.to(dtype)


EDGES = [8, 64, 72, 128, 136, 256, 264, 512, 520, 1024, 1032, 2048, 2056, 4096, 8184, 8192]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qd,rounding", [(torch.int8, "nearest"), (torch.int8, "trunc"), (FP8, "nearest")])
def test_rows(gpu, dtype, qd, rounding):
    for N in EDGES:
        x = _rows(N, dtype, N)
        q_ref, s_ref = oq.quant_rows(x.float().numpy(), "fp8" if qd == FP8 else "int8",
                                     rounding="truncate" if rounding == "trunc" else "nearest")
        q_ref, s_ref = q_ref.view(np.uint8), s_ref.view(np.uint32)
        for copies, extra in ((1, 0), (36, 3), (142, 1)):   # 29, 1047 and 4119 rows
            xb = torch.cat([x.repeat(copies, 1), x[:extra]]).to(gpu)
            q, s = per_token_quant(xb, quant_dtype=qd, rounding=rounding)
            rows = np.arange(xb.shape[0]) % 29
            assert np.array_equal(s.cpu().view(-1).numpy().view(np.uint32), s_ref.reshape(-1)[rows]), (N, copies)
            assert np.array_equal(q.cpu().view(torch.uint8).numpy(), q_ref[rows]), (N, copies)


def test_reference_kernel_form(gpu):
    """Every kernel of the dispatch in this form too.  Nothing is scrubbed: NaN is left out of the row's
    maximum and gives code 0, infinity gives scale infinity and codes 0."""
    for N in EDGES:
        x = _rows(N, torch.float16, N)
        q_ref, s_ref = oq.quant_rows_recip(torch.nan_to_num(x, nan=0.0, posinf=0.0, neginf=0.0).numpy())
        q_ref[[6, 8]], s_ref[[6, 8]] = 0, np.inf
        for copies, extra in ((1, 0), (36, 3), (142, 1)):   # 29, 1047 and 4119 rows
            xb = torch.cat([x.repeat(copies, 1), x[:extra]]).to(gpu)
            rows = np.arange(xb.shape[0]) % 29
            launch, _ = build_quant_module(N)
            q = torch.empty(xb.shape[0], N, dtype=torch.int8, device=gpu)
            s = torch.empty(xb.shape[0], dtype=torch.float32, device=gpu)
            launch(xb, q, s, xb.shape[0])
            assert np.array_equal(s.cpu().numpy().view(np.uint32), s_ref.reshape(-1).view(np.uint32)[rows]), (N, copies)
            assert np.array_equal(q.cpu().numpy(), q_ref[rows]), (N, copies)


def test_quotients_are_the_divisions(gpu):
    """fp32 rows of random significands: codes of x / scale with the division that torch makes."""
    g = torch.Generator(device=gpu).manual_seed(0)
    x = torch.randn(4096, 2048, generator=g, device=gpu) * torch.exp(8 * torch.randn(4096, 1, generator=g, device=gpu))
    for qd in (FP8, torch.int8):
        q, s = per_token_quant(x, quant_dtype=qd)
        y = x / s
        want = y.to(FP8) if qd == FP8 else torch.round(y).clamp_(-127, 127).to(torch.int8)
        assert torch.equal(q.view(torch.uint8), want.view(torch.uint8))


def _block_ops(x, qmax):
    R, C = x.shape
    t = x.to(torch.float32).view(R, C // 128, 128)
    amax = torch.maximum(t.amax(dim=-1, keepdim=True), -t.amin(dim=-1, keepdim=True))
    scale = amax / qmax
    scale[scale == 0] = 1
    return (t / scale).reshape(R, C).to(FP8), scale.reshape(R, C // 128)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,C", [(1, 128), (3, 384), (29, 1024), (515, 7168)])
@pytest.mark.parametrize("qmax", [448.0, 240])
def test_blocks(gpu, dtype, R, C, qmax):
    x = _rows(C, dtype, R)[:R].repeat((R + 28) // 29, 1)[:R].to(gpu)
    for y in (x, x.t().contiguous().t(), torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(R, C)):   # strided, unaligned
        q, s = blockscale_quant(y, 1, 128, qmax)
        q_ref, s_ref = _block_ops(x, qmax)
        assert q.shape == (R, C) and s.shape == (R, C // 128) and s.is_contiguous()
        assert torch.equal(s.view(torch.int32), s_ref.view(torch.int32))
        assert torch.equal(q.view(torch.uint8), q_ref.view(torch.uint8))


def test_blocks_keep_the_operators(gpu):
    """Under autograd, and for a code range past the type's, the operators run as before."""
    x = torch.randn(4, 256, device=gpu, requires_grad=True)
    _, s = blockscale_quant(x, 1, 128)
    s.sum().backward()
    assert x.grad is not None and int((x.grad != 0).sum()) == 8
    q, _ = blockscale_quant(x.detach(), 1, 128, 1000.0)
    assert torch.equal(q.view(torch.uint8), _block_ops(x.detach(), 1000.0)[0].view(torch.uint8))
