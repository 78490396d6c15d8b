"""The work this library is measured on: single linear layers and whole MoE layers, through the
public entry points, on synthetic operands of serving sizes.

A case is a dict of plain values.  ``op`` is one of

* ``linear``      a GEMM of operands that are already quantized, as the launcher of
                  ``compile_preshuffle_gemm_a8`` / ``_w4`` / ``compile_blockscale_preshuffle_gemm``
                  pre-bound by ``flydsl_amd.compile`` runs it: ``kind`` fp8, int8, int4 (W4A8), bf16,
                  fp16, mxfp4 or fp8_block, sizes ``M``, ``N``, ``K`` (elements), output type ``out``;
* ``act_linear``  a linear layer from 16-bit activations: ``quant_gemm`` (row quantization and GEMM in
                  one call), ``kind`` fp8, int8 or int4;
* ``moe``         an MoE layer behind its router: ``moe_sorting``, quantization of the activations,
                  stage 1, quantization of its output, stage 2 (``mode`` atomic or reduce); ``kind``
                  fp8, int8, int4 (W4A8), int4_bf16 (W4A16), bf16 or fp8_block.

Operands are drawn on the GPU from the seed: N(0, 1) activations, weights of the scale of trained
layers, quantized per row, per block or per 32 elements as the entry points expect.
"""
from __future__ import annotations

import math

import torch

import flydsl_amd as fly
from flydsl_amd import fp4
from flydsl_amd.kernels.blockscale_preshuffle_gemm import compile_blockscale_preshuffle_gemm
from flydsl_amd.kernels.moe_blockscale_2stage import (compile_moe_blockscale_gemm1,
                                                      compile_moe_blockscale_gemm2_ex)
from flydsl_amd.kernels.moe_gemm_2stage import compile_moe_gemm1, compile_moe_gemm2_ex
from flydsl_amd.kernels.preshuffle_gemm import compile_preshuffle_gemm_a8, compile_preshuffle_gemm_w4
from flydsl_amd.kernels.quant import per_token_quant, quant_gemm
from flydsl_amd.moe import moe_sorting

FP8 = torch.float8_e4m3fn
OUT = {"bf16": torch.bfloat16, "fp16": torch.float16}
MOE_OUT = {"bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # one token of a decode step through a small projection: the smallest call, all latency
        dict(name="act_linear_1", op="act_linear", kind="fp8", M=1, N=7168, K=2048, out="bf16"),
        # a decode step of 16 sequences through an up projection: streams 235 MB of weights
        dict(name="linear_fp8_16", op="linear", kind="fp8", M=16, N=28672, K=8192, out="bf16"),
        # a decode step of a busy server (128 sequences) through a square projection
        dict(name="linear_fp8_128", op="linear", kind="fp8", M=128, N=4096, K=4096, out="bf16"),
        # 4-bit weights at a large decode batch
        dict(name="linear_int4_256", op="linear", kind="int4", M=256, N=14336, K=4096, out="bf16"),
        # a prefill chunk through a block-scaled (1x128 / 128x128) projection
        dict(name="linear_block_1024", op="linear", kind="fp8_block", M=1024, N=7168, K=7168, out="bf16"),
        # a prefill chunk with MXFP4 weights and activations
        dict(name="linear_mxfp4_1024", op="linear", kind="mxfp4", M=1024, N=8192, K=8192, out="bf16"),
        # a long prompt in INT8
        dict(name="linear_int8_4096", op="linear", kind="int8", M=4096, N=4096, K=4096, out="bf16"),
        # an unquantized layer on a ragged batch of prompts: rows and K tiles that fill no tile
        dict(name="linear_bf16_5133", op="linear", kind="bf16", M=5133, N=5120, K=8320, out="fp16"),
        # a large batch of prompts, the largest product
        dict(name="linear_fp8_8192", op="linear", kind="fp8", M=8192, N=8192, K=8192, out="bf16"),
        # an MoE layer in a decode step of 8 sequences: few routes over many experts
        dict(name="moe_fp8_8", op="moe", kind="fp8", tokens=8, model_dim=7168, inter_dim=256, experts=256, topk=8,
             tile_m=32, mode="atomic"),
        # the same layer in block-scaled fp8 at 128 sequences
        dict(name="moe_block_128", op="moe", kind="fp8_block", tokens=128, model_dim=7168, inter_dim=256, experts=256,
             topk=8, tile_m=16, mode="atomic"),
        # an MoE layer in prefill, per-route rows and a reduction over the slots
        dict(name="moe_fp8_8192", op="moe", kind="fp8", tokens=8192, model_dim=7168, inter_dim=256, experts=128,
             topk=8, tile_m=64, mode="reduce"),
    ]


# model_dim, inter_dim, experts, topk of the MoE layers that draws take
MOE_DIMS = ((7168, 256, 256, 8), (7168, 256, 128, 8), (4096, 1536, 64, 8), (6144, 1024, 128, 8), (4096, 14336, 8, 2),
            (1024, 256, 8, 2), (4096, 2048, 17, 9))
# no drawn case takes more work than the largest listed ones
MOST_FLOPS, MOST_FLOPS_MOE, MOST_BYTES = 2 * 8192 ** 3, 7.2e11, 2.5e9


def _log(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    while True:
        op = rng.choice(["linear", "linear", "linear", "act_linear", "moe", "moe"])
        if op == "moe":
            d, i, e, k = rng.choice(MOE_DIMS)
            c = dict(op=op, kind=rng.choice(["fp8", "fp8", "int8", "int4", "int4_bf16", "bf16", "fp8_block"]),
                     tokens=_log(rng, 1, 8192), model_dim=d, inter_dim=i, experts=e, topk=k,
                     tile_m=rng.choice([16, 32, 64]), mode=rng.choice(["atomic", "reduce"]))
        else:
            kinds = ["fp8", "int8", "int4"] if op == "act_linear" else ["fp8", "int8", "int4", "bf16", "fp16", "mxfp4",
                                                                       "fp8_block"]
            kind = rng.choice(kinds)
            n_step, k_step = {"mxfp4": (32, 256), "fp8_block": (16, 128)}.get(kind, (16, 128))
            c = dict(op=op, kind=kind, M=_log(rng, 1, 8192), N=_log(rng, 1024, 28672, n_step),
                     K=_log(rng, 1024, 8320, k_step), out=rng.choice(["bf16", "bf16", "fp16"]))
        w = work(c)
        if w["flops"] <= (MOST_FLOPS_MOE if op == "moe" else MOST_FLOPS) and w["bytes"] <= MOST_BYTES:
            return c


# ---- operands ----------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rand(g, rows, cols, std):
    return torch.randn(rows, cols, generator=g, device="cuda").mul_(std)


def _row_quant(x, dtype, qmax):
    """Symmetric per-row quantization: codes and fp32 scales [rows]."""
    s = x.abs().amax(dim=1, keepdim=True) / qmax
    s = torch.where(s == 0, torch.ones_like(s), s)
    y = x / s
    if dtype == torch.int8:
        y = y.round_().clamp_(-qmax, qmax)
    return y.to(dtype), s.reshape(-1)


def _block_quant(x, br, bc=128):
    """fp8 codes and fp32 scales [ceil(R/br), C/bc] of br x bc blocks."""
    R, C = x.shape
    rp = -(-R // br) * br
    if rp != R:
        x = torch.cat([x, x.new_zeros(rp - R, C)])
    t = x.view(rp // br, br, C // bc, bc)
    s = t.abs().amax(dim=(1, 3), keepdim=True) / 448.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return (t / s).view(rp, C)[:R].to(FP8), s.view(rp // br, C // bc)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
_E2M1_MID = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)


def _mx_quant(x):
    """MXFP4: e2m1 codes [R, C] (uint8) and E8M0 scale bytes [R, C/32]."""
    R, C = x.shape
    b = x.view(R, C // 32, 32)
    e = torch.ceil(torch.log2(b.abs().amax(dim=2).clamp_min(1e-30) / 6.0)).clamp(-126, 126)
    y = b / torch.exp2(e)[:, :, None]
    code = torch.bucketize(y.abs(), torch.tensor(_E2M1_MID, device=x.device)).to(torch.uint8)
    code |= (y < 0).to(torch.uint8) << 3
    return code.view(R, C), (e + 127).to(torch.uint8)


def _mx_value(code, scale):
    table = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device=code.device)
    R, C = code.shape
    v = table[code.int()].view(R, C // 32, 32) * torch.exp2(scale.double() - 127.0)[:, :, None]
    return v.view(R, C)


def _linear_operands(c, seed):
    """Plain (unshuffled) operands of a linear case and their scales."""
    g = _gen(seed)
    M, N, K, kind = c["M"], c["N"], c["K"], c["kind"]
    a = _rand(g, M, K, 1.0)
    b = _rand(g, N, K, 0.02 if kind == "int4" else 1.0)
    if c["op"] == "act_linear":
        a, sa = a.to(torch.bfloat16), None
    elif kind in OUT:
        a, sa = a.to(OUT[kind]), None
    elif kind == "fp8_block":
        a, sa = _block_quant(a, 1)
    elif kind == "mxfp4":
        a, sa = _mx_quant(torch.cat([a, a.new_zeros(-M % 32, K)]))
    else:
        a, sa = _row_quant(a, FP8 if kind == "fp8" else torch.int8, 448.0 if kind == "fp8" else 127.0)
    if kind in OUT:
        b, sb = b.to(OUT[kind]), None
    elif kind == "fp8_block":
        b, sb = _block_quant(b, 128)
    elif kind == "mxfp4":
        b, sb = _mx_quant(b)
    else:
        b, sb = _row_quant(b, FP8 if kind == "fp8" else torch.int8, {"fp8": 448.0, "int8": 127.0, "int4": 7.0}[kind])
    return a, sa, b, sb


def _moe_operands(c, seed):
    """Activations (bf16), plain quantized weights and the router's choice."""
    g = _gen(seed)
    T, D, I, E, k, kind = (c[n] for n in ("tokens", "model_dim", "inter_dim", "experts", "topk", "kind"))
    x = _rand(g, T, D, 0.2).to(torch.bfloat16)
    ws = []
    for rows, cols, std in ((E * 2 * I, D, 0.2), (E * D, I, 0.2 / math.sqrt(I))):
        w = _rand(g, rows, cols, std)
        if kind == "fp8":
            ws.append(_row_quant(w, FP8, 448.0))
        elif kind == "fp8_block":
            ws.append(_block_quant(w, 128))
        elif kind == "bf16":
            ws.append((w.to(torch.bfloat16), None))
        else:
            ws.append(_row_quant(w, torch.int8, 127.0 if kind == "int8" else 7.0))
        del w
    # some experts are chosen more often than others
    score = torch.randn(T, E, generator=g, device="cuda") + 0.5 * torch.randn(1, E, generator=g, device="cuda")
    top, ids = torch.topk(score, k, dim=1)
    return x, ws[0], ws[1], ids.to(torch.int32), torch.softmax(top, dim=1).float()


def _moe_types(kind):
    """Stage output type (the 16-bit kinds' stage 2 takes bf16 rows)."""
    return "bf16" if kind in ("bf16", "int4_bf16") else "f16"


# ---- a user's program --------------------------------------------------------------------
def prepare(case, seed):
    c = case
    stream = torch.cuda.current_stream()
    s = dict(case=c, stream=stream)
    if c["op"] == "moe":
        x, (w1, sw1), (w2, sw2), ids, tw = _moe_operands(c, seed)
        T, D, I, E, k, kind = (c[n] for n in ("tokens", "model_dim", "inter_dim", "experts", "topk", "kind"))
        ot = _moe_types(kind)
        for n, w in (("w1", w1), ("w2", w2)):
            w = fly.shuffle_weight(w)
            s[n] = (fly.pack_int4(w) if kind in ("int4", "int4_bf16") else w).view(-1)
        del w1, w2, w
        empty = torch.empty(0, dtype=torch.float32, device="cuda")
        s.update(x=x, sw1=empty if sw1 is None else sw1.reshape(-1), sw2=empty if sw2 is None else sw2.reshape(-1), ids=ids,
                 tw=tw, empty=empty, out1=torch.empty(T * k, I, dtype=MOE_OUT[ot], device="cuda"),
                 out=torch.empty(T, D, dtype=MOE_OUT[ot], device="cuda"))
        kw = dict(model_dim=D, inter_dim=I, experts=E, topk=k, tile_m=c["tile_m"], tile_k=128, out_dtype=ot)
        if kind == "fp8_block":
            s["s1"] = compile_moe_blockscale_gemm1(tile_n=128, doweight_stage1=False, **kw)
            s["s2"] = compile_moe_blockscale_gemm2_ex(tile_n=256, doweight_stage2=True, mode=c["mode"], **kw)
        else:
            s["s1"] = compile_moe_gemm1(tile_n=128, doweight_stage1=False, in_dtype=kind, **kw)
            s["s2"] = compile_moe_gemm2_ex(tile_n=256, doweight_stage2=True, in_dtype=kind, mode=c["mode"], **kw)
        return s
    M, N, K, kind = c["M"], c["N"], c["K"], c["kind"]
    a, sa, b, sb = _linear_operands(c, seed)
    out = torch.empty(M, N, dtype=OUT[c["out"]], device="cuda")
    if c["op"] == "act_linear":
        bq = fly.shuffle_weight(b)
        s.update(x=a, b=fly.pack_int4(bq) if kind == "int4" else bq, sb=sb, out=out,
                 a_q=torch.empty(M, K, dtype=FP8 if kind == "fp8" else torch.int8, device="cuda"),
                 sa=torch.empty(M, 1, dtype=torch.float32, device="cuda"))
        return s
    if kind == "mxfp4":
        launch = compile_preshuffle_gemm_w4(K=K, tile_m=64, tile_n=256, tile_k=256, out_dtype=c["out"])
        args = (out, fp4.pack_fp4(a)[:M].contiguous(), fp4.shuffle_weight_w4(fp4.pack_fp4(b)),
                fp4.shuffle_scale_w4(sa), fp4.shuffle_scale_w4(sb))
    elif kind == "fp8_block":
        launch = compile_blockscale_preshuffle_gemm(K=K, tile_m=64, tile_n=128, tile_k=128, out_dtype=c["out"])
        args = (out, a, fly.shuffle_weight(b), sa.t().contiguous(), sb)
    else:
        launch = compile_preshuffle_gemm_a8(K=K, tile_m=64, tile_n=128, tile_k=64 if kind in OUT else 128,
                                            in_dtype=kind, out_dtype=c["out"])
        bs = fly.shuffle_weight(b)
        empty = torch.empty(0, dtype=torch.float32, device="cuda")
        args = (out, a, fly.pack_int4(bs) if kind == "int4" else bs, empty if sa is None else sa,
                empty if sb is None else sb)
    args = tuple(t.view(-1) for t in args)
    s.update(gemm=fly.compile(launch, *args, M, N, stream), args=args, M=M, N=N, out=out)
    return s


def _moe_layer(s):
    c = s["case"]
    T, D, I, E, k, kind = (c[n] for n in ("tokens", "model_dim", "inter_dim", "experts", "topk", "kind"))
    st, empty = s["stream"], s["empty"]
    sid, sw, eid, post = moe_sorting(s["ids"], s["tw"], E, c["tile_m"])
    nv, blocks = post[:1], eid.numel()

    def quantize(x):
        if kind == "fp8_block":
            q, sc = fly.blockscale_quant(x, 1, 128)
            return q, sc.t().contiguous().view(-1)
        if kind in ("bf16", "int4_bf16"):
            return x, empty
        return per_token_quant(x, FP8 if kind == "fp8" else torch.int8, stream=st)

    xq, sx = quantize(s["x"])
    s["s1"](s["out1"].view(-1), xq.view(-1), s["w1"], sx, s["sw1"], sid, eid, sw, nv, T, I, D, blocks, st)
    aq, sa = quantize(s["out1"])
    if c["mode"] == "atomic":
        s["out"].zero_()
    s["s2"](s["out"].view(-1), aq.view(-1), s["w2"], sa, s["sw2"], sid, eid, sw, nv, T, D, I, blocks, stream=st)
    return dict(out=s["out"], sorted_ids=sid, sorted_weights=sw, expert_ids=eid, num_valid=post)


def run(state):
    s = state
    op = s["case"]["op"]
    if op == "moe":
        return _moe_layer(s)
    if op == "act_linear":
        c = s["case"]
        out, a_q, sa = quant_gemm(s["x"], s["b"], s["sb"], c["N"], in_dtype=c["kind"], out_dtype=c["out"], out=s["out"],
                                  a_q=s["a_q"], scale_a=s["sa"], stream=s["stream"])
        return dict(out=out, a_q=a_q, scale_a=sa)
    s["gemm"](*s["args"], s["M"], s["N"], s["stream"])
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------------------
def work(case):
    c = case
    if c["op"] == "moe":
        T, D, I, E, k, kind = (c[n] for n in ("tokens", "model_dim", "inter_dim", "experts", "topk", "kind"))
        routes = T * k
        active = E * (1.0 - (1.0 - min(1.0, k / E)) ** T)   # experts that a balanced router reaches
        wb = {"bf16": 2.0, "int4": 0.5, "int4_bf16": 0.5}.get(kind, 1.0)
        scales = 0 if kind == "bf16" else (3 * I * D // 16384 if kind == "fp8_block" else 2 * I + D)
        return {"bytes": active * (3 * I * D * wb + 4 * scales) + 4 * T * D + 8 * routes, "flops": 6 * routes * I * D}
    M, N, K, kind = c["M"], c["N"], c["K"], c["kind"]
    eb = {"bf16": 2.0, "fp16": 2.0, "mxfp4": 0.5 + 1 / 32}
    a = 2.0 if c["op"] == "act_linear" else eb.get(kind, 1.0)
    b = 0.5 if kind == "int4" else eb.get(kind, 1.0)
    scales = {"mxfp4": 0, "bf16": 0, "fp16": 0, "fp8_block": 4 * (M + -(-N // 128)) * (K // 128)}.get(kind, 4 * (M + N))
    if c["op"] == "act_linear":   # the codes are an output too
        scales += M * K
    return {"bytes": a * M * K + b * N * K + 2 * M * N + scales, "flops": 2 * M * N * K}


def tolerance(case):
    # Measured with 64-bit sums over the same quantized operands: outputs are that far off by their own
    # rounding to 16 bits (bf16 1.7e-3, fp16 2.1e-4).  Another order of the fp32 sums moves a small share
    # of them by one rounding.
    if case["op"] == "moe":
        # bf16: atomic sums round in any order (two passes differ by up to 3e-3, 4e-3 off the 64-bit sums);
        # fp16: another rounding of the stage-1 output moves some of the codes that stage 2 reads
        # (two passes 5e-4, one code in 2000 moved 2e-3)
        return {"rel": 1.2e-2 if _moe_types(case["kind"]) == "bf16" else 8e-3}
    return {"rel": 7e-3 if case["out"] == "bf16" else 1e-3}


# ---- the same in 64 bits -----------------------------------------------------------------
def _dequant(w, s, kind):
    """Plain rows of a weight or activation in 64 bits; s: per row or per block, or None."""
    v = w.double()
    if s is None:
        return v
    if kind == "fp8_block":
        rows = s.double().repeat_interleave(128, dim=1)
        br = -(-v.shape[0] // s.shape[0])
        return v * rows.repeat_interleave(br if br == 1 else 128, dim=0)[: v.shape[0]]
    return v * s.double().view(-1, 1)


def _act(x, kind):
    """Activations as the layer sees them after quantization, in 64 bits."""
    if kind in ("bf16", "int4_bf16"):
        return x.double()
    if kind == "fp8_block":
        q, s = _block_quant(x.float(), 1)
        return _dequant(q, s, kind)
    q, s = _row_quant(x.float(), FP8 if kind == "fp8" else torch.int8, 448.0 if kind == "fp8" else 127.0)
    return _dequant(q, s, kind)


def _moe_exact(c, seed):
    x, (w1, sw1), (w2, sw2), ids, tw = _moe_operands(c, seed)
    T, D, I, E, k, kind = (c[n] for n in ("tokens", "model_dim", "inter_dim", "experts", "topk", "kind"))
    xd = _act(x, kind)

    def rows_of(w, s, lo, hi):
        sc = None if s is None else (s[lo // 128:hi // 128] if kind == "fp8_block" else s[lo:hi])
        return _dequant(w[lo:hi], sc, kind)

    h = torch.zeros(T * k, I, dtype=torch.float64, device="cuda")
    flat = ids.view(-1)
    routes = [torch.nonzero(flat == e).view(-1) for e in range(E)]
    for e, r in enumerate(routes):
        if r.numel():
            gu = xd[r // k] @ rows_of(w1, sw1, e * 2 * I, (e + 1) * 2 * I).t().contiguous()
            gate, up = gu[:, :I], gu[:, I:]
            h[r] = gate / (1.0 + torch.exp(-gate)) * up
    hd = _act(h.to(MOE_OUT[_moe_types(kind)]), kind)
    out = torch.zeros(T, D, dtype=torch.float64, device="cuda")
    wt = tw.view(-1).double()
    for e, r in enumerate(routes):
        if r.numel():
            out.index_add_(0, r // k, (hd[r] @ rows_of(w2, sw2, e * D, (e + 1) * D).t().contiguous()) * wt[r][:, None])
    return dict(out=out, sorted_ids=None, sorted_weights=None, expert_ids=None, num_valid=None)


def exact(case, seed):
    c = case
    if c["op"] == "moe":
        return _moe_exact(c, seed)
    a, sa, b, sb = _linear_operands(c, seed)
    M, kind = c["M"], c["kind"]
    if c["op"] == "act_linear":
        q, s = _row_quant(a.float(), FP8 if kind == "fp8" else torch.int8, 448.0 if kind == "fp8" else 127.0)
        out = _dequant(q, s, kind) @ _dequant(b, sb, kind).t().contiguous()
        return dict(out=out, a_q=q.double() if kind == "fp8" else None, scale_a=s.double().view(-1, 1))
    if kind == "mxfp4":
        return _mx_value(a, sa)[:M] @ _mx_value(b, sb).t().contiguous()
    return _dequant(a, sa, kind) @ _dequant(b, sb, kind).t().contiguous()
