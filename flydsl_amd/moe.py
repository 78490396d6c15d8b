"""Routing metadata for the MoE 2-stage GEMM: ``moe_sorting`` groups the routes of a top-k
routing by expert and pads each expert's run to the GEMM's row block.

Same outputs as the reference harness's ``moe_sorting_torch_native``
(``tests/kernels/test_moe_gemm.py:97-160``), computed without a per-expert loop or a host
synchronisation, so it runs on the device tensors it is given:

* ``sorted_ids`` int32 ``[tokens*topk + E*block - topk]``: per expert in order, its routes in
  row-major order of ``topk_ids`` as ``(slot << 24) | token``, padded to a multiple of ``block``
  with ``(topk << 24) | tokens``;
* ``sorted_weights`` fp32, aligned with ``sorted_ids`` (0 in the padding);
* ``sorted_expert_ids`` int32 ``[ceil(len(sorted_ids) / block)]``: the expert of each block,
  -1 past the last;
* ``num_tokens_post_pad`` int32 ``[2]``: the padded row count and ``tokens``.

With ``expert_mask`` (0/1 per expert), routes to masked experts are dropped and the remaining
experts are renumbered consecutively, as in the reference.
"""
from __future__ import annotations

import torch

from . import _lib
from ._tensors import on_device, plain_cuda


def _sort_kernel(topk_ids, topk_weights, E, bs, expert_mask):
    """moe_sorting through flygemm_moe_sort (one or two launches, no synchronisation)."""
    dev = topk_ids.device
    M, topk = topk_ids.shape
    max_pad = M * topk + E * bs - topk
    ids = topk_ids if topk_ids.dtype in (torch.int32, torch.int64) else topk_ids.to(torch.int64)
    ids, w = ids.contiguous(), topk_weights.to(torch.float32).contiguous()
    mask = None if expert_mask is None else (expert_mask.reshape(-1)[:E].to(torch.int64) != 0).contiguous()
    sorted_ids = torch.empty(max_pad, dtype=torch.int32, device=dev)
    sorted_w = torch.empty(max_pad, dtype=torch.float32, device=dev)
    sorted_eids = torch.empty((max_pad + bs - 1) // bs, dtype=torch.int32, device=dev)
    post = torch.empty(2, dtype=torch.int32, device=dev)
    lib = _lib.load()
    n = lib.flygemm_moe_sort_scratch(M, topk, E)
    scratch = torch.empty(n, dtype=torch.int32, device=dev) if n else None
    rc = lib.flygemm_moe_sort(sorted_ids.data_ptr(), sorted_w.data_ptr(), sorted_eids.data_ptr(), post.data_ptr(),
                              scratch.data_ptr() if n else None, ids.data_ptr(), w.data_ptr(),
                              None if mask is None else mask.data_ptr(), M, topk, E, bs,
                              int(ids.dtype == torch.int64), torch.cuda.current_stream(dev).cuda_stream)
    _lib.check(rc, "flygemm_moe_sort")
    return sorted_ids, sorted_w, sorted_eids, post


def moe_sorting(topk_ids: torch.Tensor, topk_weights: torch.Tensor, num_experts: int, block_size: int,
                expert_mask: torch.Tensor | None = None):
    if topk_ids.dim() != 2 or topk_weights.shape != topk_ids.shape:
        raise ValueError(f"topk_ids / topk_weights must both be [tokens, topk], got {tuple(topk_ids.shape)} "
                         f"and {tuple(topk_weights.shape)}")
    E, bs = int(num_experts), int(block_size)
    if E <= 0 or bs <= 0:
        raise ValueError(f"num_experts={E} and block_size={bs} must be positive")
    dev = topk_ids.device
    M, topk = topk_ids.shape
    max_pad = M * topk + E * bs - topk
    # On the GPU: the counting-sort kernel (csrc/moe_sort.hip) in place of about 40 operators, two
    # of which (bincount, torch.tensor) wait for the device.  Measured on MI355X, calls back to
    # back: 8 tokens, 256 experts, top-8 16.5 us against 400; 8192 tokens, 128 experts, top-8 21 against 440-460.
    # More experts than the kernel's counters, a top-k above the experts (whose rows may not fit
    # the buffers), empty routings and masks shorter than the experts take the operators below.
    if (0 < topk <= E <= _lib.MOE_SORT_MAX_EXPERTS and M > 0 and max_pad < 2**31 - 2**16
            and (expert_mask is None or expert_mask.numel() >= E)
            and plain_cuda(*(t for t in (topk_ids, topk_weights, expert_mask) if t is not None))):
        with on_device(dev):
            return _sort_kernel(topk_ids, topk_weights, E, bs, expert_mask)
    max_blocks = (max_pad + bs - 1) // bs

    flat = topk_ids.reshape(-1).to(torch.int64)
    route = torch.arange(M * topk, device=dev, dtype=torch.int64)     # t * topk + s
    keep = (flat >= 0) & (flat < E)
    local = torch.arange(E, device=dev, dtype=torch.int64)
    if expert_mask is not None:
        m = expert_mask.to(device=dev).reshape(-1)[:E].to(torch.int64) != 0
        keep = keep & m[flat.clamp(0, E - 1)]
        local = torch.cumsum(m.to(torch.int64), 0) - 1                # renumbered id of kept experts
    key = torch.where(keep, flat, torch.full_like(flat, E))           # dropped routes sort last
    key_sorted, order = torch.sort(key, stable=True)
    counts = torch.bincount(key, minlength=E + 1)[:E]
    padded = (counts + bs - 1) // bs * bs
    start = torch.cumsum(padded, 0) - padded                          # first row of each expert
    first = torch.cumsum(counts, 0) - counts                          # first sorted route of each expert

    n_keep = M * topk  # routes past the kept ones carry key E and are discarded below
    j = torch.arange(n_keep, device=dev, dtype=torch.int64)
    valid = key_sorted < E
    e_of = key_sorted.clamp(max=E - 1)
    dest = torch.where(valid, start[e_of] + (j - first[e_of]), torch.full_like(j, max_pad))

    t = order // topk
    s = order % topk
    sorted_ids = torch.full((max_pad + 1,), (topk << 24) | M, device=dev, dtype=torch.int64)
    sorted_ids[dest] = (s << 24) | t
    sorted_w = torch.zeros(max_pad + 1, device=dev, dtype=torch.float32)
    sorted_w[dest] = topk_weights.reshape(-1).to(torch.float32)[order]

    # expert of each block: blocks [start_e / bs, (start_e + padded_e) / bs) belong to expert e
    blk_end = torch.cumsum(padded // bs, 0)                           # exclusive end block per expert
    b = torch.arange(max_blocks, device=dev, dtype=torch.int64)
    e_blk = torch.searchsorted(blk_end, b, right=True)
    sorted_eids = torch.where(e_blk < E, local[e_blk.clamp(max=E - 1)], torch.full_like(b, -1))

    post = torch.stack([padded.sum(), torch.tensor(M, device=dev, dtype=torch.int64)]).to(torch.int32)
    return sorted_ids[:max_pad].to(torch.int32), sorted_w[:max_pad], sorted_eids.to(torch.int32), post
