"""Which tensors a kernel of this library may take in place of torch's own operators."""
from __future__ import annotations

import contextlib

import torch


def plain_cuda(*ts) -> bool:
    """Tensors whose values a kernel may read and write by pointer in place of torch's own
    operators: ordinary tensors of one GPU, outside autograd, functorch, tracing and dispatch modes."""
    dev = ts[0].device
    if dev.type != "cuda" or any(type(t) is not torch.Tensor or t.device != dev for t in ts):
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        return False
    C = torch._C
    return not (C._len_torch_dispatch_stack() or C._len_torch_function_stack() or torch.compiler.is_compiling()
                or C._get_tracing_state() is not None or C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def on_device(dev):
    """A context in which launches go to ``dev`` (nothing to do when it is current)."""
    return contextlib.nullcontext() if dev.index == torch.cuda.current_device() else torch.cuda.device(dev)
