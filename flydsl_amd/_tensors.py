"""Which tensors a kernel of this library may take in place of torch's own operators."""
from __future__ import annotations

import contextlib

import torch


def plain(*ts) -> bool:
    """Ordinary dense tensors (no subclass, no pending negation), outside autograd, functorch, tracing
    and dispatch modes: a kernel sees in their memory what an operator would see in the tensors."""
    # first of all: torch.compile can trace this question, and none of those about torch's mode stacks
    if torch.compiler.is_compiling():
        return False
    if any(type(t) is not torch.Tensor or t.layout is not torch.strided or t.is_neg() for t in ts):
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        return False
    C = torch._C
    return not (C._len_torch_dispatch_stack() or C._len_torch_function_stack() or C._get_tracing_state() is not None
                or C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def plain_cuda(*ts) -> bool:
    """Tensors whose values a kernel may read and write by pointer in place of torch's own
    operators: ``plain`` ones of one GPU."""
    dev = ts[0].device
    return dev.type == "cuda" and all(t.device == dev for t in ts) and plain(*ts)


def on_device(dev):
    """A context in which launches go to ``dev`` (nothing to do when it is current)."""
    return contextlib.nullcontext() if dev.index == torch.cuda.current_device() else torch.cuda.device(dev)
