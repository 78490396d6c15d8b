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
    grad = torch.is_grad_enabled()
    for t in ts:
        if type(t) is not torch.Tensor or t.layout is not torch.strided or t.is_neg() or (grad and t.requires_grad):
            return False
    C = torch._C
    return not (C._len_torch_dispatch_stack() or C._len_torch_function_stack() or C._get_tracing_state() is not None
                or C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def plain_cuda(*ts) -> bool:
    """Tensors whose values a kernel may read and write by pointer in place of torch's own
    operators: ``plain`` ones of one GPU."""
    if not plain(*ts):
        return False
    index = ts[0].get_device()
    for t in ts:
        if not t.is_cuda or t.get_device() != index:
            return False
    return True


def on_device(dev):
    """A context in which launches go to ``dev`` (nothing to do when it is current)."""
    return contextlib.nullcontext() if dev.index == torch.cuda.current_device() else torch.cuda.device(dev)
