"""Calls of the native autograd nodes (csrc/otx_autograd.cpp), as ``torch.jit.trace`` can follow them.

The tracer records dispatched operators and Python autograd functions.  A native
node's launch is neither: the trace would keep only the allocation of its output.
While a trace is recorded the call therefore goes through ``_Traced``, which the
tracer records as one operation.
"""

from __future__ import annotations

import torch

from .. import _lib

__all__ = ["call", "tracing"]


def tracing() -> bool:
    return torch._C._get_tracing_state() is not None


class _Traced(torch.autograd.Function):
    """The node ``name`` and the graph it makes, in one Python autograd function."""

    @staticmethod
    def forward(ctx, name, *args):
        needs = ctx.needs_input_grad[1:]
        with torch.enable_grad():
            ctx.ins = [a.detach().requires_grad_(n) if isinstance(a, torch.Tensor) else a for a, n in zip(args, needs)]
            ctx.outs = getattr(_lib.autograd(), name)(*ctx.ins)
        if isinstance(ctx.outs, tuple):
            return tuple(y.detach() for y in ctx.outs)
        return ctx.outs.detach()

    @staticmethod
    def backward(ctx, *grads):
        wrt = [a for a in ctx.ins if isinstance(a, torch.Tensor) and a.requires_grad]
        got = iter(torch.autograd.grad(ctx.outs, wrt, grads, retain_graph=True))
        return None, *(next(got) if isinstance(a, torch.Tensor) and a.requires_grad else None for a in ctx.ins)


def call(name: str, *args):
    if tracing():
        return _Traced.apply(name, *args)
    return getattr(_lib.autograd(), name)(*args)
