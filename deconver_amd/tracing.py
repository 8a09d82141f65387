"""The compiled autograd nodes under ``torch.jit.trace``.

The tracer records calls of the dispatcher and of Python autograd functions.  A compiled node is
neither: recorded through, its result is the uninitialised buffer its kernel was to fill.  While a
trace is being recorded every call of a node therefore goes through one Python function, which the
recorded graph calls again when it runs.
"""

from __future__ import annotations

import functools

import torch

__all__ = ["RecordedNodes"]


class _RecordedNode(torch.autograd.Function):
    """One call of a compiled node, by name.  It keeps the node's own small autograd graph, on
    detached inputs, and differentiates through that."""

    @staticmethod
    def forward(ctx, native, name, *args):
        needs = ctx.needs_input_grad[2:]
        state = torch._C._get_tracing_state()
        torch._C._set_tracing_state(None)      # what happens inside is not recorded
        try:
            leaves = [a.detach().requires_grad_(n) if torch.is_tensor(a) else a for a, n in zip(args, needs)]
            with torch.enable_grad():
                out = getattr(native, name)(*leaves)
            results = [t if t is None else t.detach() for t in (out if isinstance(out, tuple) else (out,))]
        finally:
            torch._C._set_tracing_state(state)
        # (a result needs an operation of its own in the record, or it is taken for a constant)
        results = [t if t is None else t.view(t.shape) for t in results]
        if any(needs):
            ctx.wanted = [i for i, n in enumerate(needs) if n]
            ctx.leaves, ctx.out = leaves, out
        return tuple(results) if isinstance(out, tuple) else results[0]

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, *gouts):
        out = ctx.out if isinstance(ctx.out, tuple) else (ctx.out,)
        grads = torch.autograd.grad(out, [ctx.leaves[i] for i in ctx.wanted], gouts, retain_graph=True, allow_unused=True)
        result = [None] * len(ctx.leaves)
        for i, g in zip(ctx.wanted, grads):
            result[i] = g
        return (None, None, *result)


class RecordedNodes:
    """The functions of the native module, each call as one recorded Python function."""

    def __init__(self, native):
        self._native = native

    def __getattr__(self, name):
        return functools.partial(_RecordedNode.apply, self._native, name)
