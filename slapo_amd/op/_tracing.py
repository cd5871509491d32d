"""What `torch.jit.trace` sees of the ops.

The ops are native functions that allocate below autograd and launch kernels: a tracer that only
watches torch's own operations would store their results in the graph as constants.  While a trace
is being taken an op therefore goes through a `torch.autograd.Function`, which the tracer records as
one node that calls the op again.
"""
from __future__ import annotations

import contextlib

import torch

# The state of the trace being taken, or None: the one test that an untraced call pays.
tracing_state = torch._C._get_tracing_state  # pylint: disable=protected-access


@contextlib.contextmanager
def _untraced():
    state = tracing_state()
    torch._C._set_tracing_state(None)  # pylint: disable=protected-access
    try:
        yield
    finally:
        torch._C._set_tracing_state(state)  # pylint: disable=protected-access


class _RecordedOp(torch.autograd.Function):
    """`_RecordedOp.apply(fn, *args)` is `fn(*args)`, recorded where a trace is being taken.  The
    node holds `apply`: outside a trace, when the graph runs, that is `fn` and nothing else."""

    # pylint: disable=arguments-differ, abstract-method
    @classmethod
    def apply(cls, fn, *args):
        if tracing_state() is None:
            return fn(*args)
        return super().apply(fn, *args)

    @staticmethod
    def forward(ctx, fn, *args):
        with _untraced():  # on leaves of its own: what an op does inside is no part of the trace
            ctx.leaves = [arg.detach().requires_grad_(need) if isinstance(arg, torch.Tensor)
                          else arg for arg, need in zip(args, ctx.needs_input_grad[1:])]
            with torch.enable_grad():
                ctx.out = fn(*ctx.leaves)
            like = dict(size=tuple(ctx.out.shape), dtype=ctx.out.dtype, device=ctx.out.device)
        # the tracer wants to have seen the result made; anything else it would keep as a constant
        result = torch.empty(**like)
        with _untraced():
            return result.copy_(ctx.out)

    @staticmethod
    def backward(ctx, grad):
        grads = [None] * len(ctx.leaves)
        wanted = [i for i, need in enumerate(ctx.needs_input_grad[1:]) if need]
        if ctx.out.requires_grad:
            with _untraced():
                found = torch.autograd.grad([ctx.out], [ctx.leaves[i] for i in wanted], [grad],
                                            retain_graph=True, allow_unused=True)
            for i, g in zip(wanted, found):
                grads[i] = g
        return (None, *grads)


record = _RecordedOp.apply
