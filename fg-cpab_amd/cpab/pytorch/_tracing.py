"""The native autograd functions under ``torch.jit.trace``.

The tracer does not see a native autograd function: it records the allocation of
its output and none of the work, so that a traced call would return memory that
nothing wrote.  While a trace is recorded the call goes through a Python autograd
function instead, which the tracer keeps as one operation and runs again with the
traced module's inputs (and which ``torch.jit.save`` refuses to export).
"""
import torch

__all__ = ["recorded"]


def recorded(function, *args):
    """``function(*args)``, kept as one operation by a trace in progress.

    The tracer compares a call's arguments by their text when it checks a trace:
    ``function`` is a module's, with everything it needs in ``args``.
    """
    if torch.jit.is_tracing():
        return _Recorded.apply(function, *args)
    return function(*args)


class _Recorded(torch.autograd.Function):
    """A native function with a graph of its own, held from forward to backward."""

    @staticmethod
    def forward(ctx, function, *args):
        with torch.enable_grad():
            ctx.args = [a.detach().requires_grad_(need) if isinstance(a, torch.Tensor) else a
                        for a, need in zip(args, ctx.needs_input_grad[1:])]
            ctx.out = function(*ctx.args)
        return ctx.out.detach()

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad):
        wanted = [i for i, need in enumerate(ctx.needs_input_grad[1:]) if need]
        grads = torch.autograd.grad(ctx.out, [ctx.args[i] for i in wanted], grad,
                                    retain_graph=True, allow_unused=True)
        found = dict(zip(wanted, grads))
        return (None, *(found.get(i) for i in range(len(ctx.args))))
