"""Operators whose autograd node is native (csrc/host_ops.cpp), kept usable where a native node is not enough.

A call normally goes straight to the native operator, which builds its own autograd node when a gradient is wanted.
Two things only a Python ``torch.autograd.Function`` does: ``torch.jit.trace`` records it as one node (the native call
writes its output through raw pointers, which a trace does not see), and it refuses inputs with a tangent or under a
function transform (the native call would drop them in silence).  So while a trace, a forward-mode level or a function
transform is active the call goes through ``forward`` / ``backward`` below, which wrap the native operator."""
import torch
from torch.autograd import forward_ad

_is_tracing = torch._C._is_tracing
_in_transform = torch._C._are_functorch_transforms_active


class NativeOp(torch.autograd.Function):
    """Base class: a subclass defines ``native(*args)``, the direct call, and ``forward(ctx, *args)`` as
    ``return NativeOp.record(ctx, <subclass>.native, args)``."""

    @classmethod
    def apply(cls, *args):
        if _is_tracing() or forward_ad._current_level >= 0 or _in_transform():
            return super().apply(*args)
        return cls.native(*args)

    @staticmethod
    def record(ctx, native, args):
        """``native`` on leaves of its own: its node is kept for ``backward``."""
        ctx.set_materialize_grads(False)
        leaves = [a.detach().requires_grad_() if need else a for a, need in zip(args, ctx.needs_input_grad)]
        with torch.set_grad_enabled(any(ctx.needs_input_grad)):
            outs = native(*leaves)
        ctx.leaves = leaves
        ctx.outs = (outs,) if isinstance(outs, torch.Tensor) else tuple(outs)
        ret = [o if o is None else o.detach() for o in ctx.outs]
        ctx.mark_non_differentiable(*[r for r, o in zip(ret, ctx.outs) if o is not None and not o.requires_grad])
        return ret[0] if isinstance(outs, torch.Tensor) else tuple(ret)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, *grads):
        given = [(o, g) for o, g in zip(ctx.outs, grads) if g is not None]
        wanted = [i for i, need in enumerate(ctx.needs_input_grad) if need]
        result = [None] * len(ctx.leaves)
        if given:
            found = torch.autograd.grad([o for o, _ in given], [ctx.leaves[i] for i in wanted], [g for _, g in given],
                                        retain_graph=True, allow_unused=True)
            for i, g in zip(wanted, found):
                result[i] = g
        return tuple(result)
