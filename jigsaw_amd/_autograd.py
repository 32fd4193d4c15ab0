"""Base of the autograd functions that keep the reference's ``forward`` / ``setup_context`` split."""

from __future__ import annotations

import torch
from torch import _functorch
from torch.autograd import forward_ad

from . import _lib


def native_nodes() -> bool:
    """Whether a :class:`NativeFunction` may stand for a layer's own autograd function: not under a functorch transform or
    forward-mode differentiation, in a trace or in a compiled graph, which know the layer's own."""
    return not (torch._C._are_functorch_transforms_active() or forward_ad._current_level >= 0
                or torch._C._get_tracing_state() is not None or torch.compiler.is_compiling())


def wants_grad(*tensors) -> bool:
    """Whether autograd records what is computed from ``tensors`` (``None`` among them)."""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def saved_rows(ctx) -> tuple:
    """``ctx.saved_tensors`` row-major, as the kernels' pointers take them: hooks of saved tensors (``saved_tensors_hooks``) may have
    given them another layout."""
    return tuple(t if t is None else t.contiguous() for t in ctx.saved_tensors)


class PositionalFunction(torch.autograd.Function):
    """A ``torch.autograd.Function`` with ``setup_context`` whose ``apply`` takes positional arguments as they are.

    ``torch.autograd.Function.apply`` builds and binds the signature of ``forward`` on every call to fill in
    defaults, 5 to 20 us of host time. The functions here have no defaults; functorch transforms and keyword
    calls still take torch's own route."""

    @classmethod
    def apply(cls, *args, **kwargs):
        if kwargs or torch._C._are_functorch_transforms_active():
            return super().apply(*args, **kwargs)
        return super(torch.autograd.Function, cls).apply(*_functorch.utils.unwrap_dead_wrappers(args))


class NativeFunction(torch.autograd.Function):
    """The node behind a result that the native host module has computed already: ``apply(result, saved, rest, *inputs)``
    hands ``result`` out with the module's function ``entry`` as its backward, which finds the tensors ``saved`` and ``rest``
    in the context. Without ``zeros`` an output that nobody used comes as ``None``.

    The node is a Python function's like any other: the collector sees what it keeps (an exchange that keeps the result makes
    a cycle through it), and compiled autograd can record it. A node of a C++ class offers neither. What it leaves out is Python on the way: a layer's own ``forward`` and ``setup_context``, and all of the
    backward, which the engine calls on a thread of its own. Of steps that wait for the host, us on the layer's own function
    : here (: a node in C++): convolution 118 : 102 (: 94), sharded LayerNorm 116 : 100 (: 92), GroupNorm 100 : 74 (: 62, two launches less among
    both), projections 87 : 83 (: 78). The Swin block's 340 stay with it."""

    entry = ""
    zeros = True

    @classmethod
    def apply(cls, result, saved, rest, *inputs):
        if "apply" not in cls._backward_cls.__dict__:
            # the engine calls a context's ``apply``, compiled autograd the class's ``backward``
            cls.backward = cls._backward_cls.apply = getattr(_lib.host(), cls.entry)
        return super(torch.autograd.Function, cls).apply((result,), saved, rest, cls.zeros, *inputs)

    @staticmethod
    def forward(ctx, result, saved, rest, zeros, *inputs):  # noqa: D102
        ctx.save_for_backward(*saved)
        ctx.rest = rest
        if not zeros:
            ctx.set_materialize_grads(False)
        return result[0]
