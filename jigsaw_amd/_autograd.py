"""Base of the autograd functions that keep the reference's ``forward`` / ``setup_context`` split."""

from __future__ import annotations

import torch
from torch import _functorch


def native_nodes() -> bool:
    """Whether a layer may leave its autograd node to the native host module: not under a functorch transform, in a trace or in
    a compiled graph, which know the Python functions."""
    return not (torch._C._are_functorch_transforms_active() or torch._C._get_tracing_state() is not None or torch.compiler.is_compiling())


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
