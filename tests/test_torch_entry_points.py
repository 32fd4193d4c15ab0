"""The places where this package goes round torch's public calls: what each stands in for, so that a torch that changes
one fails here by name."""

import pytest
import torch

from jigsaw_amd import layernorm as jl
from jigsaw_amd._autograd import PositionalFunction
from jigsaw_amd.halo import HaloGeometry, new_strips, slot


class _Twice(PositionalFunction):
    generate_vmap_rule = True

    @staticmethod
    def forward(x, factor):
        return x * factor

    @staticmethod
    def setup_context(ctx, inputs, output):
        ctx.factor = inputs[1]
        ctx.save_for_backward(inputs[0])

    @staticmethod
    def backward(ctx, g):
        assert ctx.saved_tensors[0].shape == g.shape
        return g * ctx.factor, None


class _TwiceTorch(_Twice):
    apply = classmethod(lambda cls, *a, **k: torch.autograd.Function.apply.__func__(cls, *a, **k))


def test_positional_functions_do_what_torchs_own_apply_does():
    assert callable(torch._C._are_functorch_transforms_active) and callable(torch._functorch.utils.unwrap_dead_wrappers)
    results = []
    for fn in (_Twice, _TwiceTorch):
        x = torch.arange(6.0).view(2, 3).requires_grad_()
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
            y = fn.apply(x, 2.0)
        grad, = torch.autograd.grad(y, x, torch.ones_like(y))
        under_vmap = torch.func.vmap(lambda t: fn.apply(t, 2.0))(x.detach())
        under_grad = torch.func.grad(lambda t: fn.apply(t, 2.0).sum())(x.detach())
        with torch.no_grad():
            quiet = fn.apply(x, 2.0)
        results.append([y, grad, under_vmap, under_grad, torch.tensor(len(packed)), torch.tensor(quiet.requires_grad)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_strips_cut_from_one_buffer_are_what_as_strided_gives():
    geom = HaloGeometry.for_conv((5, 7), (3, 3), (1, 1), (1, 1), (1, 1), (1, 1), (3, 3))
    for dtype in (torch.float32, torch.bfloat16):
        strips, tab = new_strips(geom, "pack_fwd", (2, 3), geom.offsets(), dtype, torch.device("cpu"))
        ends = []
        for o, t in strips.items():
            assert tuple(t.shape) == (2, 3, *geom.strip_extent(o, "pack_fwd")) and t.is_contiguous() and t.dtype == dtype
            assert tab[slot(o)] == t.data_ptr()
            assert t.storage_offset() * t.element_size() % 256 == 0
            ends.append((t.storage_offset(), t.storage_offset() + t.numel()))
        ends.sort()
        assert all(a[1] <= b[0] for a, b in zip(ends, ends[1:])), "strips overlap"


class _Ctx:
    def mark_non_differentiable(self, *t): ...

    def set_materialize_grads(self, on): ...

    def save_for_backward(self, *t):
        self.saved = t


def test_the_root_handed_over_on_var_may_be_missing():
    """LayerNorm hands the root its kernel formed to setup_context as an attribute of ``var``; an output that arrives there
    without it (a wrapper of some transform) gets the root taken again."""
    x, w, var = torch.randn(4, 6), torch.ones(6), torch.rand(4, 1) + 0.5
    ctx = _Ctx()
    jl._LayerNorm.setup_context(ctx, (x, w, None, None, 1e-5), (x, x, w, var))
    assert torch.equal(ctx.saved[2], var.sqrt())
    var._jg_std = std = torch.rand(4, 1)
    jl._LayerNorm.setup_context(ctx, (x, w, None, None, 1e-5), (x, x, w, var))
    assert ctx.saved[2] is std


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_the_root_handed_over_on_var_is_its_root(dtype):
    x = torch.randn(33, 64, device="cuda").to(dtype)
    w, b = (torch.randn(64, device="cuda").to(dtype) for _ in range(2))
    var = jl._LayerNorm.forward(x, w, b, None, 1e-5)[3]
    assert torch.allclose(var._jg_std, var.float().sqrt(), rtol=1e-6, atol=0)
