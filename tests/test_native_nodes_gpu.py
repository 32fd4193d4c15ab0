"""Autograd nodes behind results of the native host module (``_autograd.NativeFunction``) against the functions they stand for, and what
autograd asks of the node of any layer."""

import gc
import itertools
import weakref

import pytest
import torch

from jigsaw_amd import _autograd, _lib, attention, conv, groupnorm, layernorm, projection, swin
from jigsaw_amd.halo import HaloGeometry

pytestmark = pytest.mark.gpu


class Exchange:
    def __init__(self, forward, backward):
        self._forward, self._backward = forward, backward

    def forward(self, send):
        return self._forward

    def backward(self, send):
        if isinstance(self._backward, Exception):
            raise self._backward
        return self._backward


class Half:  # a channel group of two whose other half is the same rows
    def size(self):
        return 2

    def all_reduce(self, t, op):
        if op == "sum":
            t.mul_(2)


def layer(kind, dev, back=None, group=None):
    """(call, differentiable tensors, name of the node) of one layer; its input first, its weight second."""
    group = group or Half()
    gen = torch.Generator(device=dev).manual_seed(3)
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=gen).to(dtype)  # noqa: E731
    size, stride, dtype = {"conv": ((20, 36), 1, torch.bfloat16), "conv of stride 2": ((20, 36), 2, torch.float16),
                           "conv of a volume": ((8, 10, 12), 1, torch.float32)}.get(kind, ((), 1, torch.bfloat16))
    if size:
        n = len(size)
        k, one, s = (3,) * n, (1,) * n, (stride,) * n
        geom = HaloGeometry.for_conv(size, k, s, one, one, one, (3,) * n)
        strips = {v: {o: rand(2, 12, *e) for o in itertools.product((-1, 0, 1), repeat=n) if any(o) and all(e := geom.strip_extent(o, v))}
                  for v in ("assemble", "fold")}
        leaves = [rand(2, 12, *size), rand(24, 12, *k), rand(24)]
        cfg = conv.HipConvNdConfig.for_rank(n, leaves[2], Exchange(strips["assemble"], back or strips["fold"]))
        groups = (conv.TileGroup(3, 1),) * n
        return (lambda x, w, b: conv._ConvNd.apply(x, w, b, s, one, one, groups, None, cfg)[0]), leaves, "ConvNd"
    if kind == "layernorm":
        return (lambda x, w, b: layernorm.layer_norm(x, w, b, group)), [rand(5, 7, 72), rand(72), rand(72)], "LayerNorm"
    if kind == "groupnorm":
        return (lambda x, w, b: groupnorm.group_norm(x, 3, w, b)), [rand(2, 12, 9, 11), rand(12), rand(12)], "GroupNorm"
    if kind == "qkv":
        return (lambda x, w, b: projection.qkv_projection(x, w, b, 2)), [rand(2, 33, 64), rand(192, 64), rand(192)], "Projection"
    if kind == "heads":
        return projection.heads_projection, [rand(2, 2, 33, 32), rand(48, 64), rand(48)], "Projection"
    torch.manual_seed(4)
    block = swin.SwinBlock(64, 2, 8, (16, 24), shift=4, device=dev)

    def call(x, *params):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return torch.func.functional_call(block, dict(zip(names, params)), (x,))

    names = [n for n, _ in block.named_parameters()]
    return call, [rand(1, 16, 24, 64), *(p.detach().clone() for p in block.parameters())], "WholeBlock"


NATIVE = ["conv", "conv of stride 2", "conv of a volume", "layernorm", "groupnorm", "qkv", "heads"]
KINDS = [*NATIVE, "swin"]


def is_native(y):
    return issubclass(type(y.grad_fn)._forward_cls, _autograd.NativeFunction)


def steps(kind, dev, need, monkeypatch, native, hooks=False):
    call, leaves, name = layer(kind, dev)
    if not native:
        for module in (conv, layernorm, groupnorm, projection):
            monkeypatch.setattr(module, "native_nodes", lambda: False)
    leaves = [t.clone().requires_grad_(need[min(i, len(need) - 1)]) for i, t in enumerate(leaves)]
    packed = []
    if hooks:  # what comes back is laid out otherwise
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: torch.stack([t, t], -1)[..., 0]):
            y = call(*leaves)
    else:
        y = call(*leaves)
    assert name in type(y.grad_fn).__name__
    wanted = [t for t in leaves if t.requires_grad]
    off = int(kind != "swin")  # a gradient off the 16-byte grid, which the block composed of its parts refuses
    g = torch.randn(y.numel() + off, device=dev, generator=torch.Generator(device=dev).manual_seed(8)).to(y.dtype)[off:].view_as(y)
    once = torch.autograd.grad(y, wanted, g, retain_graph=kind != "swin")
    if kind != "swin":
        for a, b in zip(once, torch.autograd.grad(y, wanted, g)):
            assert torch.equal(a, b)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, wanted, g)
    return [y.detach(), *once], is_native(y), packed


@pytest.mark.parametrize("need", [n for n in itertools.product((True, False), repeat=3) if any(n)], ids=lambda n: "".join(c for c, on in zip("xwb", n) if on))
@pytest.mark.parametrize("kind", NATIVE)
def test_a_native_node_has_the_bits_of_the_python_function(kind, need, dev, monkeypatch):
    here, native, _ = steps(kind, dev, need, monkeypatch, True)
    assert native
    want, native, _ = steps(kind, dev, need, monkeypatch, False)
    assert not native
    for a, b in zip(here, want, strict=True):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("kind", KINDS[:-1])  # the block keeps nothing through save_for_backward
def test_hooks_of_saved_tensors_see_what_a_native_node_keeps(kind, dev, monkeypatch):
    here, _, packed = steps(kind, dev, (True, True), monkeypatch, True, hooks=True)
    want, _, by_python = steps(kind, dev, (True, True), monkeypatch, False, hooks=False)
    assert len(packed) >= 2
    for a, b in zip(here, want, strict=True):
        assert torch.equal(a, b)


def other_layers(dev):
    """(name, call, leaves) of what has a function of its own beside those of ``layer``."""
    gen = torch.Generator(device=dev).manual_seed(6)
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=gen).bfloat16()  # noqa: E731

    def autocast(call):
        def under(*a):
            with torch.autocast("cuda", dtype=torch.bfloat16):
                return call(*a)
        return under

    block = swin.SwinBlock(64, 2, 8, (16, 24), device=dev, one_node=False)
    norm = lambda x, w, b: layernorm.layer_norm(x, w, b, Half())  # noqa: E731
    groups = lambda x, w, b: groupnorm.group_norm(x, 3, w, b)  # noqa: E731
    return [
        ("linear", projection.linear, [rand(2, 33, 64), rand(48, 64), rand(48)]),
        ("mlp", projection.gelu_mlp, [rand(40, 64), rand(128, 64), rand(128), rand(64, 128), rand(64)]),
        ("heads on top of rows", projection.heads_projection_add, [rand(2, 2, 32, 32), rand(64, 64), rand(64), rand(2, 32, 64)]),
        ("rows that one rank holds", layernorm.plain_layer_norm, [rand(5, 64), rand(64), rand(64)]),
        ("LayerNorm under autocast", autocast(norm), [rand(5, 7, 72), rand(72).float(), rand(72).float()]),
        ("all of LayerNorm's results", lambda x, w, b: layernorm._LayerNorm.apply(x, w, b, Half(), 1e-5)[0], [rand(5, 7, 72), rand(72), rand(72)]),
        ("GroupNorm under autocast", autocast(groups), [rand(2, 12, 9, 11), rand(12).float(), rand(12).float()]),
        ("all of GroupNorm's results", lambda x, w, b: groupnorm._GroupNorm.apply(x, 3, w, b, (), 1e-5)[0], [rand(2, 12, 9, 11), rand(12), rand(12)]),
        ("window attention", attention.window_attention, [rand(2, 2, 64, 32), rand(2, 2, 64, 32), rand(2, 2, 64, 32)]),
        ("block of its parts", autocast(block), [rand(1, 16, 24, 64)]),
    ]


@pytest.mark.parametrize("n", range(10))
def test_hooks_that_hand_back_another_layout_change_no_gradient(n, dev):
    name, call, leaves = other_layers(dev)[n]
    leaves = [t.requires_grad_() for t in leaves]

    def gradients():
        y = call(*leaves)
        g = torch.randn(y.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(8)).to(y.dtype)
        return torch.autograd.grad(y, leaves, g)

    want = gradients()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: torch.stack([t, t], -1)[..., 0]):
        got = gradients()
    for a, b in zip(got, want, strict=True):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("kind", KINDS)
def test_what_a_native_node_refuses(kind, dev):
    call, leaves, _ = layer(kind, dev)
    with torch.no_grad():
        assert not call(*(t.clone().requires_grad_() for t in leaves)).requires_grad
    leaves = [t.requires_grad_() for t in leaves]
    if kind != "swin":
        y = call(*leaves)
        with torch.no_grad():
            leaves[1].add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()
    import torch.autograd.forward_ad as fw

    with fw.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):  # no forward-mode derivative, as on the Python functions
        call(fw.make_dual(leaves[0].detach(), torch.ones_like(leaves[0])), *(t.detach() for t in leaves[1:]))
    with pytest.raises(RuntimeError):  # functorch asks the Python function, which has no rule for its saved tensors or its kernels
        torch.func.vmap(call, in_dims=(0,) + (None,) * (len(leaves) - 1))(torch.stack([leaves[0], leaves[0]]), *leaves[1:])
    assert _autograd.native_nodes()


def test_an_exception_of_the_exchange_arrives_as_it_was_raised(dev):
    call, leaves, _ = layer("conv", dev, back=KeyError("a strip that never came"))
    y = call(*(t.requires_grad_() for t in leaves))
    assert is_native(y)
    with pytest.raises(KeyError, match="a strip that never came"):
        y.sum().backward()


@pytest.mark.parametrize("way", ["forward", "backward"])
def test_strips_in_another_layout_take_the_python_route(way, dev, monkeypatch):
    results = []
    for turned in (False, True):
        call, leaves, _ = layer("conv", dev)
        cell = call.__closure__[[c for c in call.__code__.co_freevars].index("cfg")].cell_contents
        table = getattr(cell.halo_exchange, "_" + way)
        if turned:
            for o, t in table.items():
                table[o] = t.transpose(-1, -2).contiguous().transpose(-1, -2)
        y = call(*(t.requires_grad_() for t in leaves))
        results.append([y.detach(), *torch.autograd.grad(y, leaves, torch.ones_like(y))])
    assert _lib.host() is not None
    for a, b in zip(*results, strict=True):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", KINDS)
def test_a_graph_built_eagerly_runs_backward_under_compiled_autograd(kind, dev):
    from torch._dynamo import compiled_autograd

    call, leaves, _ = layer(kind, dev)
    y = call(*(t.requires_grad_() for t in leaves))
    g = torch.randn(y.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(8)).to(y.dtype)
    want = torch.autograd.grad(y, leaves, g)
    for _ in range(2):  # recorded, and again from the record
        y = call(*leaves)
        for t in leaves:
            t.grad = None
        with compiled_autograd._enable(lambda graph: graph):
            y.backward(g)
        for t, v in zip(leaves, want, strict=True):
            assert torch.equal(t.grad, v)


@pytest.mark.parametrize("kind", ["conv", "layernorm"])
def test_the_collector_frees_a_result_that_its_exchange_keeps(kind, dev):
    group = Half()
    call, leaves, _ = layer(kind, dev, group=group)
    keeper = call.__closure__[[c for c in call.__code__.co_freevars].index("cfg")].cell_contents.halo_exchange if kind == "conv" else group
    keeper.kept = call(*(t.requires_grad_() for t in leaves))
    assert is_native(keeper.kept)
    gone = weakref.ref(keeper)
    del call, leaves, group, keeper
    gc.collect()
    assert gone() is None


@pytest.mark.parametrize("kind", KINDS)
def test_a_wrapper_that_a_transform_left_behind_is_taken(kind, dev):
    call, leaves, _ = layer(kind, dev)
    left = []
    torch.func.grad(lambda t: (left.append(t), t.float().sum())[1])(leaves[0])
    assert torch.equal(call(left[0], *leaves[1:]), call(*leaves))
