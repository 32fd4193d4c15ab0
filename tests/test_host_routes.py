"""The native host module of the distributed convolution beside the Python route it shortens."""

import itertools
import sys

import pytest
import torch

from jigsaw_amd import _lib
from jigsaw_amd import conv as jc
from jigsaw_amd.halo import HaloGeometry


def test_a_host_module_that_does_not_load_leaves_the_python_route(monkeypatch):
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setitem(sys.modules, "jigsaw_amd._host", None)  # import raises ImportError
    monkeypatch.delattr("jigsaw_amd._host", raising=False)
    jc._step.cache_clear()
    try:
        with pytest.warns(RuntimeWarning, match="_host.so"):
            step = jc._step((1, 4, 8, 8), torch.float32, (4, 4, 3, 3), (1, 1), (1, 1), (1, 1), (0, 0), (2, 2), 1, True)
        assert step is None and _lib.host() is None  # said once
    finally:
        jc._step.cache_clear()


class _Held:
    """The halo exchange of a rank whose neighbours' strips are here already."""

    def __init__(self, fwd, bwd):
        self.fwd, self.bwd, self.sent = fwd, bwd, []

    def forward(self, send):
        self.sent.append(send)
        return self.fwd

    def backward(self, send):
        self.sent.append(send)
        return self.bwd


ROUTE_CASES = [
    # size, batch, c_in, c_out, kernel, stride, padding, mesh, rank, groups, dtype, bias
    ((16, 24), 2, 3, 16, 3, 1, 1, 3, 1, 1, torch.float32, True),
    ((16, 64), 2, 64, 64, 3, 1, 1, 3, 1, 1, torch.bfloat16, True),    # the fused fold
    ((17, 23), 1, 40, 72, 3, 1, 1, 2, 0, 1, torch.bfloat16, True),    # the fold of its own
    ((16, 32), 2, 32, 64, 3, 2, 1, 2, 1, 1, torch.bfloat16, False),   # stride 2
    ((12, 16), 1, 4, 6, 3, 1, 0, 2, 1, 1, torch.float16, True),       # halos that differ from rank to rank
    ((6, 8, 16), 1, 32, 32, 3, 1, 1, 3, 1, 1, torch.bfloat16, True),
    ((8, 12), 2, 6, 9, 3, 1, 1, 3, 1, 3, torch.float32, True),        # grouped
    ((8, 12), 2, 6, 9, 3, 1, 1, 1, 0, 1, torch.float32, True),        # nothing to exchange
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ROUTE_CASES, ids=lambda c: f"{c[2]}to{c[3]}_{'x'.join(map(str, c[0]))}_s{c[5]}_mesh{c[7]}")
def test_native_and_python_route_of_a_step_agree_bit_for_bit(case, monkeypatch):
    size, batch, ci, co, k, s, p, mesh, rank, cgroups, dtype, bias = case
    dev, n = torch.device("cuda:0"), len(size)
    torch.manual_seed(3)
    kernel, stride, padding, dilation = (k,) * n, (s,) * n, (p,) * n, (1,) * n
    geom = HaloGeometry.for_conv(size, kernel, stride, padding, dilation, (rank,) * n, (mesh,) * n)
    mk = lambda *shape: torch.randn(*shape, device=dev).to(dtype)  # noqa: E731
    present = [o for o in itertools.product((-1, 0, 1), repeat=n) if any(o) and all(0 <= rank + v < mesh for v in o)]
    strips = [{o: mk(batch, ci, *geom.strip_extent(o, verb)) for o in present} for verb in ("assemble", "fold")]
    x, w = mk(batch, ci, *size).requires_grad_(), mk(co, ci // cgroups, *kernel).requires_grad_()
    b = mk(co).requires_grad_() if bias else None
    spatial = tuple(jc.TileGroup(mesh, rank) for _ in size)
    made = []
    step_for = jc._step_for

    def run(native):
        def chosen(*a):
            made.append(step_for(*a))
            return made[-1] if native else None

        monkeypatch.setattr(jc, "_step_for", chosen)
        held = _Held(*strips)
        y, x_aug = jc._ConvNd.apply(x, w, b, stride, padding, dilation, spatial, None,
                                    jc.HipConvNdConfig.for_rank(n, b, held, groups=cgroups))
        torch.manual_seed(4)
        grads = torch.autograd.grad(y, [t for t in (x, w, b) if t is not None], mk(*y.shape))
        return [y, x_aug, *grads, *(d[o] for d in held.sent for o in sorted(d))]

    native, python = run(True), run(False)
    assert all(m is not None for m in made), "the native route does not take this case"
    assert len(native) == len(python)
    for a, c in zip(native, python):
        assert a.shape == c.shape and a.dtype == c.dtype and torch.equal(a, c)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [c for c in ROUTE_CASES if c[9] == 1 and c[7] > 1], ids=lambda c: f"{c[2]}to{c[3]}_{'x'.join(map(str, c[0]))}_s{c[5]}_mesh{c[7]}")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_the_python_route_writes_the_input_gradient_to_its_owners_for_every_type(case, dtype, monkeypatch):
    """Without the native module too: one launch for the input gradient, the tile's part and the strips, with the bits of the
    separate steps."""
    size, batch, ci, co, k, s, p, mesh, rank = case[:9]
    dev, n = torch.device("cuda:0"), len(size)
    torch.manual_seed(6)
    kernel, stride, padding, dilation = (k,) * n, (s,) * n, (p,) * n, (1,) * n
    geom = HaloGeometry.for_conv(size, kernel, stride, padding, dilation, (rank,) * n, (mesh,) * n)
    mk = lambda *shape: torch.randn(*shape, device=dev).to(dtype)  # noqa: E731
    present = [o for o in itertools.product((-1, 0, 1), repeat=n) if any(o) and all(0 <= rank + v < mesh for v in o)]
    strips = [{o: mk(batch, ci, *geom.strip_extent(o, verb)) for o in present} for verb in ("assemble", "fold")]
    x, w = mk(batch, ci, *size).requires_grad_(), mk(co, ci, *kernel)
    fold, taken = jc._input_fold, []
    monkeypatch.setattr(jc, "_step_for", lambda *a: None)
    monkeypatch.setattr(jc, "_input_fold", lambda *a, **kw: taken.append(fold(*a, **kw)) or taken[-1])
    res = []
    for fused in (True, False):
        held = _Held(*strips)
        y, _ = jc._ConvNd.apply(x, w, None, stride, padding, dilation, tuple(jc.TileGroup(mesh, rank) for _ in size), None,
                                jc.HipConvNdConfig.for_rank(n, None, held, fused_fold=fused))
        torch.manual_seed(7)
        gx, = torch.autograd.grad(y, x, mk(*y.shape))
        res.append((gx, *(d[o] for d in held.sent for o in sorted(d))))
    assert len(taken) == 1 and taken[0] is not None
    for a, c in zip(*res):
        assert torch.equal(a, c)


@pytest.mark.gpu
@pytest.mark.parametrize("ci, co, size, dtype, held", [
    (40, 72, (97, 120), torch.bfloat16, True),     # partials alone
    (24, 40, (480, 500), torch.float32, False),    # sums of bf16 parts: copies of both tensors beside the partials
    (8, 8, (24, 64, 96), torch.float32, False),    # all part products in one block: no sums are left
], ids=str)
def test_a_step_holds_no_more_of_the_weight_gradients_scratch_than_the_sums_left_need(ci, co, size, dtype, held):
    """The weight gradient's scratch makes room for the input gradient, unless sums over it are left for the border's launch: then it is
    64 MiB at most."""
    dev, n, lib = torch.device("cuda:0"), len(size), _lib.load()
    kernel, ones, ranks, mesh = (3,) * n, (1,) * n, (0,) * n, (2,) * n
    x_shape, w_shape = (1, ci, *size), (co, ci, *kernel)
    geom = HaloGeometry.for_conv(size, kernel, ones, ones, ones, ranks, mesh)
    assert lib.jg_halo_fold_border_takes_sums(geom.theirs().c_geom(ci), _lib.dtype_code(dtype)) == 1
    step = jc._step(x_shape, dtype, w_shape, ones, ones, ones, ranks, mesh, 1, True)
    local = jc._local_padding(ones, mesh)
    ws_x, ws_w = (jc._launch_for(op, dtype, x_shape[:2] + geom.padded, w_shape, ones, local, ones, 1).nbytes for op in (1, 2))
    mk = lambda *shape: torch.randn(*shape, device=dev).to(dtype)  # noqa: E731
    x_aug, w, g = mk(*x_shape[:2], *geom.padded), mk(*w_shape), mk(1, co, *size)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    parts = step.backward(g, x_aug, w, True, True, True, _lib.stream_handle(dev))
    peak = torch.cuda.max_memory_allocated() - before
    gx, gw, gb, send, folded, left = parts
    assert folded and (left is not None) == held
    step.finish(gx, folded, {}, _lib.stream_handle(dev), left)
    results = sum(t.numel() * t.element_size() for t in (gx, gw, gb, *send.values()))
    room = 6 << 20  # the allocator leaves up to 1 MiB behind a block of more than that as part of it
    assert peak <= room + (ws_w + ws_x + results if held else max(ws_w + gw.numel() * 4, ws_x + results))
    assert not held or ws_w <= 64 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_norms_and_rings_by_the_native_and_the_python_route_agree_bit_for_bit(dtype, monkeypatch):
    from jigsaw_amd import attention, groupnorm, layernorm

    dev = torch.device("cuda:0")

    class Half:  # a channel group of two whose other half is the same rows
        def size(self):
            return 2

        def all_reduce(self, t, op):
            if op == "sum":
                t.mul_(2)

    def leaf(*shape):
        return torch.randn(*shape, device=dev, generator=gen).to(dtype).requires_grad_()

    def steps():
        res = []
        for group, bias in ((None, True), (Half(), True), (Half(), False)):
            x, w, b = leaf(3, 37, 72), leaf(72), leaf(72) if bias else None
            y, x_norm, _, var = layernorm._LayerNorm.apply(x, w, b, group, 1e-5)
            res += [y, x_norm, var, *torch.autograd.grad(y, [t for t in (x, w, b) if t is not None], torch.ones_like(y) * x)]
            res += [layernorm.layer_norm(x, w, b, group).detach()]
        for affine in (True, False):
            x, w, b = leaf(2, 12, 9, 11), leaf(12) if affine else None, leaf(12) if affine else None
            y = groupnorm.group_norm(x, 3, w, b)
            res += [y, *torch.autograd.grad(y, [t for t in (x, w, b) if t is not None], torch.ones_like(y) * x)]
        for shape, sk, P in (((2, 3, 70, 32), 50, 3), ((1, 2, 128, 64), 128, 2)):
            q, ks, vs = leaf(*shape), [leaf(*shape[:2], sk, shape[3]) for _ in range(P)], [leaf(*shape[:2], sk, shape[3]) for _ in range(P)]
            out, lse = attention.ring_forward(q, ks, vs, 0.3, rank=1)
            dq, dk, dv = attention.ring_backward(leaf(*shape), q, out, lse, ks, vs, 0.3)
            assert not out.requires_grad and not dq.requires_grad
            res += [out, lse, dq, *dk, *dv]
        return res

    gen = torch.Generator(device=dev).manual_seed(5)
    native = steps()
    monkeypatch.setattr(_lib, "host", lambda: None)
    gen = torch.Generator(device=dev).manual_seed(5)
    python = steps()
    assert len(native) == len(python)
    for a, c in zip(native, python):
        assert a.shape == c.shape and a.dtype == c.dtype and a.is_contiguous() == c.is_contiguous() and torch.equal(a, c)


@pytest.mark.gpu
def test_the_native_route_declines_what_needs_a_copy():
    host, dev = _lib.host(), torch.device("cuda:0")
    stream = _lib.stream_handle(dev)
    q = torch.randn(2, 3, 64, 64, device=dev).bfloat16()
    k = [torch.randn(2, 3, 32, 64, device=dev).bfloat16()]
    assert host.ring_forward(q, k, k, 1.0, stream) is not None
    odd = torch.empty(q.numel() + 1, dtype=q.dtype, device=dev)[1:].view_as(q)  # not on a 16-byte boundary
    for bad_q, bad_k in ((q.transpose(1, 2), k), (odd, k), (q.float(), k), (q, [k[0].half()]), (q, []), (q, k * 17), (q[0], k),
                         (q[..., :36].contiguous(), [k[0][..., :36].contiguous()]), (q, [k[0][:, :2]])):
        assert host.ring_forward(bad_q, bad_k, bad_k, 1.0, stream) is None
        assert host.ring_backward(q, bad_q, q, torch.zeros(2, 3, 64, device=dev), bad_k, bad_k, 1.0, stream) is None
    assert host.ring_backward(q, q, q, torch.zeros(2, 3, 64, device=dev).half(), k, k, 1.0, stream) is None
    assert host.ring_forward(torch.zeros(1, 1, 4096, 32, device=dev).bfloat16(), [torch.zeros(1, 1, 4096, 32, device=dev).bfloat16()] * 2,
                             [torch.zeros(1, 1, 4096, 32, device=dev).bfloat16()] * 2, 1.0, stream) is None  # attention._as_64_columns is asked first
    x = torch.randn(4, 6, device=dev)
    assert host.ln_partial(x.t(), False, stream) is None and host.ln_partial(x.double(), False, stream) is None
    assert host.gn_forward(x.half(), 2, torch.ones(6, device=dev), None, 1e-5, False, stream) is None  # another type


def test_the_native_route_asks_about_every_head_that_may_be_better_off_as_64_columns():
    """The rule for zero columns has one place, ``attention._as_64_columns``; the native module takes no such head unasked."""
    from jigsaw_amd import attention

    may = _lib.host().may_want_64_columns
    yes = 0
    for d, sq, sk, P, lead in itertools.product((8, 16, 24, 32, 40, 56, 64, 96), (1024, 2040, 2048, 4096, 8192), (512, 2048, 4096, 4104),
                                                (1, 2, 4, 16), ((1, 1), (1, 8), (2, 16), (4, 64))):
        q, k = torch.empty(*lead, sq, d, dtype=torch.bfloat16, device="meta"), torch.empty(*lead, sk, d, dtype=torch.bfloat16, device="meta")
        wants = attention._as_64_columns(q, k, P)
        yes += wants
        assert may(d, sq, sk * P) or not wants, (d, sq, sk, P, lead)
    assert yes > 50 and not may(32, 128, 256)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(40, 2048, 32), (33, 2048, 48)], ids=str)
def test_narrow_heads_with_many_rows_take_the_native_route(shape, monkeypatch):
    from jigsaw_amd import attention

    heads, n, d = shape
    dev = torch.device("cuda:0")
    torch.manual_seed(2)
    q, dout, *kv = (torch.randn(1, heads, n, d, device=dev).bfloat16() for _ in range(6))
    assert not attention._as_64_columns(q, kv[0], 2)

    def run():
        out, lse = attention.ring_forward(q, kv[:2], kv[2:], 0.2)
        dq, dk, dv = attention.ring_backward(dout, q, out, lse, kv[:2], kv[2:], 0.2)
        return [out, lse, dq, *dk, *dv]

    with monkeypatch.context() as m:
        m.setattr(attention, "_pointers", None)  # the Python route's pointer tables
        native = run()
    monkeypatch.setattr(_lib, "host", lambda: None)
    for a, c in zip(native, run(), strict=True):
        assert torch.equal(a, c)
