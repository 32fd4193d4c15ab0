"""Spatially sharded GroupNorm: HIP kernels (through the C ABI) against the oracle.

The shards of a spatial split run one after the other in this process; the all-reduces
of a shard see the other shards' contributions through a stand-in group that holds them
(computed in fp64 from the same inputs), in the order the operator asks for them:
(count, sum), centred squares, and in the backward the two per-group sums.
Tolerances: rel-L2 <= 1e-5 in fp32, 2e-2 in bf16.
"""

import math

import pytest
import torch

from helpers import rel_l2
from jigsaw_amd import groupnorm as jgn
from oracle import groupnorm as ogn

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


class Others:
    """Stand-in process group: adds what the other ranks would contribute to each sum."""

    def __init__(self, contributions):
        self.contributions, self.calls = list(contributions), 0

    def size(self):
        return 2

    def all_reduce(self, t, op):
        assert op == "sum"
        t += self.contributions[self.calls].to(device=t.device, dtype=t.dtype)
        self.calls += 1


CASES = [
    # global shape, groups, dtype, weight, bias, shards along the first spatial axis
    ((2, 8, 6, 10), 4, torch.float32, True, True, 2),
    ((1, 6, 6, 7, 3), 3, torch.float32, True, False, 3),       # odd extents: element-wise path
    ((2, 64, 64, 64), 8, torch.bfloat16, True, True, 2),
    ((1, 4, 256, 300), 2, torch.float32, True, True, 2),       # long spans: several chunks per group and row
    ((3, 16, 8, 8), 16, torch.float32, False, False, 2),       # one channel per group, no affine
    ((2, 32, 32, 48), 4, torch.bfloat16, False, True, 4),
    ((2, 12, 10, 16), 3, torch.float16, True, True, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}_g{c[1]}_{str(c[2]).split('.')[-1]}_p{c[5]}")
def test_sharded_groupnorm_matches_oracle(case, dev):
    shape, G, dtype, has_w, has_b, P = case
    torch.manual_seed(5)
    X = (torch.randn(*shape) * 1.5 + 0.3).to(dtype)
    W = (1 + 0.2 * torch.randn(shape[1])).to(dtype) if has_w else None
    B = (0.2 * torch.randn(shape[1])).to(dtype) if has_b else None
    GR = torch.randn(*shape).to(dtype)
    eps = 1e-5
    xs, gs = list(X.chunk(P, dim=2)), list(GR.chunk(P, dim=2))
    xd, gd = [t.double() for t in xs], [t.double() for t in gs]
    wd, bd = (None if W is None else W.double()), (None if B is None else B.double())
    outs, rstd, n = ogn.forward(xd, G, wd, bd, eps)
    back = ogn.backward(gd, [o[1] for o in outs], rstd, n, G, wd)

    # what every shard contributes to the three sums (fp64)
    N = shape[0]
    seg = [t.reshape(N, G, -1) for t in xd]
    mean = (sum(t.sum(-1) for t in seg) / n.squeeze(-1)).unsqueeze(-1)
    c1 = [torch.stack([torch.full((N, G), float(t.shape[-1]), dtype=torch.float64), t.sum(-1)], -1) for t in seg]
    c2 = [((t - mean) ** 2).sum(-1) for t in seg]
    gg = [(g if wd is None else g * wd.reshape((1, -1) + (1,) * (g.dim() - 2))).reshape(N, G, -1) for g in gd]
    xn = [o[1].reshape(N, G, -1) for o in outs]
    c3 = [torch.stack([a.sum(-1), (a * b).sum(-1)], -1) for a, b in zip(gg, xn)]

    tol = TOL[dtype]
    for i in range(P):
        others = Others([sum(c[j] for j in range(P) if j != i) for c in (c1, c2, c3)])
        x = xs[i].to(dev).requires_grad_()
        w = None if W is None else W.to(dev).requires_grad_()
        b = None if B is None else B.to(dev).requires_grad_()
        y, x_norm, rstd_g, n_g = jgn._GroupNorm.apply(x, G, w, b, (others,), eps)
        assert y.dtype == dtype and not x_norm.requires_grad
        assert rel_l2(y, outs[i][0]) < tol and rel_l2(x_norm, outs[i][1]) < tol
        assert rel_l2(rstd_g, rstd) < tol and torch.equal(n_g.double().cpu(), n)
        y.backward(gs[i].to(dev))
        assert others.calls == 3
        gx, gw, gb = back[i]
        assert rel_l2(x.grad, gx) < tol
        if has_w:
            assert rel_l2(w.grad, gw) < tol
        if has_b:
            assert rel_l2(b.grad, gb) < tol


def test_unsharded_groupnorm_equals_torch(dev):
    """No spatial groups: the operator is F.group_norm, forward and backward; under bf16
    autocast it computes in fp32 (promote_to_fp32_under_autocast)."""
    torch.manual_seed(6)
    x = torch.randn(2, 12, 9, 11)
    w, b = 1 + 0.1 * torch.randn(12), 0.1 * torch.randn(12)
    g = torch.randn_like(x)
    xd, wd, bd = (t.double().requires_grad_() for t in (x, w, b))
    want = torch.nn.functional.group_norm(xd, 3, wd, bd, 1e-5)
    want.backward(g.double())
    xg, wg, bg = (t.to(dev).requires_grad_() for t in (x, w, b))
    y = jgn.group_norm(xg, 3, wg, bg, (), 1e-5)
    y.backward(g.to(dev))
    assert rel_l2(y, want) < 1e-5 and rel_l2(xg.grad, xd.grad) < 1e-5
    assert rel_l2(wg.grad, wd.grad) < 1e-5 and rel_l2(bg.grad, bd.grad) < 1e-5
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y16 = jgn.group_norm(xg.detach().bfloat16(), 3, wg.detach(), bg.detach(), (), 1e-5)
    assert y16.dtype == torch.float32
    want16 = torch.nn.functional.group_norm(x.bfloat16().double(), 3, w.double(), b.double(), 1e-5)
    assert rel_l2(y16, want16) < 1e-5


def test_groupnorm_argument_errors(dev):
    x = torch.zeros(1, 6, 4, 4, device=dev)
    with pytest.raises(ValueError):
        jgn.group_norm(x, 4)


@pytest.mark.parametrize("case", CASES + [
    ((1, 4, 1, 1), 2, torch.bfloat16, True, True, 1), ((2, 6, 3, 7), 2, torch.bfloat16, True, True, 1),
    ((3, 8, 1, 257), 4, torch.float16, True, False, 1), ((2, 4, 513, 130), 2, torch.bfloat16, False, False, 1),
    ((40, 8, 640, 650), 4, torch.bfloat16, True, True, 1),
], ids=str)
def test_group_norm_without_x_norm(case, dev):
    """``group_norm`` (statistics from one pass, x_hat recomputed in the backward) whole and sharded: rows that start off
    the 16-byte grid, spans of one element, spans of many chunks, a mean far above the spread, more samples than one
    step of the last-level cache takes."""
    shape, G, dtype, has_w, has_b, P = case
    torch.manual_seed(9)
    big = math.prod(shape) > 1 << 24
    x = (torch.randn(*shape, device=dev) * 0.5 + (0.3 if dtype != torch.float32 else 40.0)).to(dtype)
    w = (1 + 0.2 * torch.randn(shape[1], device=dev)).to(dtype) if has_w else None
    b = (0.2 * torch.randn(shape[1], device=dev)).to(dtype) if has_b else None
    g = torch.randn(*shape, device=dev).to(dtype)
    ref = torch.float32 if big else torch.float64
    leaves = [None if t is None else t.to(ref).requires_grad_() for t in (x, w, b)]
    affine = [torch.ones(shape[1], device=dev, dtype=ref) if leaves[1] is None else leaves[1], leaves[2]]  # torch's own backward wants a weight
    want = torch.nn.functional.group_norm(leaves[0], G, *affine, 1e-5)
    grads = torch.autograd.grad(want, [t for t in leaves if t is not None], g.to(ref))
    tol = max(TOL[dtype], 2e-5)
    got_leaves = [None if t is None else t.clone().requires_grad_() for t in (x, w, b)]
    y = jgn.group_norm(got_leaves[0], G, got_leaves[1], got_leaves[2])
    got = torch.autograd.grad(y, [t for t in got_leaves if t is not None], g)
    assert y.dtype == dtype and rel_l2(y, want) < tol
    for a, r in zip(got, grads):
        assert a.dtype == dtype and (rel_l2(a, r) < tol or r.norm() < 1e-6 * g.norm())
    if P == 1:
        return

    class Half:  # the other shards' (count, sum), centred squares and backward sums, added to this one's
        def __init__(self, parts):
            self.parts = list(parts)

        def size(self):
            return P

        def all_reduce(self, t, op):
            t += self.parts.pop(0).to(t.dtype)

    xs, gs = [t.double() for t in x.chunk(P, 2)], [t.double() for t in g.chunk(P, 2)]
    seg = [t.reshape(shape[0], G, -1) for t in xs]
    n = sum(t.shape[-1] for t in seg)
    mean = sum(t.sum(-1) for t in seg) / n
    sq = [((t - mean[..., None]) ** 2).sum(-1) for t in seg]
    rstd = (sum(sq) / n + 1e-5) ** -0.5
    wd = torch.ones(shape[1], device=dev, dtype=torch.float64) if w is None else w.double()
    gw_ = [(t * wd.reshape(1, -1, *[1] * (len(shape) - 2))).reshape(shape[0], G, -1) for t in gs]
    xn = [(t - mean[..., None]) * rstd[..., None] for t in seg]
    rest = lambda f: sum(f(i) for i in range(1, P))  # noqa: E731
    others = Half([rest(lambda i: torch.stack([torch.full_like(mean, seg[i].shape[-1]), seg[i].sum(-1)], -1)), rest(lambda i: sq[i]),
                   rest(lambda i: torch.stack([gw_[i].sum(-1), (gw_[i] * xn[i]).sum(-1)], -1))])
    x0 = x.chunk(P, 2)[0].clone().requires_grad_()
    y0 = jgn.group_norm(x0, G, w, b, (others,))
    g0, = torch.autograd.grad(y0, x0, g.chunk(P, 2)[0])
    assert not others.parts and rel_l2(y0, want.chunk(P, 2)[0]) < tol and rel_l2(g0, grads[0].chunk(P, 2)[0]) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 8, 16, 24), (1, 6, 7, 9)], ids=str)  # rows on and off the 16-byte grid
@pytest.mark.parametrize("sharded", [False, True])
def test_input_changed_in_place_before_the_backward(shape, dtype, sharded, dev):
    """``x += group_norm(x)`` and an activation in place on the result: the backward has what it needs of its own."""
    torch.manual_seed(5)
    leaf = torch.randn(*shape, device=dev).to(dtype).requires_grad_()
    w = (1 + 0.2 * torch.randn(shape[1], device=dev)).to(dtype).requires_grad_()
    b = (0.2 * torch.randn(shape[1], device=dev)).to(dtype).requires_grad_()
    g = torch.randn(*shape, device=dev).to(dtype)

    class Alone:  # a spatial group whose other ranks hold nothing
        def size(self):
            return 2

        def all_reduce(self, t, op):
            pass

    x = leaf * 1
    y = jgn.group_norm(x, 2, w, b, (Alone(),) if sharded else ())
    x += y
    grads = torch.autograd.grad(x, (leaf, w, b), g)
    ref = [t.detach().double().requires_grad_() for t in (leaf, w, b)]
    want = ref[0] + torch.nn.functional.group_norm(ref[0], 2, ref[1], ref[2], 1e-5)
    for a, r in zip(grads, torch.autograd.grad(want, ref, g.double())):
        assert rel_l2(a, r) < max(TOL[dtype], 2e-5)
    assert rel_l2(x, want) < TOL[dtype]


OWN_CHOICE = 2**32 - 1  # for `polls`: what group_norm takes, a whole group a block where that covers the tensor


@pytest.mark.parametrize("polls", [0, 1, 256, OWN_CHOICE])  # separate launches; nearly every chunk left to the second launch; hardly any; group_norm's
@pytest.mark.parametrize("shape", [
    # batch, channels, groups, positions; a block keeps 16384 (backward) or 32768 (forward) 16-bit elements, half as many fp32
    (2, 6, 3, 1), (2, 6, 2, 7), (1, 8, 2, 4097), (1, 4, 2, 16384), (2, 4, 2, 16385), (1, 2, 1, 32777),
    (1, 8, 1, 9 * 16384 + 5),                         # more chunks than every block adds up itself
    (1, 64, 2, 16 * 16384), (1, 33, 1, 16 * 16384),   # the most chunks of a group that wait for each other; more
    (40, 8, 4, 8 * 16384 - 8),                        # more blocks than fit the chip
    (1, 64, 8, 1 << 20),                              # tensors that go past the last-level cache
], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_chunks_kept_in_registers(shape, dtype, polls, dev):
    """The launches behind ``group_norm`` at the edges of their chunks, whether the blocks of a group meet or not."""
    from jigsaw_amd import _lib

    N, C, G, S = shape
    gen = torch.Generator(device=dev).manual_seed(3)
    x = (torch.randn(N, C, S, device=dev, generator=gen) * 0.5 + 0.3).to(dtype)
    g = torch.randn(N, C, S, device=dev, generator=gen).to(dtype)
    w = (1 + 0.2 * torch.randn(C, device=dev, generator=gen)).to(dtype)
    b = (0.2 * torch.randn(C, device=dev, generator=gen)).to(dtype)
    lib, p, code = _lib.load(), _lib.ptr, _lib.dtype_code(dtype)
    y, kept, gx = (torch.full_like(x, float("nan")) for _ in range(3))
    stats = torch.full((2, N, G), float("nan"), device=dev)
    gw, gb = torch.full((2, C), float("nan"), device=dev).unbind(0)
    nbytes = lib.jg_gn_workspace_bytes(N, C, S)
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device=dev)
    rc = lib.jg_gn_forward_polls(p(y), p(kept), p(stats[0]), p(stats[1]), p(x), p(w), p(b), N, C, S, G, 1e-5, code, polls, p(ws), nbytes,
                                 _lib.stream_ptr(dev))
    assert rc == 0
    rc = lib.jg_gn_backward_polls(p(gx), p(gw), p(gb), p(g), p(x), p(stats[0]), p(stats[1]), p(w), N, C, S, G, code, _lib.dtype_code(gw.dtype),
                                  polls, p(ws), nbytes, _lib.stream_ptr(dev))
    assert rc == 0 and torch.equal(kept, x)
    # in fp64, x_hat rounded as the operator rounds it on the way to y
    xd, gd = x.double().reshape(N, G, -1), (g.double() * w.double()[:, None]).reshape(N, G, -1)
    mean = xd.mean(-1, keepdim=True)
    rstd = ((xd - mean).square().mean(-1, keepdim=True) + 1e-5).rsqrt()
    xn = (xd - mean) * rstd
    want_gx = rstd * (gd - gd.mean(-1, keepdim=True) - xn * (gd * xn).mean(-1, keepdim=True))
    xn = xn.reshape(N, C, S)
    # a rounding to 16 bits of x_hat and one of y (2^-8 bf16, 2^-11 fp16, halved, of values up to 1.5 of the rms); fp32 sums
    tol = {torch.bfloat16: 4e-3, torch.float16: 5e-4, torch.float32: 3e-6}[dtype]
    assert rel_l2(y, xn * w.double()[:, None] + b.double()[:, None]) < tol
    assert rel_l2(stats[0], mean.squeeze(-1)) < 3e-6 and rel_l2(stats[1], rstd.squeeze(-1)) < 3e-6
    # gx is a difference of terms of the size of rstd g w, which cancel where a group has few elements (two: all but eps)
    err, term = (gx.double() - want_gx.reshape(N, C, S)).abs(), (rstd * gd).abs()
    assert err.norm() < tol * term.norm() and err.max() < 8 * tol * term.max()
    scale = math.sqrt(N * S)  # what a sum of N S values of both signs is measured against
    assert (gw - (g.double() * xn).sum((0, 2))).abs().max() < 1e-5 * scale + 1e-6 * math.sqrt(N * S) * scale
    assert (gb - g.double().sum((0, 2))).abs().max() < 1e-5 * scale + 1e-6 * math.sqrt(N * S) * scale


def _whole_tensor(shape, dtype, dev):
    """Inputs of the launches behind ``group_norm`` and a function (polls) -> every tensor that they write."""
    from jigsaw_amd import _lib

    N, C, G, S = shape
    gen = torch.Generator(device=dev).manual_seed(4)
    x, g = (torch.randn(N, C, S, device=dev, generator=gen).add_(0.3).to(dtype) for _ in range(2))
    w, b = (torch.randn(C, device=dev, generator=gen).to(dtype) for _ in range(2))
    lib, p, code, nbytes = _lib.load(), _lib.ptr, _lib.dtype_code(dtype), _lib.load().jg_gn_workspace_bytes(N, C, S)

    def run(polls):
        y, kept, gx = (torch.full_like(x, float("nan")) for _ in range(3))
        stats, grads = torch.full((2, N, G), float("nan"), device=dev), torch.full((2, C), float("nan"), device=dev)
        ws, stream = torch.full((nbytes,), 255, dtype=torch.uint8, device=dev), _lib.stream_ptr(dev)
        assert lib.jg_gn_forward_polls(p(y), p(kept), p(stats[0]), p(stats[1]), p(x), p(w), p(b), N, C, S, G, 1e-5, code, polls, p(ws), nbytes,
                                       stream) == 0
        assert lib.jg_gn_backward_polls(p(gx), p(grads[0]), p(grads[1]), p(g), p(x), p(stats[0]), p(stats[1]), p(w), N, C, S, G, code,
                                        _lib.dtype_code(grads.dtype), polls, p(ws), nbytes, stream) == 0
        return {"y": y, "kept": kept, "gx": gx, "stats": stats, "grads": grads}

    run.x = x
    return run


@pytest.mark.parametrize("shape", [
    (2, 6, 2, 7), (1, 8, 2, 4097), (1, 4, 2, 16385),
    (1, 8, 1, 9 * 16384 + 5),   # more chunks than every block adds up itself
    (4, 32, 4, 93300),
    (1, 64, 2, 16 * 16384),     # the most chunks of a group that wait for each other
], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_the_launch_that_writes_a_chunk_does_not_show(shape, dtype, dev):
    """A chunk whose block gave up waiting (all but a few at one poll) and one whose block did not have the same bits."""
    run = _whole_tensor(shape, dtype, dev)
    want = run(256)
    for polls in (1, 2, 8):
        for name, t in run(polls).items():
            assert torch.equal(t, want[name]), f"{name} at {polls} polls"


@pytest.mark.parametrize("shape", [
    # batch, channels, groups, positions: the edges of a block that keeps a whole group, forward (4 x 32768 16-bit elements) and backward (half of it)
    (1, 1, 1, 1), (3, 6, 2, 7), (2, 4, 1, 16384), (2, 8, 2, 16385), (1, 2, 1, 32768), (5, 2, 1, 32769), (1, 1, 1, 4 * 16384 - 1), (1, 2, 2, 4 * 16384 + 9),
    (2, 3, 1, 32767), (1, 1, 1, 4 * 32768), (1, 5, 1, 100), (9, 32, 32, 211),
], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_a_group_that_one_block_keeps_has_the_bits_of_several(shape, dtype, dev):
    """What group_norm takes, where small groups meet in LDS, and the same with blocks that wait for each other."""
    run = _whole_tensor(shape, dtype, dev)
    got, want = run(OWN_CHOICE), run(256)
    for name, t in got.items():
        assert not t.isnan().any() and torch.equal(t, want[name]), name


@pytest.mark.parametrize("shape", [(2, 8, 4, 1000), (1, 4, 2, 16384), (3, 4, 4, 40001)], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_infinities_and_nan_stay_in_their_group(shape, dtype, dev):
    """x with one infinity in the first group and one NaN in the last: those come out without a finite value, the others as without
    them, and a block that keeps a whole group has the same results as blocks that wait for each other."""
    N, C, G, S = shape
    run = _whole_tensor(shape, dtype, dev)
    clean = run(OWN_CHOICE)
    run.x[0, 0, S // 2], run.x[N - 1, C - 1, S - 1] = float("inf"), float("nan")
    got, want = run(OWN_CHOICE), run(256)
    sick = torch.zeros(N, G, dtype=torch.bool, device=dev)
    sick[0, 0] = sick[N - 1, G - 1] = True
    for name in ("y", "kept", "gx", "stats"):
        a, b, c = (t[name].permute(1, 2, 0) if name == "stats" else t[name].view(N, G, -1) for t in (got, want, clean))
        assert torch.equal(a.nan_to_num(nan=7.0), b.nan_to_num(nan=7.0)) and torch.equal(a[~sick], c[~sick]), name
        assert name == "kept" or not a[sick][..., :1].isfinite().any(), name
    a, b = got["grads"], want["grads"]
    assert torch.equal(a.nan_to_num(nan=7.0), b.nan_to_num(nan=7.0)) and a[1].isfinite().all()


def test_a_busy_chip_does_not_show_in_the_results(dev):
    """Beside a kernel of another stream that keeps four fifths of the compute units, where blocks do give up, bit for bit what
    the same call gives alone; and again on the free chip after it."""
    from jigsaw_amd import attention

    run = _whole_tensor((2, 64, 2, 1 << 18), torch.bfloat16, dev)
    want = run(128)
    q, k = (torch.randn(1, 200, n, 64, device=dev).bfloat16() for n in (128, 8192))  # 200 workgroups, about 1 ms a call
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        busy = [attention.ring_forward(q, [k] * 16, [k] * 16, 0.125) for _ in range(3)]
    got = [run(128) for _ in range(3)]
    torch.cuda.synchronize()
    got.append(run(128))
    assert busy[0][0].isfinite().all()
    for results in got:
        for name, t in results.items():
            assert torch.equal(t, want[name]), name


def test_blocks_wait_again_once_the_chip_is_free(dev):
    """What gives up waiting beside a kernel of another stream that leaves less room than a group needs does not send the rest of
    the tensor, whose blocks have the chip to themselves, through the second launch."""
    from jigsaw_amd import _lib, attention

    N, C, G, S, chunk = 8, 64, 8, 1 << 20, 32768  # 256 chunks a group; 224 places beside the other kernel
    lib, p = _lib.load(), _lib.ptr
    x = torch.randn(N, C, S, device=dev, dtype=torch.bfloat16)
    y, stats, w = torch.empty_like(x), torch.empty(2, N, G, device=dev), torch.ones(C, device=dev, dtype=torch.bfloat16)
    nbytes = lib.jg_gn_workspace_bytes(N, C, S)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    q, k = (torch.randn(1, 200, n, 64, device=dev).bfloat16() for n in (128, 8192))
    side, chunks = torch.cuda.Stream(), N * C * S // chunk
    for calls in (0, 1, 1):
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(calls):
                attention.ring_forward(q, [k] * 4, [k] * 4, 0.125)  # about 0.25 ms
        assert lib.jg_gn_forward(p(y), p(stats[0]), p(stats[1]), p(x), p(w), p(w), N, C, S, G, 1e-5, _lib.dtype_code(x.dtype), p(ws), nbytes,
                                 _lib.stream_ptr(dev)) == 0
        torch.cuda.synchronize()
        left = int(ws.view(torch.int32)[2 * (chunks + N * G)])  # behind a word for every chunk and every group
        assert left < chunks // 2, f"{left} of {chunks} chunks beside {calls} calls"


def test_group_norm_in_a_captured_graph(dev):
    """Replays with other inputs, eager work in between, against the eager result."""
    torch.manual_seed(8)
    x, g = (torch.randn(2, 32, 64, 130, device=dev).bfloat16() for _ in range(2))
    w = (1 + 0.2 * torch.randn(32, device=dev)).bfloat16().requires_grad_()
    x.requires_grad_()
    step = lambda: (lambda y: [y, *torch.autograd.grad(y, (x, w), g)])(jgn.group_norm(x, 4, w))  # noqa: E731
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        with torch.no_grad():
            x.copy_(torch.randn_like(x))
        graph.replay()
        got = [t.clone() for t in out]
        for a, r in zip(got, step()):
            assert torch.equal(a, r)
