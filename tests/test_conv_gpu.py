"""HIP convolution kernels against the oracle (torch CPU operators in fp64) (GPU).

Tolerances (rel-L2 of the whole tensor): fp32 tensors 1e-5 and bf16 tensors 2e-2, as the north-star
states, fp16 tensors 2e-3; the reference's own conv tests use atol/rtol 1e-4 for
y / dx / db and a looser bound for dw (tests/modules/convolution/conv/test_conv2d_multi_spatial.py:207-233).
"""

import itertools

import pytest
import torch

from helpers import conv_geometry, mesh_coords, neighbour, rel_l2
from jigsaw_amd import _lib
from jigsaw_amd import conv as jc
from jigsaw_amd.halo import halo_pack
from oracle import conv as oc
from oracle import halo as oh

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 2e-3}

PRIM_CASES = [
    # (N, Cin, Cout, in spatial, kernel, stride, padding, dilation)
    (2, 3, 16, (18, 18), (3, 3), (1, 1), (0, 0), (1, 1)),
    (2, 16, 3, (18, 20), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 5, 7, (13, 11), (3, 2), (2, 1), (1, 0), (1, 2)),
    (2, 4, 4, (9, 9), (1, 1), (1, 1), (0, 0), (1, 1)),
    (2, 4, 6, (12, 12), (5, 5), (1, 1), (2, 2), (1, 1)),
    (1, 3, 5, (40,), (3,), (1,), (1,), (1,)),
    (1, 4, 6, (8, 9, 10), (3, 3, 3), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    (2, 3, 4, (7, 8, 9), (3, 1, 2), (1, 2, 1), (1, 0, 1), (1, 1, 1)),
    (2, 64, 64, (18, 34), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 32, (10, 10, 18), (3, 3, 3), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    (1, 64, 64, (20, 70), (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 64, 64, (37, 53), (3, 3), (1, 1), (0, 0), (1, 1)),
    # several stages per workgroup, strips that start in the middle of a workgroup's range
    (2, 64, 64, (260, 131), (3, 3), (1, 1), (0, 0), (1, 1)),
    (2, 32, 32, (6, 70, 130), (3, 3, 3), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    (1, 32, 64, (131, 200), (3, 3), (1, 1), (1, 1), (1, 1)),
    # row lengths of whole cache lines: the input gradient's tile grid moves so that its staged rows start on
    # a line (an odd distance: staged from one pixel earlier), the first tile column mostly hangs out of the tensor
    (2, 32, 32, (20, 128), (3, 3), (1, 1), (1, 1), (1, 1)),
    (1, 64, 64, (35, 192), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 16, (4, 18, 64), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    # weight gradient: several stages per workgroup with column strips of unequal cost (windows that stick out
    # across W, a last strip with fewer columns), odd padding across even rows (staged one pixel early)
    (2, 64, 64, (150, 330), (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 32, 32, (140, 200), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 32, (5, 40, 136), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    # weight gradient without padding over whole stages (even rows, 64-column strips), every window inside x: the
    # kernel without the border path, whose stage loop loads and stores without conditions. One stage per
    # workgroup, two or three (the load cursor stops at the last one), each channel blocking
    (2, 64, 64, (4, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 64, 64, (1030, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (2, 64, 64, (8, 130), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 64, (262, 130), (3, 3), (1, 1), (0, 0), (1, 1)),
    (2, 64, 32, (6, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 32, (518, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 32, 32, (5, 260, 66), (3, 3, 3), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    # channel counts beyond one group of LDS-resident weights, and produced channels that are
    # not a multiple of the 32-row MFMA tile (padded with zero weight rows, not stored)
    (1, 128, 128, (20, 70), (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 16, 3, (37, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 48, 80, (33, 40), (3, 3), (1, 1), (1, 1), (1, 1)),
    (1, 256, 64, (18, 34), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 96, 32, (5, 18, 34), (3, 3, 3), (1, 1, 1), (1, 0, 1), (1, 1, 1)),
    (1, 80, 16, (4, 20, 36), (3, 3, 3), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    # contraction channels that are not a multiple of the 16-channel MFMA step (first / last layers)
    (2, 69, 64, (37, 66), (3, 3), (1, 1), (0, 0), (1, 1)),
    (1, 64, 69, (20, 70), (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 20, 24, (5, 18, 34), (3, 3, 3), (1, 1, 1), (1, 0, 1), (1, 1, 1)),
    # non-overlapping kernels (patch embeddings, 1 x 1): a GEMM over the patches in bf16
    (2, 8, 16, (16, 24), (4, 4), (4, 4), (0, 0), (1, 1)),
    (2, 16, 32, (9, 11), (1, 1), (1, 1), (0, 0), (1, 1)),
    (2, 8, 8, (17, 19), (4, 4), (4, 4), (0, 0), (1, 1)),
    (1, 4, 8, (4, 8, 10), (2, 2, 2), (2, 2, 2), (0, 0, 0), (1, 1, 1)),
    (3, 72, 264, (64, 48), (8, 8), (8, 8), (0, 0), (1, 1)),
    (2, 16, 32, (20, 36), (2, 2), (2, 2), (0, 0), (1, 1)),
    # extents 1 or 3 at stride 1: embedded in the 3 x 3 (x 3) MFMA kernels
    (2, 64, 64, (20, 70), (1, 1), (1, 1), (0, 0), (1, 1)),
    (1, 16, 24, (19, 33), (1, 3), (1, 1), (0, 1), (1, 1)),
    (2, 8, 5, (12, 40), (3, 1), (1, 1), (1, 0), (1, 1)),
    (1, 16, 16, (5, 10, 34), (1, 1, 1), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    (1, 8, 8, (6, 9, 20), (3, 1, 3), (1, 1, 1), (1, 0, 0), (1, 1, 1)),
    # strided 3 x 3 (down-sampling): kernels of their own at 2 x 2, else the stride-1 kernels, sampled / zero-stuffed
    (2, 16, 32, (33, 40), (3, 3), (2, 2), (1, 1), (1, 1)),
    (1, 8, 8, (20, 31), (3, 3), (2, 3), (0, 1), (1, 1)),
    (1, 8, 16, (7, 12, 18), (3, 3, 3), (2, 2, 2), (1, 1, 1), (1, 1, 1)),
    (2, 8, 8, (16, 16), (1, 1), (2, 2), (0, 0), (1, 1)),
    # dilated 3-tap kernels whose padding is a multiple of the dilation: the residue images as batch
    # entries of the undilated MFMA kernels (extents that the dilation does and does not divide)
    (2, 32, 64, (33, 47), (3, 3), (1, 1), (2, 3), (2, 3)),
    (1, 64, 64, (40, 64), (3, 3), (1, 1), (0, 0), (2, 2)),
    (2, 16, 8, (21, 30), (3, 3), (1, 1), (4, 0), (2, 1)),
    (1, 8, 16, (9, 3), (3, 1), (1, 1), (4, 0), (4, 5)),
    (1, 32, 32, (6, 19, 34), (3, 3, 3), (1, 1, 1), (1, 2, 2), (1, 2, 2)),
    (2, 16, 32, (33, 40), (3, 3), (2, 2), (2, 2), (2, 2)),   # strided and dilated
    (1, 4, 6, (17, 23), (3, 3), (1, 1), (1, 1), (2, 2)),     # padding not a multiple: the direct kernels
    # more than three taps on an axis: tap blocks of three as channel blocks of a three-tap layer
    (1, 16, 32, (20, 33), (5, 5), (1, 1), (2, 2), (1, 1)),
    (2, 8, 8, (15, 18), (7, 7), (1, 1), (3, 3), (1, 1)),
    (1, 8, 16, (12, 14), (4, 4), (2, 2), (1, 1), (1, 1)),
    (1, 6, 4, (13, 16), (1, 5), (1, 1), (0, 0), (1, 1)),
    (2, 4, 6, (11, 9), (5, 2), (1, 1), (4, 1), (1, 1)),
    (1, 4, 6, (6, 9, 10), (5, 3, 3), (1, 1, 1), (2, 1, 1), (1, 1, 1)),
    (1, 3, 5, (14, 14), (7, 7), (2, 2), (3, 3), (1, 1)),     # a 7 x 7 stem at stride 2
    # grouped layers (ninth entry: groups), depthwise among them: the direct kernels
    (2, 8, 12, (13, 17), (3, 3), (1, 1), (1, 1), (1, 1), 4),
    (1, 32, 32, (20, 22), (3, 3), (1, 1), (1, 1), (1, 1), 32),
    (2, 6, 9, (11, 14), (3, 5), (2, 1), (1, 2), (1, 2), 3),
    (1, 16, 16, (5, 9, 10), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 2),
    (2, 64, 64, (18, 34), (3, 3), (1, 1), (0, 0), (1, 1), 2),   # a shape the MFMA kernels would take ungrouped
    (1, 12, 8, (30,), (5,), (1,), (2,), (1,), 4),
    # dilated kernels of more than three taps (residue images on the tap-block route), a padding that is no multiple of
    # the dilation (the remainder as a rim of zeros around the input), two taps an axis (a block with a zero tap in front)
    (2, 3, 5, (15, 18), (5, 3), (1, 1), (4, 2), (2, 2)),
    (1, 4, 6, (13, 17), (3, 3), (1, 1), (1, 3), (2, 2)),
    (2, 5, 4, (14, 15), (3, 3), (2, 2), (1, 1), (2, 3)),
    (1, 6, 7, (9, 11), (2, 2), (1, 1), (1, 0), (1, 1)),
    (1, 3, 4, (6, 7, 8), (1, 2, 2), (1, 1, 1), (0, 1, 1), (1, 1, 1)),
    (2, 4, 4, (12, 12), (2, 2), (1, 1), (0, 0), (2, 2)),
    # groups of at least 8 channels a side: each group as an ungrouped layer of its own (matrix cores, and the routes above)
    (2, 48, 32, (20, 22), (3, 3), (2, 2), (1, 1), (1, 1), 2),
    (1, 32, 64, (17, 19), (5, 5), (1, 1), (2, 2), (1, 1), 4),
    (1, 24, 24, (6, 10, 12), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 2, 2), 3),
    # fp32: few channels or a few beyond a multiple of 16 (the part products of all blocks counted through); several
    # tiles of produced channels that share the chip, with more and with fewer pixel tiles than it has compute units
    (2, 3, 5, (40, 71), (3, 3), (1, 1), (1, 1), (1, 1)),
    (1, 17, 33, (19, 66), (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 5, 65, (36, 70), (3, 3), (2, 2), (1, 1), (1, 1)),
    (1, 4, 8, (5, 18, 20), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    (3, 8, 160, (129, 200), (3, 3), (1, 1), (1, 1), (1, 1)),
]


def _pid(c):
    name = "n{}_ci{}_co{}_in{}_k{}_s{}_p{}_d{}".format(c[0], c[1], c[2], *["x".join(map(str, v)) for v in c[3:8]])
    return name + (f"_g{c[8]}" if len(c) > 8 else "")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", PRIM_CASES, ids=_pid)
def test_conv_primitives_match_oracle(case, dtype, dev):
    N, cin, cout, insp, k, s, p, d = case[:8]
    groups = case[8] if len(case) > 8 else 1
    torch.manual_seed(0)
    x = torch.randn(N, cin, *insp).to(dtype)
    fan_in = cin // groups * int(torch.tensor(k).prod())
    w = ((torch.rand(cout, cin // groups, *k) * 2 - 1) / fan_in**0.5).to(dtype)
    b = (torch.randn(cout) * 0.1).to(dtype)
    xd, wd, bd = x.double(), w.double(), b.double()
    y_want = oc.forward(xd, wd, bd, s, p, d, groups)
    g = torch.randn_like(y_want).to(dtype)
    gd = g.double()
    gx_want = oc.dgrad(x.shape, wd, gd, s, p, d, groups)
    gw_want = oc.wgrad(xd, w.shape, gd, s, p, d, groups)
    gb_want = oc.grad_bias(gd, len(k))

    xg, wg, bg, gg = x.to(dev), w.to(dev), b.to(dev), g.to(dev)
    kw = dict(stride=s, padding=p, dilation=d, groups=groups)
    y = jc.conv_nd(xg, wg, bg, **kw)
    assert y.dtype == dtype and y.shape == y_want.shape
    assert rel_l2(y, y_want) < TOL[dtype], f"fwd rel-L2 {rel_l2(y, y_want):.3e}"
    y0 = jc.conv_nd(xg, wg, None, **kw)
    assert rel_l2(y0, oc.forward(xd, wd, None, s, p, d, groups)) < TOL[dtype]
    gx = jc.conv_nd_input(x.shape, wg, gg, **kw)
    assert rel_l2(gx, gx_want) < TOL[dtype], f"dgrad rel-L2 {rel_l2(gx, gx_want):.3e}"
    gw = jc.conv_nd_weight(xg, w.shape, gg, **kw)
    assert gw.shape == w.shape
    assert rel_l2(gw, gw_want) < TOL[dtype], f"wgrad rel-L2 {rel_l2(gw, gw_want):.3e}"
    gb = jc.sum_grad_bias(gg, len(k))
    assert rel_l2(gb, gb_want) < TOL[dtype], f"bias grad rel-L2 {rel_l2(gb, gb_want):.3e}"
    # both gradients from one pass over g (falls back to the two kernels where not covered)
    gw2, gb2 = jc.conv_nd_weight(xg, w.shape, gg, with_bias_grad=True, **kw)
    assert torch.equal(gw2, gw)
    assert gb2.dtype == dtype and rel_l2(gb2, gb_want) < TOL[dtype], f"fused bias grad rel-L2 {rel_l2(gb2, gb_want):.3e}"


# rows that start on odd pixels, windows over every edge, several blocks of channels a side with a short last one
ODD_CASES = [
    (2, 40, 72, (21, 131), (0, 0)),
    (1, 70, 97, (9, 65), (2, 2)),
    (1, 3, 5, (2, 3), (1, 1)),
    (3, 17, 16, (16, 63), (0, 1)),
    (1, 5, 33, (3, 5, 67), (1, 1, 1)),
]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", ODD_CASES, ids=lambda c: f"{c[1]}to{c[2]}_{'x'.join(map(str, c[3]))}_p{c[4][-1]}")
def test_odd_rows_and_blocks_of_channels(case, dtype, offset, dev):
    N, ci, co, size, pad = case
    ns, ones = len(size), (1,) * len(size)
    torch.manual_seed(11)

    def placed(t):  # `offset` elements into its storage
        flat = torch.empty(t.numel() + offset, dtype=dtype, device=dev)
        flat[offset:] = t.to(dev).flatten()
        return flat[offset:].view(t.shape)

    x = torch.randn(N, ci, *size).to(dtype)
    w = ((torch.rand(co, ci, *(3,) * ns) * 2 - 1) / (ci * 3**ns) ** 0.5).to(dtype)
    b = torch.randn(co).to(dtype)
    y_want = oc.forward(x.double(), w.double(), b.double(), ones, pad, ones)
    g = torch.randn(y_want.shape).to(dtype)
    xg, wg, gg = placed(x), w.to(dev), placed(g)
    assert rel_l2(jc.conv_nd(xg, wg, b.to(dev), padding=pad), y_want) < TOL[dtype]
    xd = x.double().requires_grad_(True)
    wd = w.double().requires_grad_(True)
    gx_want, gw_want = torch.autograd.grad(oc.forward(xd, wd, None, ones, pad, ones), (xd, wd), g.double())
    assert rel_l2(jc.conv_nd_input(x.shape, wg, gg, padding=pad), gx_want) < TOL[dtype]
    gw, gb = jc.conv_nd_weight(xg, w.shape, gg, padding=pad, with_bias_grad=True)
    assert rel_l2(gw, gw_want) < TOL[dtype]
    assert rel_l2(gb, g.double().sum(dim=(0, *range(2, 2 + ns)))) < TOL[dtype]


# 3 x 3 at stride 2: forward tiles of 64 and of 32 produced channels, one and several of them and of contraction steps; weight
# gradient blocks of 64 x 64, 64 x 32, 32 x 64 and 32 x 32 channels, several a side, short last ones; rows of several tiles (32
# produced pixels forward, 64 in the weight gradient) that end inside one; paddings 0 to 2; images whose last row or column
# no window reaches; many stages a workgroup
STRIDED_CASES = [
    (2, 64, 64, (33, 150), (1, 1)),
    (1, 64, 128, (18, 260), (1, 1)),
    (2, 32, 64, (20, 71), (2, 2)),
    (1, 64, 32, (37, 134), (0, 0)),
    (1, 96, 160, (17, 66), (1, 2)),
    (2, 128, 64, (9, 259), (2, 0)),
    (1, 40, 72, (31, 145), (1, 1)),
    (1, 16, 256, (3, 2), (1, 1)),
    (4, 64, 64, (130, 514), (1, 1)),
]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", STRIDED_CASES, ids=lambda c: f"{c[1]}to{c[2]}_{'x'.join(map(str, c[3]))}_p{c[4][0]}{c[4][1]}")
def test_strided_3x3_layers_exactly(case, dtype, offset, dev):
    """Small whole numbers: every product and fp32 sum is exact in any order, so that each cell of the four results is the
    rounded exact value. ``offset``: elements into its storage at which a tensor starts."""
    N, ci, co, size, pad = case
    torch.manual_seed(ci + co)

    def placed(t):
        flat = torch.empty(t.numel() + offset, dtype=dtype, device=dev)
        flat[offset:] = t.to(dev, dtype).flatten()
        return flat[offset:].view(t.shape)

    x = torch.randint(-2, 3, (N, ci, *size)).double()
    w = torch.randint(-1, 2, (co, ci, 3, 3)).double()
    b = torch.randint(-3, 4, (co,)).double()
    args = ((2, 2), pad, (1, 1))
    y = oc.forward(x, w, b, *args)
    g = torch.randint(-1, 2, y.shape).double()
    xg, wg, bg, gg = placed(x), placed(w), placed(b), placed(g)
    kw = dict(stride=2, padding=pad)
    same = lambda got, want: got.dtype == dtype and torch.equal(got.cpu(), want.to(dtype))  # noqa: E731
    assert same(jc.conv_nd(xg, wg, bg, **kw), y)
    assert same(jc.conv_nd(xg, wg, None, **kw), y - b.view(1, -1, 1, 1))
    assert same(jc.conv_nd_input(x.shape, wg, gg, **kw), oc.dgrad(x.shape, w, g, *args))
    gw, gb = jc.conv_nd_weight(xg, w.shape, gg, with_bias_grad=True, **kw)
    assert same(gw, oc.wgrad(x, w.shape, g, *args)) and same(gb, g.sum(dim=(0, 2, 3)))
    assert same(jc.conv_nd_weight(xg, w.shape, gg, **kw), oc.wgrad(x, w.shape, g, *args))


def test_partial_channel_step_ignores_what_lies_behind_the_last_channel(dev):
    """3 input channels fill 3 of the 16 slots of an MFMA step; the slots behind them are read
    from whatever follows in memory (the next batch entry) and must not reach the result:
    batch entry 1 is all NaN, batch entry 0 must still match the oracle (and stay finite)."""
    torch.manual_seed(3)
    x = torch.randn(2, 3, 40, 70).bfloat16()
    x[1] = float("nan")
    w = ((torch.rand(16, 3, 3, 3) * 2 - 1) / 27**0.5).bfloat16()
    y = jc.conv_nd(x.to(dev), w.to(dev), None)
    assert torch.isfinite(y[0]).all() and torch.isnan(y[1]).all()
    assert rel_l2(y[0:1], oc.forward(x[0:1].double(), w.double(), None, (1, 1), (0, 0), (1, 1))) < TOL[torch.bfloat16]
    g = torch.randn(2, 3, 38, 68).bfloat16()  # gradient of a 16 -> 3 layer: dgrad contracts over 3 channels
    g[1] = float("nan")
    wt = ((torch.rand(3, 16, 3, 3) * 2 - 1) / 12).bfloat16()
    gx = jc.conv_nd_input((2, 16, 40, 70), wt.to(dev), g.to(dev))
    assert torch.isfinite(gx[0]).all()
    assert rel_l2(gx[0:1], oc.dgrad((1, 16, 40, 70), wt.double(), g[0:1].double(), (1, 1), (0, 0), (1, 1))) < TOL[torch.bfloat16]


def test_conv_argument_errors(dev):
    x = torch.zeros(1, 4, 8, 8, device=dev)
    w = torch.zeros(4, 4, 3, 3, device=dev)
    with pytest.raises(NotImplementedError):
        jc.conv_nd(x, w, padding="same")
    with pytest.raises(RuntimeError):  # 4 input channels against a weight that takes 4 per group, two groups
        jc.conv_nd(x, w, groups=2)
    with pytest.raises(ValueError):
        jc.conv_nd(x, w, groups=3)
    with pytest.raises(RuntimeError):
        jc.conv_nd(x, w.bfloat16())
    with pytest.raises(RuntimeError):
        jc.conv_nd(x[:, :3], w)
    with pytest.raises(RuntimeError):
        jc.conv_nd(x.cpu(), w.cpu())
    with pytest.raises(RuntimeError):
        jc.conv_nd(x[:, :, :2, :2], w)


class TableExchange:
    """HaloExchange stand-in on one GPU: the strips the neighbours would send are
    computed beforehand (by packing the neighbours' tensors) and handed over."""

    def __init__(self, fwd, bwd):
        self.fwd, self.bwd = fwd, bwd
        self.sent_fwd = self.sent_bwd = None

    def forward(self, send):
        self.sent_fwd = send
        return self.fwd

    def backward(self, send):
        self.sent_bwd = send
        return self.bwd


def _recv_tables(tensors, geoms, mesh, from_padded):
    """For every rank: offset -> strip received from the neighbour at that offset."""
    ns = len(mesh)
    out = {}
    for c in mesh_coords(mesh):
        tab = {}
        for o in itertools.product((-1, 0, 1), repeat=ns):
            nb = neighbour(c, o, mesh) if any(o) else None
            if nb is None:
                continue
            back = tuple(-v for v in o)
            tab[o] = halo_pack(tensors[nb], geoms[nb], from_padded=from_padded, present=[back])[back]
        out[c] = tab
    return out


DIST_CASES = [
    # mesh, local spatial, N, Cin, Cout, kernel, padding, dtype
    ((2, 2), (32, 32), 2, 3, 16, (3, 3), (1, 1), torch.float32),
    ((2, 2), (32, 32), 2, 16, 3, (3, 3), (1, 1), torch.float32),
    # the reference's CPU-runnable configuration at its real size: 2 x 2 mesh of 256 x 256 tiles, batch 4, fp32
    ((2, 2), (256, 256), 4, 3, 16, (3, 3), (1, 1), torch.float32),
    ((2, 2), (256, 256), 4, 16, 3, (3, 3), (1, 1), torch.float32),
    ((3, 3), (8, 12), 1, 4, 5, (5, 3), (2, 1), torch.float32),
    ((2, 1), (16, 20), 2, 4, 4, (3, 3), (1, 1), torch.float32),
    ((2, 2), (32, 64), 1, 64, 64, (3, 3), (1, 1), torch.bfloat16),
    ((2, 2, 2), (8, 8, 16), 1, 32, 32, (3, 3, 3), (1, 1, 1), torch.bfloat16),
    ((2, 2, 2), (6, 6, 6), 1, 3, 4, (3, 3, 3), (1, 1, 1), torch.float32),
    # strided / dilated halos (needed_input_span with s > 1, d > 1): one-sided and 2-wide halos
    ((2, 2), (8, 12), 2, 4, 6, (3, 3), (1, 1), torch.float32, (2, 2), (1, 1)),
    ((3, 2), (8, 10), 1, 3, 5, (3, 3), (2, 2), torch.float32, (1, 1), (2, 2)),
    ((2, 2), (16, 32), 1, 32, 32, (3, 3), (1, 2), torch.bfloat16, (2, 1), (1, 2)),
    ((2, 1, 2), (4, 6, 8), 1, 2, 3, (3, 3, 3), (1, 1, 2), torch.float32, (2, 1, 1), (1, 1, 2)),
    ((2, 2), (32, 160), 2, 64, 128, (3, 3), (1, 1), torch.bfloat16, (2, 2), (1, 1)),
    # need spans that drift against the tiles (halo.py:49-63 with out_local * stride != n): the widths change from rank to rank
    ((2, 2), (16, 20), 2, 4, 6, (3, 3), (0, 0), torch.float32),                    # no padding: (0, 1) and (1, 0)
    ((4, 2), (6, 12), 1, 3, 5, (5, 3), (0, 1), torch.float32),                     # four ranks: (r, 3 - r)
    ((2, 2), (8, 8), 1, 3, 4, (6, 6), (0, 0), torch.float32, (2, 2), (1, 1)),      # strided and drifting
    ((2, 2), (16, 32), 1, 32, 32, (3, 3), (0, 0), torch.bfloat16),                 # MFMA path, fused fold, framed forward
    ((2, 1, 2), (4, 6, 8), 1, 2, 3, (3, 3, 5), (0, 1, 1), torch.float32),
    # grouped layers (eleventh entry: groups) through the distributed functions
    ((2, 2), (8, 12), 2, 6, 9, (3, 3), (1, 1), torch.float32, (1, 1), (1, 1), 3),
    ((2, 2), (16, 32), 1, 32, 32, (3, 3), (1, 1), torch.bfloat16, (1, 1), (1, 1), 32),
    ((2, 2), (16, 32), 2, 32, 48, (3, 3), (1, 1), torch.bfloat16, (1, 1), (1, 1), 2),   # 16 -> 24 channels a group: each group on the matrix cores
]


@pytest.mark.parametrize("case", DIST_CASES, ids=lambda c: f"mesh{'x'.join(map(str, c[0]))}_{c[3]}to{c[4]}_{str(c[7]).split('.')[-1]}" + (f"_s{''.join(map(str, c[8]))}_d{''.join(map(str, c[9]))}" if len(c) > 8 else "") + (f"_g{c[10]}" if len(c) > 10 else ""))
def test_distributed_conv_matches_global_conv(case, dev):
    """The reference's parity method: every rank's y / dx and the summed dw / db equal
    the serial conv on the gathered tensor (test_conv2d_multi_spatial.py:73-233)."""
    # bf16 cases also take the framed forward (only the frame of the padded tile is built)
    _run_mesh_case(case, dev, framed=case[7] == torch.bfloat16, autocast=None)


@pytest.mark.parametrize("framed", [False, True], ids=["assembled", "framed"])
@pytest.mark.parametrize("case", [
    ((2, 2), (32, 64), 1, 64, 64, (3, 3), (1, 1), torch.float32),
    ((2, 2, 2), (8, 8, 16), 1, 32, 32, (3, 3, 3), (1, 1, 1), torch.float32),
], ids=["2d", "3d"])
def test_distributed_conv_under_autocast(case, framed, dev):
    """fp32 leaves under bf16 autocast: the forward casts x / w / b down
    (_core/autocast.py:44-66, functional.py:53), the backward runs outside autocast in the
    weight's dtype on the saved bf16 padded tile (functional.py:126-129). Gradients come
    back in the leaves' dtype. Bar: bf16 (the forward's operands are rounded to it)."""
    _run_mesh_case(case, dev, framed=framed, autocast=torch.bfloat16)


def _run_mesh_case(case, dev, framed, autocast):
    mesh, n, N, cin, cout, k, p, dtype = case[:8]
    ns = len(mesh)
    s, d = (case[8], case[9]) if len(case) > 8 else ((1,) * ns, (1,) * ns)
    conv_groups = case[10] if len(case) > 10 else 1
    torch.manual_seed(0)
    gshape = tuple(a * b for a, b in zip(n, mesh))
    X = torch.randn(N, cin, *gshape).to(dtype)
    fan_in = cin // conv_groups * int(torch.tensor(k).prod())
    W = ((torch.rand(cout, cin // conv_groups, *k) * 2 - 1) / fan_in**0.5).to(dtype)
    B = (torch.randn(cout) * 0.1).to(dtype)
    Xd = X.double().requires_grad_()
    Wd = W.double().requires_grad_()
    Bd = B.double().requires_grad_()
    Y = oc.forward(Xd, Wd, Bd, s, p, d, conv_groups)
    G = torch.randn_like(Y).to(dtype)
    Y.backward(G.double())

    tiles = {c: t.to(dev) for c, t in oh.split_global(X, mesh).items()}
    gtiles = {c: t.to(dev) for c, t in oh.split_global(G, mesh).items()}
    geoms = {c: conv_geometry(n, mesh, c, k, s, p, d) for c in tiles}
    if autocast is not None:
        # the strips travel in the autocast dtype; the upstream gradient arrives rounded to it
        fwd_tabs = _recv_tables({c: t.to(autocast) for c, t in tiles.items()}, geoms, mesh, from_padded=False)
        gtiles = {c: t.to(autocast).to(dtype) for c, t in gtiles.items()}
    else:
        fwd_tabs = _recv_tables(tiles, geoms, mesh, from_padded=False)
    Wg, Bg = W.to(dev), B.to(dev)

    # pass 1: forward of every rank, and the padded dgrad every rank will send from
    cfgs, outs, leaves, gx_need = {}, {}, {}, {}
    for c in mesh_coords(mesh):
        cfgs[c] = jc.HipConvNdConfig.for_rank(ns, Bg, TableExchange(fwd_tabs[c], None), groups=conv_groups, framed=framed)
        groups = tuple(jc.TileGroup(mesh[a], c[a]) for a in range(ns))
        xl = tiles[c].clone().requires_grad_()
        wl, bl = Wg.clone().requires_grad_(), Bg.clone().requires_grad_()
        with torch.autocast("cuda", dtype=autocast or torch.bfloat16, enabled=autocast is not None):
            y, x_aug = jc._ConvNd.apply(xl, wl, bl, s, p, d, groups, None, cfgs[c])
        outs[c], leaves[c] = y, (xl, wl, bl)
        assert not x_aug.requires_grad
        assert y.dtype == (autocast or dtype) and x_aug.dtype == (autocast or dtype)
        lp = oh.local_padding(p, mesh)
        gx_need[c] = jc.conv_nd_input(x_aug.shape, Wg, gtiles[c], stride=s, padding=lp, dilation=d, groups=conv_groups)
    bwd_tabs = _recv_tables(gx_need, geoms, mesh, from_padded=True)

    # pass 2: backward of every rank
    gw_sum = torch.zeros_like(W, dtype=torch.float64)
    gb_sum = torch.zeros_like(B, dtype=torch.float64)
    tol = TOL[autocast or dtype]
    for c in mesh_coords(mesh):
        cfgs[c].halo_exchange.bwd = bwd_tabs[c]
        outs[c].backward(gtiles[c].to(outs[c].dtype))
        xl, wl, bl = leaves[c]
        assert xl.grad.dtype == dtype and wl.grad.dtype == dtype and bl.grad.dtype == dtype
        sl = (slice(None), slice(None)) + tuple(slice(c[a] * n[a], (c[a] + 1) * n[a]) for a in range(ns))
        no = tuple(Y.shape[2 + a] // mesh[a] for a in range(ns))  # output rows per rank
        so = (slice(None), slice(None)) + tuple(slice(c[a] * no[a], (c[a] + 1) * no[a]) for a in range(ns))
        assert rel_l2(outs[c], Y.detach()[so]) < tol, f"y of rank {c}: {rel_l2(outs[c], Y.detach()[so]):.3e}"
        assert rel_l2(xl.grad, Xd.grad[sl]) < tol, f"dx of rank {c}: {rel_l2(xl.grad, Xd.grad[sl]):.3e}"
        gw_sum += wl.grad.double().cpu()
        gb_sum += bl.grad.double().cpu()
    # replicated weights: gradients are summed over the spatial ranks (parallel/_sync.py:33-46)
    assert rel_l2(gw_sum, Wd.grad) < tol, f"dw: {rel_l2(gw_sum, Wd.grad):.3e}"
    assert rel_l2(gb_sum, Bd.grad) < tol, f"db: {rel_l2(gb_sum, Bd.grad):.3e}"


GENERAL_SPAN_CASES = [
    # mesh, local spatial, N, Cin, Cout, kernel, padding, dtype, stride, dilation: need spans that leave out owned
    # rows or reach past the adjacent rank (halo.py:49-63, 134-154): one split axis at a time
    ((2, 2), (9, 9), 2, 3, 4, (3, 3), (0, 0), torch.float32, (2, 2), (1, 1)),
    ((3, 2), (2, 8), 1, 4, 5, (7, 3), (3, 1), torch.float32, (1, 1), (1, 1)),
    ((4, 1), (3, 10), 2, 2, 3, (9, 3), (4, 1), torch.float32, (1, 1), (1, 1)),
    ((3, 2), (2, 16), 1, 16, 16, (3, 3), (3, 1), torch.bfloat16, (1, 1), (3, 1)),
    ((2, 3, 1), (4, 2, 5), 1, 2, 3, (5, 7, 3), (2, 3, 1), torch.float32, (1, 1, 1), (1, 1, 1)),
]


@pytest.mark.parametrize("case", GENERAL_SPAN_CASES, ids=lambda c: "mesh" + "x".join(map(str, c[0])) + "_k" + "x".join(map(str, c[5])) + "_" + str(c[7]).split(".")[-1])
def test_distributed_conv_with_general_spans(case, dev):
    """``conv_halo_nway`` and ``conv_halo_nway_backward`` on every rank of the mesh (in lockstep, one thread a rank)
    where the need spans do not fit the strip exchange: y, dx of every rank and the summed dw, db against the
    serial conv on the gathered tensor (the parity method of test_conv2d_multi_spatial.py:73-233). The two
    functions are called directly: the autograd engine runs every rank's backward node on its one device thread,
    where ranks that wait for each other cannot meet."""
    from helpers import LockstepMesh
    from jigsaw_amd.halo import spans_fit_the_strips

    mesh, n, N, cin, cout, k, p, dtype, s, d = case
    ns = len(mesh)
    assert not spans_fit_the_strips(n, k, s, p, d, mesh)
    torch.manual_seed(1)
    gshape = tuple(a * b for a, b in zip(n, mesh))
    X = torch.randn(N, cin, *gshape).to(dtype)
    W = ((torch.rand(cout, cin, *k) * 2 - 1) / (cin * int(torch.tensor(k).prod())) ** 0.5).to(dtype)
    B = (torch.randn(cout) * 0.1).to(dtype)
    Xd, Wd, Bd = X.double().requires_grad_(), W.double().requires_grad_(), B.double().requires_grad_()
    Y = oc.forward(Xd, Wd, Bd, s, p, d)
    G = torch.randn_like(Y).to(dtype)
    Y.backward(G.double())
    tiles = oh.split_global(X, mesh)
    gtiles = oh.split_global(G, mesh)
    lock = LockstepMesh(mesh)

    def rank(c, exchange):
        cfg = jc.HipConvNdConfig.for_rank(ns, B.to(dev), exchange)
        groups = tuple(jc.TileGroup(mesh[a], c[a]) for a in range(ns))
        xl, wl, bl = tiles[c].to(dev), W.to(dev), B.to(dev)
        y, x_aug = jc.conv_halo_nway(xl, wl, bl, s, p, d, groups, None, cfg)
        gx, gw, gb = jc.conv_halo_nway_backward(gtiles[c].to(dev), x_aug, wl, s, p, d, n, groups, None, cfg, need=(True, True, True))
        return y.cpu(), gx.cpu(), gw.double().cpu(), gb.double().cpu()

    got = lock.run(rank)
    tol = TOL[dtype]
    gw_sum, gb_sum = torch.zeros_like(Wd), torch.zeros_like(Bd)
    for c in mesh_coords(mesh):
        y, gx, gw, gb = got[c]
        sl = (slice(None), slice(None)) + tuple(slice(c[a] * n[a], (c[a] + 1) * n[a]) for a in range(ns))
        no = tuple(Y.shape[2 + a] // mesh[a] for a in range(ns))
        so = (slice(None), slice(None)) + tuple(slice(c[a] * no[a], (c[a] + 1) * no[a]) for a in range(ns))
        assert rel_l2(y, Y.detach()[so]) < tol, f"y of rank {c}: {rel_l2(y, Y.detach()[so]):.3e}"
        assert rel_l2(gx, Xd.grad[sl]) < tol, f"dx of rank {c}: {rel_l2(gx, Xd.grad[sl]):.3e}"
        gw_sum += gw
        gb_sum += gb
    assert rel_l2(gw_sum, Wd.grad) < tol and rel_l2(gb_sum, Bd.grad) < tol
    # the exchange ran once per split axis and direction on every rank, forward first to last, backward last to first
    per_rank = [call for call in lock.calls if call[0] == (0,) * ns]
    split = [a for a in range(ns) if mesh[a] > 1]
    assert [(a, b) for _, a, b, _ in per_rank] == [(a, False) for a in split] + [(a, True) for a in reversed(split)]


def test_frame_without_its_tile_is_refused(dev):
    """A caller that keeps only ``x_aug`` (as the reference's own autograd function does)
    cannot take the weight gradient from a frame: the backward says so instead of
    reading the undefined interior."""
    torch.manual_seed(0)
    mesh, n = (2, 2), (32, 64)
    X = torch.randn(1, 64, 64, 128).bfloat16()
    tiles = {c: t.to(dev) for c, t in oh.split_global(X, mesh).items()}
    geoms = {c: conv_geometry(n, mesh, c, (3, 3), (1, 1), (1, 1), (1, 1)) for c in tiles}
    tabs = _recv_tables(tiles, geoms, mesh, from_padded=False)
    c = (0, 1)
    cfg = jc.HipConvNdConfig.for_rank(2, None, TableExchange(tabs[c], {}), framed=True)
    groups = tuple(jc.TileGroup(mesh[a], c[a]) for a in range(2))
    w = (torch.randn(64, 64, 3, 3) / 24).bfloat16().to(dev)
    y, x_aug = jc.conv_halo_nway(tiles[c], w, None, (1, 1), (1, 1), (1, 1), groups, None, cfg)
    with pytest.raises(RuntimeError, match="x_tile"):
        jc.conv_halo_nway_backward(torch.ones_like(y), x_aug, w, (1, 1), (1, 1), (1, 1), n, groups, None, cfg)


def test_first_layer_skips_dgrad(dev):
    """needs_input_grad gating (functional.py:131-148): no input grad -> no dgrad, no fold."""
    cfg = jc.HipConvNdConfig.for_rank(2, None, TableExchange({}, {}))
    x = torch.randn(1, 3, 8, 8, device=dev)
    w = torch.randn(4, 3, 3, 3, device=dev, requires_grad=True)
    groups = (jc.TileGroup(1, 0), jc.TileGroup(1, 0))
    y, _ = jc._ConvNd.apply(x, w, None, (1, 1), (1, 1), (1, 1), groups, None, cfg)
    y.sum().backward()
    assert w.grad is not None and cfg.halo_exchange.sent_bwd is None


def test_string_padding_is_rejected(dev):
    cfg = jc.HipConvNdConfig.for_rank(2, None, TableExchange({}, {}))
    x = torch.randn(1, 3, 8, 8, device=dev)
    w = torch.randn(4, 3, 3, 3, device=dev)
    with pytest.raises(NotImplementedError):
        jc.conv_halo_nway(x, w, None, (1, 1), "same", (1, 1), (None, None), None, cfg)


FUSED_CASES = [
    # size, lo, hi, conv padding on the padded tile, N, channels, strips that exist
    ((32, 64), (1, 1), (1, 1), (0, 0), 2, 64, "all"),
    ((40, 72), (1, 1), (1, 1), (0, 0), 1, 64, "some"),
    ((24, 40), (0, 2), (2, 0), (0, 0), 1, 32, "all"),
    ((16, 96), (1, 0), (1, 0), (0, 1), 1, 64, "all"),     # W axis not split: the conv pads it itself
    ((48, 128), (1, 1), (1, 1), (0, 0), 2, 64, "all"),    # rows of g are whole cache lines: the tile grid is shifted
    ((20, 192), (1, 1), (1, 1), (0, 0), 1, 32, "some"),
    ((8, 8, 16), (1, 1, 1), (1, 1, 1), (0, 0, 0), 1, 32, "all"),
    ((6, 10, 24), (1, 0, 1), (1, 0, 1), (0, 1, 0), 1, 32, "some"),
]


@pytest.mark.parametrize("case", FUSED_CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}_lo{''.join(map(str, c[1]))}_hi{''.join(map(str, c[2]))}")
def test_fused_dgrad_fold_has_the_bits_of_the_three_steps(case, dev):
    """conv_nd_input_fold + halo_fold_border_ == conv_nd_input + halo_pack + halo_fold, bit for bit."""
    from jigsaw_amd.halo import HaloGeometry, halo_fold, halo_fold_border_

    size, lo, hi, pad, N, ch, which = case
    ns = len(size)
    geom = HaloGeometry(size, lo, hi)
    torch.manual_seed(3)
    k = (3,) * ns
    out_sp = tuple(geom.padded[a] + 2 * pad[a] - 2 for a in range(ns))
    w = ((torch.rand(ch, ch, *k, device=dev) * 2 - 1) / (ch * 3**ns) ** 0.5).bfloat16()
    g = torch.randn(N, ch, *out_sp, device=dev).bfloat16()
    g[0, 0].zero_()          # exact zeros: the fold clears the sign of -0.0
    g[0, 1] = -g[0, 1].abs() * 1e-30
    offs = [o for o in geom.offsets() if all(geom.strip_extent(o, "fold")[a] > 0 for a in range(ns))]
    if which == "some":
        offs = offs[::2]
    recv = {o: torch.randn(N, ch, *geom.strip_extent(o, "fold"), device=dev).bfloat16() for o in offs}

    gx_aug = jc.conv_nd_input((N, ch, *geom.padded), w, g, padding=pad)
    send_u = halo_pack(gx_aug, geom, from_padded=True)
    gx_u = halo_fold(gx_aug, recv, geom)

    fused = jc.conv_nd_input_fold(geom, w, g, padding=pad)
    assert fused is not None, "the MFMA path should cover this case"
    gx_f, send_f = fused
    halo_fold_border_(gx_f, recv, geom)
    assert torch.equal(gx_f.view(torch.int16), gx_u.view(torch.int16))
    assert set(send_f) == set(send_u)
    for o in send_u:
        assert torch.equal(send_f[o].view(torch.int16), send_u[o].view(torch.int16)), f"strip {o}"


def test_fused_dgrad_fold_declines_what_the_mfma_kernel_does_not_cover(dev):
    """The function's own limit: bf16 (the layers reach the kernels of the other types through ``_input_fold``)."""
    from jigsaw_amd.halo import HaloGeometry

    geom = HaloGeometry((8, 8), (1, 1), (1, 1))
    w = torch.randn(4, 3, 3, 3, device=dev)
    g = torch.randn(1, 4, 8, 8, device=dev)
    assert jc.conv_nd_input_fold(geom, w, g, padding=(0, 0)) is None


FRAMED_CASES = [
    # size, lo, hi, conv padding on the padded tile, N, channels
    ((96, 256), (1, 1), (1, 1), (0, 0), 2, 64),
    ((70, 200), (1, 1), (1, 1), (0, 0), 1, 64),
    ((40, 330), (1, 0), (1, 0), (0, 1), 1, 32),       # W axis not split: the conv pads it itself
    ((66, 130), (0, 2), (2, 0), (0, 0), 1, 64),
    ((4, 40, 140), (1, 1, 1), (1, 1, 1), (0, 0, 0), 1, 32),
]


@pytest.mark.parametrize("case", FRAMED_CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}_lo{''.join(map(str, c[1]))}_hi{''.join(map(str, c[2]))}")
def test_framed_conv_has_the_bits_of_the_assembled_tile(case, dev):
    """Forward and weight gradient that read the own tile directly, plus a frame of the padded
    tile near the edges, equal the kernels on the fully assembled tile bit for bit; what lies
    outside the frame is never read (it holds NaN here)."""
    from jigsaw_amd.halo import HaloGeometry, halo_assemble

    size, lo, hi, pad, N, ch = case
    ns = len(size)
    geom = HaloGeometry(size, lo, hi)
    torch.manual_seed(5)
    k = (3,) * ns
    x = torch.randn(N, ch, *size, device=dev).bfloat16()
    strips = {o: torch.randn(N, ch, *geom.strip_extent(o, "assemble"), device=dev).bfloat16() for o in geom.offsets()}
    w = ((torch.rand(ch, ch, *k, device=dev) * 2 - 1) / (ch * 3**ns) ** 0.5).bfloat16()
    b = (torch.randn(ch, device=dev) * 0.1).bfloat16()
    x_aug = halo_assemble(x, strips, geom)
    y_ref = jc.conv_nd(x_aug, w, b, padding=pad)
    g = torch.randn_like(y_ref)
    gw_ref, gb_ref = jc.conv_nd_weight(x_aug, w.shape, g, padding=pad, with_bias_grad=True)

    bands = jc.frame_bands(x, geom, w.shape, padding=pad)
    if bands is None:
        # the framed weight-gradient kernel needs an even padding along W; callers assemble the whole tile then
        assert pad[-1] % 2 == 1
        return
    frame = torch.full_like(x_aug, float("nan"))
    halo_assemble(x, strips, geom, out=frame, bands=bands)
    # the frame holds exactly the band cells of the assembled tile
    inside = torch.ones(geom.padded, dtype=torch.bool, device=dev)
    for a in range(ns):
        idx = torch.arange(geom.padded[a], device=dev)
        in_band = (idx < bands[0][a]) | (idx >= geom.padded[a] - bands[1][a])
        shape = [1] * ns
        shape[a] = -1
        inside &= ~in_band.view(shape)
    assert torch.equal(frame[..., ~inside].view(torch.int16), x_aug[..., ~inside].view(torch.int16))
    assert torch.isnan(frame[..., inside]).all()

    y = jc.conv_nd_framed(frame, x, geom, w, b, padding=pad)
    assert y is not None and torch.equal(y.view(torch.int16), y_ref.view(torch.int16))
    gw, gb = jc.conv_nd_weight_framed(frame, x, geom, w.shape, g, padding=pad, with_bias_grad=True)
    assert torch.equal(gw.view(torch.int16), gw_ref.view(torch.int16))
    assert torch.equal(gb.view(torch.int16), gb_ref.view(torch.int16))


def _crop_check(y, x_aug, w, b, windows, what):
    """Output windows of the full-size result against the oracle on the matching input
    crops (a k=3, pad-0 conv: output rows h0..h0+H come from input rows h0..h0+H+2)."""
    ns = y.dim() - 2
    for n, *org in windows:
        ext = (32,) * (ns - 1) + (64,)
        ext = tuple(min(e, y.shape[2 + a] - org[a]) for a, e in enumerate(ext))
        osl = (n, slice(None)) + tuple(slice(o, o + e) for o, e in zip(org, ext))
        isl = (slice(n, n + 1), slice(None)) + tuple(slice(o, o + e + 2) for o, e in zip(org, ext))
        want = oc.forward(x_aug[isl].float().cpu(), w.float().cpu(), None if b is None else b.float().cpu(),
                          (1,) * ns, (0,) * ns, (1,) * ns)[0]
        assert rel_l2(y[osl], want) < 2e-2, f"{what}: window {n, *org}"


def test_config2_full_size_properties(dev):
    """Configuration 2 at full size (8 x 64 x 1024^2 bf16, all 8 neighbours live): output
    windows from the corners, edges and interior of several batch entries against the oracle
    on the matching crops; the fused backward against the separate steps bit for bit; the
    weight gradient as the sum of per-entry weight gradients, one of them against the oracle;
    the bias gradient against the plain sum."""
    from jigsaw_amd.halo import HaloGeometry, halo_assemble, halo_fold, halo_fold_border_

    torch.manual_seed(0)
    N, C, T = 8, 64, 1024
    geom = HaloGeometry((T, T), (1, 1), (1, 1))
    x = torch.randn(N, C, T, T, device=dev).bfloat16()
    w = ((torch.rand(C, C, 3, 3, device=dev) * 2 - 1) / 24).bfloat16()
    b = ((torch.rand(C, device=dev) * 2 - 1) / 24).bfloat16()
    g = torch.randn(N, C, T, T, device=dev).bfloat16()
    sf = {o: torch.randn(N, C, *geom.strip_extent(o, "assemble"), device=dev).bfloat16() for o in geom.offsets()}
    sb = {o: torch.randn(N, C, *geom.strip_extent(o, "fold"), device=dev).bfloat16() for o in geom.offsets()}

    x_aug = halo_assemble(x, sf, geom)
    y = jc.conv_nd(x_aug, w, b)
    wins = [(0, 0, 0), (0, 0, T - 64), (3, T - 32, 0), (7, T - 32, T - 64), (5, 496, 480), (2, 16, 960), (6, 1000, 64)]
    _crop_check(y, x_aug, w, b, wins, "forward")

    # backward: fused == separate, and the padded gradient against the oracle (dgrad of a
    # k=3 conv is the conv of the zero-padded g with the flipped, transposed weight)
    gx_aug = jc.conv_nd_input(x_aug.shape, w, g)
    wt = w.flip(-1, -2).transpose(0, 1).contiguous()
    g_pad = torch.nn.functional.pad(g, (2, 2, 2, 2))
    wins_aug = [(0, 0, 0), (1, 0, T + 2 - 64), (4, T + 2 - 32, 0), (7, T + 2 - 32, T + 2 - 64), (3, 500, 500)]
    _crop_check(gx_aug, g_pad, wt, None, wins_aug, "dgrad")
    gx_u = halo_fold(gx_aug, sb, geom)
    send_u = halo_pack(gx_aug, geom, from_padded=True)
    del gx_aug, g_pad
    gx_f, send_f = jc.conv_nd_input_fold(geom, w, g)
    halo_fold_border_(gx_f, sb, geom)
    assert torch.equal(gx_f.view(torch.int16), gx_u.view(torch.int16))
    for o in send_u:
        assert torch.equal(send_f[o].view(torch.int16), send_u[o].view(torch.int16)), f"strip {o}"
    del gx_u, gx_f

    gw, gb = jc.conv_nd_weight(x_aug, w.shape, g, with_bias_grad=True)
    parts = [jc.conv_nd_weight(x_aug[n:n + 1], w.shape, g[n:n + 1]).float() for n in range(N)]
    assert rel_l2(gw, sum(parts)) < 1e-2
    want1 = oc.wgrad(x_aug[5:6].float().cpu(), w.shape, g[5:6].float().cpu(), (1, 1), (0, 0), (1, 1))
    assert rel_l2(parts[5], want1) < 2e-2
    assert rel_l2(gb, g.float().sum((0, 2, 3))) < 1e-2


def test_config3_full_size_properties(dev):
    """Configuration 3 at full size (2 x 32 x 128^3 bf16, 26 neighbours): forward and padded
    gradient windows against the oracle on crops, the fused backward against the separate
    steps bit for bit, the weight gradient of one entry against the oracle."""
    from jigsaw_amd.halo import HaloGeometry, halo_assemble, halo_fold, halo_fold_border_

    torch.manual_seed(1)
    N, C, T = 2, 32, 128
    geom = HaloGeometry((T, T, T), (1, 1, 1), (1, 1, 1))
    x = torch.randn(N, C, T, T, T, device=dev).bfloat16()
    w = ((torch.rand(C, C, 3, 3, 3, device=dev) * 2 - 1) / 864 ** 0.5).bfloat16()
    b = ((torch.rand(C, device=dev) * 2 - 1) / 864 ** 0.5).bfloat16()
    g = torch.randn(N, C, T, T, T, device=dev).bfloat16()
    sf = {o: torch.randn(N, C, *geom.strip_extent(o, "assemble"), device=dev).bfloat16() for o in geom.offsets()}
    sb = {o: torch.randn(N, C, *geom.strip_extent(o, "fold"), device=dev).bfloat16() for o in geom.offsets()}

    x_aug = halo_assemble(x, sf, geom)
    y = jc.conv_nd(x_aug, w, b)
    wins = [(0, 0, 0, 0), (1, T - 32, T - 32, T - 64), (0, 0, T - 32, 64), (1, 96, 0, 0), (0, 50, 50, 30)]
    _crop_check(y, x_aug, w, b, wins, "forward")

    gx_aug = jc.conv_nd_input(x_aug.shape, w, g)
    wt = w.flip(-1, -2, -3).transpose(0, 1).contiguous()
    g_pad = torch.nn.functional.pad(g, (2,) * 6)
    wins_aug = [(0, 0, 0, 0), (1, T + 2 - 32, T + 2 - 32, T + 2 - 64), (0, 40, 98, 66), (1, 0, 98, 0)]
    _crop_check(gx_aug, g_pad, wt, None, wins_aug, "dgrad")
    gx_u = halo_fold(gx_aug, sb, geom)
    send_u = halo_pack(gx_aug, geom, from_padded=True)
    fused = jc.conv_nd_input_fold(geom, w, g)
    assert fused is not None
    gx_f, send_f = fused
    halo_fold_border_(gx_f, sb, geom)
    assert torch.equal(gx_f.view(torch.int16), gx_u.view(torch.int16))
    for o in send_u:
        assert torch.equal(send_f[o].view(torch.int16), send_u[o].view(torch.int16)), f"strip {o}"

    gw, gb = jc.conv_nd_weight(x_aug, w.shape, g, with_bias_grad=True)
    parts = [jc.conv_nd_weight(x_aug[n:n + 1], w.shape, g[n:n + 1]).float() for n in range(N)]
    assert rel_l2(gw, sum(parts)) < 1e-2
    want0 = oc.wgrad(x_aug[0:1].float().cpu(), w.shape, g[0:1].float().cpu(), (1, 1, 1), (0, 0, 0), (1, 1, 1))
    assert rel_l2(parts[0], want0) < 2e-2
    assert rel_l2(gb, g.float().sum((0, 2, 3, 4))) < 1e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [
    # size, lo, hi, conv padding on the padded tile, stride, N, c_in, c_out, strips present
    ((17, 23), (1, 1), (1, 1), (0, 0), 1, 2, 40, 24, "all"),       # ragged channels, odd rows
    ((33, 65), (1, 1), (1, 1), (0, 0), 1, 1, 3, 16, "all"),
    ((16, 62), (0, 1), (1, 0), (1, 0), 1, 1, 72, 8, "some"),       # the padded row is a tile; one axis padded by the conv
    ((16, 130), (2, 1), (0, 1), (0, 0), 1, 1, 65, 16, "all"),
    ((5, 9, 33), (1, 1, 1), (1, 1, 1), (0, 0, 0), 1, 1, 5, 7, "some"),
    ((16, 32), (1, 1), (0, 0), (0, 0), 2, 2, 32, 24, "all"),       # stride 2: whole and ragged channel tiles
    ((34, 66), (1, 1), (0, 0), (0, 0), 2, 1, 40, 16, "all"),
    ((34, 66), (0, 0), (0, 0), (1, 1), 2, 1, 7, 16, "all"),
    ((32, 130), (1, 0), (1, 0), (0, 1), 2, 1, 33, 16, "some"),
], ids=str)
def test_fused_dgrad_fold_any_channels_types_and_strides(case, dtype, dev):
    """jg_conv_dgrad_fold == jg_conv_dgrad and halo_pack, bit for bit, the sign of zeros cleared."""
    from jigsaw_amd.halo import HaloGeometry, halo_fold, new_strips

    size, lo, hi, pad, stride, N, ci, co, which = case
    ns = len(size)
    geom = HaloGeometry(size, lo, hi)
    torch.manual_seed(4)
    out_sp = tuple((geom.padded[a] + 2 * pad[a] - 3) // stride + 1 for a in range(ns))
    w = ((torch.rand(co, ci, *(3,) * ns, device=dev) * 2 - 1) / (co * 3**ns) ** 0.5).to(dtype)
    g = torch.randn(N, co, *out_sp, device=dev).to(dtype)
    g[0].mul_(1e-7 if dtype == torch.float16 else 1e-38)  # results that round to zero, of both signs
    offs = [o for o in geom.offsets() if all(geom.strip_extent(o, "pack_bwd")[a] > 0 for a in range(ns))]
    if which == "some":
        offs = offs[::2]
    want = jc.conv_nd_input((N, ci, *geom.padded), w, g, stride=stride, padding=pad)
    want_send = halo_pack(want, geom, from_padded=True, present=offs) if offs else {}
    launch = jc._launch_for(1, dtype, (N, ci, *geom.padded), w.shape, (stride,) * ns, pad, (1,) * ns, 1)
    send, tab = new_strips(geom, "pack_bwd", (N, ci), tuple(offs), dtype, dev)
    for t in send.values():
        t.fill_(7)
    gx = torch.full((N, ci, *size), 7.0, dtype=dtype, device=dev)
    ws = jc._scratch(launch, dev)
    rc = _lib.load().jg_conv_dgrad_fold(_lib.ptr(gx), tab, _lib.ptr(w), _lib.ptr(g), launch.desc, geom.c_geom(N * ci), _lib.dtype_code(dtype),
                                        _lib.ptr(ws), launch.nbytes, _lib.stream_ptr(dev))
    assert rc == 0, _lib.load().jg_last_error()
    bits = {torch.float32: torch.int32}.get(dtype, torch.int16)
    assert torch.equal(gx.view(bits), halo_fold(want, {}, geom).view(bits))
    for o in offs:
        assert torch.equal(send[o].view(bits), (want_send[o] + 0).view(bits)), f"strip {o}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [
    # as above, with images enough for several tiles a workgroup: produced tensors one or two rows and columns larger than a whole number
    # of tiles, which are made beside the tiles at the edge, rows with 32 produced channels only
    ((16, 64), (1, 1), (1, 1), (0, 0), 1, 200, 32, 16, "all"),
    ((16, 64), (1, 1), (1, 1), (0, 0), 1, 140, 64, 40, "some"),
    ((16, 128), (1, 2), (1, 0), (0, 0), 1, 90, 50, 8, "all"),
    ((32, 64), (0, 1), (1, 1), (1, 0), 1, 150, 20, 16, "all"),
    ((13, 64), (1, 1), (1, 1), (0, 0), 1, 280, 7, 24, "all"),     # columns only, the tile row not full
    ((14, 64), (1, 1), (1, 1), (0, 0), 1, 600, 64, 8, "some"),    # the same with 64 produced channels, all and 50 of them there
    ((14, 64), (1, 1), (1, 1), (0, 0), 1, 600, 50, 8, "all"),
    ((16, 30), (1, 1), (1, 1), (0, 0), 1, 300, 32, 16, "all"),    # rows only
    ((3, 16, 64), (1, 1, 1), (1, 1, 1), (0, 0, 0), 1, 40, 32, 8, "all"),
    ((32, 128), (1, 1), (0, 0), (0, 0), 2, 60, 40, 16, "all"),
    ((32, 256), (0, 1), (1, 0), (1, 0), 2, 40, 33, 24, "some"),
], ids=str)
def test_rows_and_columns_beside_the_tile_grid(case, dtype, dev):
    test_fused_dgrad_fold_any_channels_types_and_strides(case, dtype, dev)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [
    # batch, c_in, c_out, size, stride: tiles of 64 produced channels (launches that fill the chip) and, with fewer images, of 32; whole
    # 16-byte rows and others, channels that end inside a tile, more contraction steps than LDS holds weights for
    (600, 16, 64, (16, 64), 1), (40, 16, 64, (16, 64), 1), (600, 7, 50, (9, 33), 1), (40, 7, 50, (9, 33), 1), (300, 80, 64, (5, 40), 1), (3, 80, 128, (5, 40), 1),
    (600, 16, 64, (16, 64), 2), (40, 16, 64, (16, 64), 2), (600, 9, 60, (11, 35), 2), (30, 70, 60, (11, 35), 2), (3, 88, 24, (10, 30), 2), (3, 5, 9, (10, 30), 1),
], ids=str)
def test_tiles_of_64_and_of_32_channels_exactly(case, dtype, dev):
    """Whole numbers, as in test_strided_3x3_layers_exactly."""
    N, ci, co, size, stride = case
    gen = torch.Generator().manual_seed(9)
    x = torch.randint(-2, 3, (N, ci, *size), generator=gen).float()
    w = torch.randint(-1, 2, (co, ci, 3, 3), generator=gen).float()
    b = torch.randint(-3, 4, (co,), generator=gen).float()
    want = torch.nn.functional.conv2d(x, w, b, stride=stride, padding=1)  # sums below 2^24: exact in fp32
    y = jc.conv_nd(x.to(dtype).to(dev), w.to(dtype).to(dev), b.to(dtype).to(dev), stride=stride, padding=1)
    assert torch.equal(y.cpu(), want.to(dtype))
    # the input gradient, whose workgroups put the same weights in another order: channel by channel, where that is whole 16-byte pieces
    g = torch.randint(-1, 2, want.shape, generator=gen).float()
    gx = jc.conv_nd_input(x.shape, w.to(dtype).to(dev), g.to(dtype).to(dev), stride=stride, padding=1)
    assert torch.equal(gx.cpu(), torch.nn.grad.conv2d_input(x.shape, w, g, stride=stride, padding=1).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [
    # batch, c_in, c_out, padded size, stride: row ends inside a stage's window, with the tensors' ends behind them and not
    (1, 32, 32, (33, 65), 2), (2, 40, 24, (9, 129), 2), (1, 64, 128, (17, 257), 2), (1, 16, 16, (5, 66), 2), (1, 16, 16, (6, 64), 2),
    (1, 16, 16, (34, 130), 1), (2, 24, 72, (10, 131), 1), (1, 70, 40, (7, 68), 1), (1, 8, 8, (4, 65), 1),
], ids=str)
def test_weight_gradient_at_the_ends_of_rows(case, dtype, dev):
    """Integers small enough for every sum to be exact: the kernel's result is the exact one, rounded once."""
    N, ci, co, size, stride = case
    gen = torch.Generator().manual_seed(6)
    out = tuple((s - 3) // stride + 1 for s in size)
    x = torch.randint(-3, 4, (N, ci, *size), generator=gen).double()
    g = torch.randint(-3, 4, (N, co, *out), generator=gen).double()
    want = torch.nn.grad.conv2d_weight(x, (co, ci, 3, 3), g, stride=stride)
    gw, gb = jc.conv_nd_weight(x.to(dtype).to(dev), (co, ci, 3, 3), g.to(dtype).to(dev), stride=stride, with_bias_grad=True)
    assert torch.equal(gw.cpu(), want.to(dtype)) and torch.equal(gb.cpu(), g.sum((0, 2, 3)).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [
    # batch, c_in, c_out, padded size, stride: blocks of one and two pairs, whose wavefronts share a stage's columns and rows: rows that
    # end inside each quarter, one row of a stage's two, more stages than workgroups
    (1, 32, 32, (3, 18), 1), (1, 64, 32, (4, 35), 1), (2, 32, 64, (5, 51), 1), (1, 64, 24, (130, 258), 1), (3, 8, 50, (67, 195), 1),
    (1, 32, 32, (3, 33), 2), (1, 64, 32, (5, 32), 2), (2, 32, 64, (9, 37), 2), (1, 50, 24, (131, 261), 2), (3, 96, 32, (66, 130), 2),
], ids=str)
def test_weight_gradient_of_narrow_blocks(case, dtype, dev):
    test_weight_gradient_at_the_ends_of_rows(case, dtype, dev)


@pytest.mark.parametrize("case", [
    # batch, c_in, c_out, size of x, padding: 8 x 64 tiles of the outputs (4 x 64 in the weight gradient), stages of 8 channels, blocks of
    # 16 and 32 produced channels, 7 or 14 input channels of the weight gradient, rows that are whole cache lines
    (1, 1, 1, (3, 3), (0, 0)), (2, 3, 16, (10, 66), (0, 0)), (1, 3, 17, (11, 67), (0, 0)), (2, 2, 33, (9, 65), (1, 1)), (1, 7, 5, (8, 64), (2, 2)),
    (2, 8, 32, (8, 128), (1, 1)), (1, 9, 15, (17, 129), (0, 1)), (3, 14, 16, (5, 40), (2, 0)), (1, 15, 65, (12, 96), (1, 1)), (1, 70, 4, (18, 70), (1, 0)),
    (2, 64, 64, (24, 33), (0, 0)), (1, 33, 63, (40, 100), (1, 1)), (5, 12, 12, (70, 200), (0, 0)),
], ids=str)
def test_fp32_on_the_matrix_instruction(case, dev):
    """Integers: every sum is exact, so are the results. Then no result further from float64's than its longest chain of fp32 additions allows:
    nine taps of a stage's 8 channels and the stages; eight pixels, then doubles, and two roundings to fp32, in the weight gradient."""
    N, ci, co, size, pad = case
    gen = torch.Generator().manual_seed(7)
    out = tuple(s + 2 * p - 2 for s, p in zip(size, pad))
    shapes = (N, ci, *size), (co, ci, 3, 3), (co,), (N, co, *out)

    def check(x, w, b, g, chain_y, chain_x, chain_w):
        y = jc.conv_nd(*(t.float().to(dev) for t in (x, w, b)), padding=pad)
        gx = jc.conv_nd_input(x.shape, w.float().to(dev), g.float().to(dev), padding=pad)
        gw, gb = jc.conv_nd_weight(x.float().to(dev), w.shape, g.float().to(dev), padding=pad, with_bias_grad=True)
        f, fx, fw = torch.nn.functional.conv2d, torch.nn.grad.conv2d_input, torch.nn.grad.conv2d_weight
        a = [t.abs() for t in (x, w, b, g)]
        for name, got, want, size_of, chain in (
                ("y", y, f(x, w, b, padding=pad), f(a[0], a[1], a[2], padding=pad), chain_y),
                ("gx", gx, fx(x.shape, w, g, padding=pad), fx(x.shape, a[1], a[3], padding=pad), chain_x),
                ("gw", gw, fw(x, w.shape, g, padding=pad), fw(a[0], w.shape, a[3], padding=pad), chain_w),
                ("gb", gb, g.sum((0, 2, 3)), a[3].sum((0, 2, 3)), chain_w)):
            off = (got.cpu().double() - want).abs() - chain * 2.0**-24 * size_of
            assert off.max() <= 0, f"{name}: {off.max()}"

    check(*(torch.randint(-3, 4, s, generator=gen).double() for s in shapes), 0, 0, 0)
    check(*(torch.randn(s, generator=gen).double() for s in shapes), 74 + ci // 8, 74 + co // 8, 12)


@pytest.mark.parametrize("case", [(2, 16, 128, 70, 131), (2, 128, 16, 66, 100), (1, 15, 18, 150, 200), (3, 12, 48, 90, 70)], ids=str)
def test_fp32_layers_of_few_channels_are_as_exact_as_their_kernels_in_every_direction(case, dev):
    """Also the directions that sums of bf16 parts do faster (relative error 2.5e-7 and 1.5e-7 to 3.7e-7 in the weight gradient) keep
    products and sums in fp32. A chain of n additions whose terms are as large on average is off by 2.5e-8 sqrt(n / 2), 2.5e-8 being
    what one rounding is off by on average: 1.5e-7 for a stage's 72 products, and a third of that again for what follows; 0.5e-7 for the
    weight gradient's eight pixels, and as much again for its last roundings."""
    N, ci, co, h, w_ = case
    gen = torch.Generator().manual_seed(8)
    x, w, g = (torch.randn(*s, generator=gen) for s in ((N, ci, h + 2, w_ + 2), (co, ci, 3, 3), (N, co, h, w_)))
    xd, wd, gd = x.double(), w.double(), g.double()
    y = jc.conv_nd(x.to(dev), w.to(dev))
    gx = jc.conv_nd_input(x.shape, w.to(dev), g.to(dev))
    gw = jc.conv_nd_weight(x.to(dev), w.shape, g.to(dev))
    assert rel_l2(y, torch.nn.functional.conv2d(xd, wd)) < 2e-7
    assert rel_l2(gx, torch.nn.grad.conv2d_input(xd.shape, wd, gd)) < 2e-7
    assert rel_l2(gw, torch.nn.grad.conv2d_weight(xd, wd.shape, gd)) < 1e-7


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n, c_in, c_out, size, mesh, beside", [
    (2, 32, 32, (40, 72), (2, 2), True),      # 36 runs of sums in pieces of four, beside the border
    (1, 5, 7, (9, 11), (3, 3), True),         # a single workgroup's partials, odd rows
    (2, 64, 64, (40, 70), (2, 2), True),      # 144 runs
    (1, 96, 80, (24, 66), (3, 1), True),      # several blocks of channels, no neighbour across W
    (1, 24, 7, (6, 20, 18), (2, 2, 2), True),  # three depth taps
    (4, 40, 8, (300, 310), (3, 3), True),     # long rows and columns; an odd number of whole octets of channels
    (4, 96, 8, (700, 24), (3, 3), False),     # a border of more blocks than the chip holds (8 a compute unit): launches of their own
])
def test_sums_left_for_the_border_launch_have_the_bits_of_their_own(n, c_in, c_out, size, mesh, beside, dtype, dev, monkeypatch):
    """Weight and bias gradient of the halo convolution, whose last sums run beside the border cells, == conv_nd_weight's."""
    ways, step_for = [], jc._step_for

    class Watched:  # a native step that says whether it left sums
        def __init__(self, step):
            self.step = step

        def __getattr__(self, name):
            return getattr(self.step, name)

        def finish(self, *a):
            ways.append(a[-1] is not None)
            return self.step.finish(*a)

    monkeypatch.setattr(jc, "_step_for", lambda *a: Watched(step_for(*a)))
    ns, gen = len(size), torch.Generator().manual_seed(5)
    k, ones = (3,) * ns, (1,) * ns
    rank = tuple(1 if m == 3 else 0 for m in mesh)
    geom = conv_geometry(size, mesh, rank, k, ones, ones, ones)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(dtype).to(dev)  # noqa: E731
    lead = (n, c_in)
    present = [o for o in geom.offsets() if all(v == 0 or 0 <= r + v < m for v, r, m in zip(o, rank, mesh))]
    recv_f = {o: rand(*lead, *geom.strip_extent(o, "assemble")) for o in present}
    recv_b = {o: rand(*lead, *geom.strip_extent(o, "fold")) for o in present}
    w, b = rand(c_out, c_in, *k).div_(8), rand(c_out)
    cfg = jc.HipConvNdConfig.for_rank(ns, b, TableExchange(recv_f, recv_b))
    groups = tuple(jc.TileGroup(m, r) for m, r in zip(mesh, rank))
    x, wl, bl = rand(*lead, *size).requires_grad_(), w.clone().requires_grad_(), b.clone().requires_grad_()
    y, x_aug = jc._ConvNd.apply(x, wl, bl, ones, ones, ones, groups, None, cfg)
    g = rand(*y.shape)
    gx, gw, gb = torch.autograd.grad(y, (x, wl, bl), g)
    lp = oh.local_padding(ones, mesh)
    want_w, want_b = jc.conv_nd_weight(x_aug, w.shape, g, padding=lp, with_bias_grad=True)
    assert torch.equal(gw, want_w) and torch.equal(gb, want_b)
    need = jc.conv_nd_input(x_aug.shape, w, g, padding=lp)
    from jigsaw_amd.halo import halo_fold

    assert torch.equal(gx, halo_fold(need, recv_b, geom))
    assert ways == [beside]
    assert _lib.load().jg_halo_fold_border_takes_sums(geom.theirs().c_geom(n * c_in), _lib.dtype_code(dtype)) == beside
    # y, rounded once: 2^-9 and 2^-12 of a value at most; fp32 sums of at most 864 products are off by 1e-6 at the most
    conv = torch.nn.functional.conv2d if ns == 2 else torch.nn.functional.conv3d
    exact = conv(x_aug.detach().cpu().double(), w.cpu().double(), b.cpu().double(), padding=lp)
    assert rel_l2(y, exact) < {torch.bfloat16: 2**-9, torch.float16: 2**-12, torch.float32: 0.0}[dtype] + 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("c_in, c_out, size", [
    (1, 1, (1, 1)), (3, 4, (8, 64)), (8, 3, (9, 65)), (9, 4, (17, 130)), (16, 5, (7, 63)), (17, 2, (30, 66)), (5, 33, (12, 70)), (20, 24, (25, 67)),
])
def test_fp32_layers_of_few_channels_at_the_edges_of_tiles(c_in, c_out, size, dev):
    """Four produced channels and fewer have products of their own (conv_f32.hip); stages of eight channels, tiles of 8 x 64."""
    torch.manual_seed(3)
    x, w, b = torch.randn(2, c_in, *size), torch.randn(c_out, c_in, 3, 3) / (9 * c_in) ** 0.5, torch.randn(c_out)
    g = torch.randn(2, c_out, *size)
    y = jc.conv_nd(x.to(dev), w.to(dev), b.to(dev), padding=1)
    gx = jc.conv_nd_input(x.shape, w.to(dev), g.to(dev), padding=1)
    # sums of at most 300 fp32 products: a relative error of 1e-6 is several times what their rounding leaves
    assert rel_l2(y, torch.nn.functional.conv2d(x.double(), w.double(), b.double(), padding=1)) < 1e-6
    assert rel_l2(gx, torch.nn.functional.conv_transpose2d(g.double(), w.double(), padding=1)) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("case", [
    # more than 64 channels on one side and up to 64 on the other, few workgroups: blocks of 32 produced channels and what they leave,
    # more stages than a patch is held for, several blocks of the weight gradient's columns
    (1, 17, 65, (10, 66), (0, 0)), (1, 128, 17, (9, 67), (1, 1)), (2, 64, 128, (19, 40), (1, 0)), (1, 97, 64, (8, 64), (2, 2)), (3, 40, 66, (30, 90), (0, 1)),
], ids=str)
def test_fp32_layers_of_many_channels_and_few_workgroups(case, dev):
    test_fp32_on_the_matrix_instruction(case, dev)
