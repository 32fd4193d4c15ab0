"""HIP attention core, fused ring step and ring loops against the oracle (GPU).

Tolerances: rel-L2 1e-5 for fp32 tensors, 2e-2 for bf16 / fp16; the
reference's own ring tests use atol 1e-3 fp32 / 1e-2 bf16
(tests/modules/attention/test_ring_attention.py:159-368).
"""

import pytest
import torch

from helpers import rel_l2
from jigsaw_amd import attention as ja
from oracle import attention as oa
from test_attention_routes import ONE_LAUNCH, one_launch_rows

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def _compute_units() -> int:
    return torch.cuda.get_device_properties(0).multi_processor_count


def _qkv(b, h, sq, sk, d, dtype, seed=0):
    torch.manual_seed(seed)
    q = (torch.randn(b, h, sq, d) / d**0.5).to(dtype)
    k = torch.randn(b, h, sk, d).to(dtype)
    v = torch.randn(b, h, sk, d).to(dtype)
    return q, k, v


CORE_SHAPES = [
    (3, 6, 64, 64, 16),   # the reference's ring test shape per chunk (b=3, h=6, n=16*4, d=16)
    (2, 2, 50, 70, 32),   # ragged
    (1, 3, 130, 33, 64),
    (1, 2, 128, 128, 64),  # MFMA path for bf16; few workgroups of 64 queries: the kernel of any head size
    (2, 2, 256, 384, 64),  # the same
    (1, 70, 256, 384, 64),  # the forward kernel of head size 64
    (1, 1, 40, 40, 128),
    (1, 2, 17, 9, 8),
    (1, 3, 256, 128, 32),  # head sizes below 64: kernels of 32 and 64 columns
    (2, 2, 128, 256, 16),
    (1, 2, 200, 300, 32),  # ragged queries and keys below head size 64
    (1, 2, 130, 260, 64),  # ragged at head size 64
    (1, 100, 130, 260, 64),  # and in its own forward kernel: 256 keys in the pipeline, 4 behind it
    (2, 1, 128, 130, 16),
    (1, 1, 70, 1000, 64),
    (1, 2, 128, 256, 128),  # head sizes 96 and 128: their own MFMA kernels for bf16
    (2, 2, 256, 128, 96),
    (1, 1, 384, 640, 128),
    (1, 2, 200, 300, 80),   # the kernel of 96 columns, 16 of them zero
    (1, 1, 130, 260, 128),  # ragged at head size 128: 256 keys rounded, 4 not
    (1, 1, 70, 200, 96),
    (1, 2, 256, 128, 72),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", CORE_SHAPES, ids=lambda s: "b{}h{}q{}k{}d{}".format(*s))
def test_core_forward_backward_match_oracle(shape, dtype, dev):
    b, h, sq, sk, d = shape
    q, k, v = _qkv(b, h, sq, sk, d, dtype)
    scale = d**-0.5
    want_o, want_l = oa.core_forward(q.double(), k.double(), v.double(), scale)
    out, lse, rng = ja.forward(q.to(dev), k.to(dev), v.to(dev), scale, 0.0, layout="bhsd")
    assert rng is None and out.dtype == dtype and lse.dtype == torch.float32
    assert rel_l2(out, want_o) < TOL[dtype], f"out {rel_l2(out, want_o):.3e}"
    assert rel_l2(lse, want_l) < max(TOL[dtype] * 0.1, 1e-5), f"lse {rel_l2(lse, want_l):.3e}"

    dout = torch.randn(b, h, sq, d).to(dtype)
    # backward from the oracle's own (global) out / lse, rounded as the ring would hold them
    o_in, l_in = want_o.to(dtype), want_l.float()
    wdq, wdk, wdv = oa.core_backward(dout.double(), q.double(), k.double(), v.double(), o_in.double(), l_in.double(), scale)
    dq, dk, dv = ja.backward(dout.to(dev), q.to(dev), k.to(dev), v.to(dev), o_in.to(dev), l_in.to(dev), scale, sq, sk)
    assert dq.dtype == dtype
    for name, got, want in (("dq", dq, wdq), ("dk", dk, wdk), ("dv", dv, wdv)):
        assert rel_l2(got, want) < TOL[dtype], f"{name} {rel_l2(got, want):.3e}"


@pytest.mark.parametrize(
    "b,h,n,d,P,dtype",
    [
        (3, 6, 16, 16, 4, torch.float32),
        (3, 6, 16, 16, 4, torch.bfloat16),
        (1, 2, 256, 64, 4, torch.bfloat16),
        (1, 2, 128, 64, 3, torch.float32),
        (1, 2, 128, 128, 3, torch.bfloat16),  # head sizes 128 and 96: their own kernels, merge fused as well
        (1, 1, 256, 96, 2, torch.bfloat16),
        (1, 2, 128, 128, 2, torch.float16),   # fp16 on the matrix cores, merge fused
        (1, 2, 256, 64, 2, torch.float16),    # fp16, head size 64
    ],
)
@pytest.mark.parametrize("rank", [0, 2])
def test_ring_forward_backward_match_full_attention(b, h, n, d, P, dtype, rank, dev):
    """Ring over P local chunks == full softmax attention over the concatenated K/V
    (the reference's method, test_ring_attention.py:267-275), forward and backward."""
    torch.manual_seed(1)
    scale = d**-0.5
    q = (torch.randn(b, h, n, d) / d**0.5).to(dtype)
    ks = [torch.randn(b, h, n, d).to(dtype) for _ in range(P)]
    vs = [torch.randn(b, h, n, d).to(dtype) for _ in range(P)]
    K = torch.cat(ks, 2).double().requires_grad_()
    V = torch.cat(vs, 2).double().requires_grad_()
    Q = q.double().requires_grad_()
    s = (Q @ K.mT) * scale
    full = torch.softmax(s, -1) @ V
    dout = torch.randn(b, h, n, d).to(dtype)
    full.backward(dout.double())

    out, lse = ja.ring_forward(q.to(dev), [t.to(dev) for t in ks], [t.to(dev) for t in vs], scale, rank=rank % P)
    assert out.dtype == dtype and lse.dtype == torch.float32
    assert rel_l2(out, full.detach()) < TOL[dtype], f"out {rel_l2(out, full.detach()):.3e}"
    lse_tol = 1e-5 if dtype == torch.float32 else 1e-3
    lse_err = rel_l2(lse, torch.logsumexp(s.detach(), -1))
    assert lse_err < lse_tol, f"lse {lse_err:.3e}"
    # the oracle's ring loop (its chunk order, merge form and roundings) agrees too
    o_or, l_or = oa.ring_forward(q.float(), [t.float() for t in ks], [t.float() for t in vs], scale, rank=rank % P)
    assert rel_l2(out, o_or) < TOL[dtype]

    dq, dks, dvs = ja.ring_backward(dout.to(dev), q.to(dev), out, lse, [t.to(dev) for t in ks], [t.to(dev) for t in vs], scale)
    assert rel_l2(dq, Q.grad) < TOL[dtype], f"dq {rel_l2(dq, Q.grad):.3e}"
    assert rel_l2(torch.cat(dks, 2), K.grad) < TOL[dtype], f"dk {rel_l2(torch.cat(dks, 2), K.grad):.3e}"
    assert rel_l2(torch.cat(dvs, 2), V.grad) < TOL[dtype], f"dv {rel_l2(torch.cat(dvs, 2), V.grad):.3e}"


@pytest.mark.parametrize("d", [64, 96, 128])
def test_fused_step_equals_core_plus_merge(d, dev):
    """The fused epilogue merge and the separate merge kernel give the same accumulator."""
    q, k, v = _qkv(1, 4, 256, 512, d, torch.bfloat16, seed=2)
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    scale = d**-0.5
    acc1 = torch.randn(1, 4, 256, d, device=dev)
    l1 = torch.randn(1, 4, 256, device=dev)
    acc2, l2 = acc1.clone(), l1.clone()
    ja.core_forward(q, k, v, scale, out_acc=acc1, lse_acc=l1, want_out=False)
    out_j, l_j = ja.core_forward(q, k, v, scale)
    acc2, l2 = ja.fused_online_softmax_merge_(acc2, l2, out_j, l_j, "bhsd")
    torch.testing.assert_close(acc1, acc2, atol=1e-6, rtol=1e-6)
    torch.testing.assert_close(l1, l2, atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("d,sq,sk", [(32, 200, 300), (64, 130, 33), (128, 257, 96), (64, 128, 4096)])
def test_fp32_matrix_core_step_with_merge(d, sq, sk, dev):
    """fp32 on the matrix cores, ragged lengths: the step against the oracle in fp64, the fused merge
    against the separate merge kernel and against the merge done in fp64, and a second merge on top."""
    q, k, v = _qkv(2, 3, sq, sk, d, torch.float32, seed=3)
    scale = d**-0.5
    want_o, want_l = oa.core_forward(q.double(), k.double(), v.double(), scale)
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    out_j, l_j = ja.core_forward(q, k, v, scale)
    assert rel_l2(out_j, want_o) < 1e-5 and rel_l2(l_j, want_l) < 1e-5
    acc1 = torch.randn(2, 3, sq, d, device=dev)
    l1 = torch.randn(2, 3, sq, device=dev)
    acc0, l0 = acc1.double().cpu(), l1.double().cpu()
    acc2, l2 = acc1.clone(), l1.clone()
    assert ja.core_forward(q, k, v, scale, out_acc=acc1, lse_acc=l1, want_out=False) == (None, None)
    acc2, l2 = ja.fused_online_softmax_merge_(acc2, l2, out_j, l_j, "bhsd")
    torch.testing.assert_close(acc1, acc2, atol=2e-6, rtol=2e-6)
    torch.testing.assert_close(l1, l2, atol=2e-6, rtol=2e-6)
    l_new = torch.logaddexp(l0, want_l)
    acc_new = acc0 * (l0 - l_new).exp().unsqueeze(-1) + want_o * (want_l - l_new).exp().unsqueeze(-1)
    assert rel_l2(acc1, acc_new) < 1e-5 and rel_l2(l1, l_new) < 1e-5
    # a fresh accumulator (lse -inf) takes the step as it is, and hands it out on request
    acc3 = torch.zeros_like(acc1)
    l3 = torch.full_like(l1, float("-inf"))
    out3, lse3 = ja.core_forward(q, k, v, scale, out_acc=acc3, lse_acc=l3)
    assert torch.equal(out3, out_j) and torch.equal(lse3, l_j)
    torch.testing.assert_close(acc3, out_j, atol=1e-7, rtol=1e-6)
    torch.testing.assert_close(l3, l_j, atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("d", [8, 16, 96])
def test_fp32_head_sizes_between_the_matrix_core_sizes(d, dev):
    q, k, v = _qkv(1, 2, 70, 45, d, torch.float32, seed=4)
    scale = d**-0.5
    want_o, want_l = oa.core_forward(q.double(), k.double(), v.double(), scale)
    dout = torch.randn(1, 2, 70, d)
    wdq, wdk, wdv = oa.core_backward(dout.double(), q.double(), k.double(), v.double(), want_o, want_l, scale)
    out, lse = ja.core_forward(q.to(dev), k.to(dev), v.to(dev), scale)
    assert out.shape == q.shape and rel_l2(out, want_o) < 1e-5 and rel_l2(lse, want_l) < 1e-5
    dq, dk, dv = ja.core_backward(dout.to(dev), q.to(dev), k.to(dev), v.to(dev), want_o.float().to(dev), want_l.float().to(dev), scale)
    for got, want in ((dq, wdq), (dk, wdk), (dv, wdv)):
        assert got.shape == want.shape and rel_l2(got, want) < 1e-5


@pytest.mark.parametrize("h", [2, 70], ids=["kernel of any head size", "kernel of head size 64"])
@pytest.mark.parametrize("pattern", ["late_spike", "rising", "first_tile_low", "huge_logits", "one_hot_rows"])
def test_mfma_forward_when_the_running_max_moves(pattern, h, dev):
    """Launches of few workgroups of 64 queries run the kernel of any head size; the head-size-64 kernel keeps a per-query reference exponent that follows the running
    max lazily (it moves only when a tile exceeds it by 2^8) and folds it into the score
    product. Score patterns that move the max late, often, by hundreds of powers of two, or
    start far below zero must give the fp64 softmax all the same (bf16 bar), and so must
    the merge into a ring accumulator that already holds a chunk."""
    torch.manual_seed(11)
    b, sq, sk, d = 1, 256, 1024, 64
    assert (h * (sq // 64) > _compute_units()) == (h == 70)
    q = torch.randn(b, h, sq, d)
    k = torch.randn(b, h, sk, d)
    v = torch.randn(b, h, sk, d)
    if pattern == "late_spike":        # a few keys near the end dominate everything before them
        k[:, :, 900:905] *= 12.0
    elif pattern == "rising":          # the max moves in almost every tile
        k *= torch.linspace(0.2, 6.0, sk)[None, None, :, None]
    elif pattern == "first_tile_low":  # the first tiles hold only very negative scores
        k[:, :, :128] = -3.0 * q[:, :, :1].mean(2, keepdim=True).expand(b, h, 128, d) - 4.0
        q = q.abs()
    elif pattern == "huge_logits":     # logits in the thousands: softmax is one-hot, nothing may overflow
        q, k = q * 30.0, k * 30.0
    elif pattern == "one_hot_rows":    # every query has exactly one matching key, somewhere in the chunk
        k = torch.nn.functional.normalize(k, dim=-1) * 40.0
        q = k[:, :, torch.randperm(sk)[:sq]].clone()
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    scale = d**-0.5
    want_o, want_l = oa.core_forward(q.double(), k.double(), v.double(), scale)
    out, lse = ja.core_forward(q.to(dev), k.to(dev), v.to(dev), scale)
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    assert rel_l2(out, want_o) < 2e-2, f"out {rel_l2(out, want_o):.3e}"
    assert rel_l2(lse, want_l) < 2e-3, f"lse {rel_l2(lse, want_l):.3e}"  # the core test's bar for bf16
    # the same chunk as the second step of a ring whose first chunk is ordinary
    k0, v0 = torch.randn(b, h, 256, d).bfloat16(), torch.randn(b, h, 256, d).bfloat16()
    ring_o, ring_l = ja.ring_forward(q.to(dev), [k0.to(dev), k.to(dev)], [v0.to(dev), v.to(dev)], scale)
    full_o, full_l = oa.core_forward(q.double(), torch.cat([k0, k], 2).double(), torch.cat([v0, v], 2).double(), scale)
    assert rel_l2(ring_o, full_o) < 2e-2 and rel_l2(ring_l, full_l) < 2e-3


def test_config4_shape_properties(dev):
    """Config 4 at full size: 8 heads, 4096 queries, 4 chunks of 4096 keys, d = 64, bf16.
    Size-independent checks: ring over 4 chunks == one core call over the concatenated
    K/V; permuting the chunks changes nothing beyond rounding; 128 sampled query rows
    match the fp64 oracle over all 16384 keys."""
    torch.manual_seed(3)
    b, h, n, d, P = 1, 8, 4096, 64, 4
    scale = d**-0.5
    q = (torch.randn(b, h, n, d, device=dev) / 8).bfloat16()
    ks = [torch.randn(b, h, n, d, device=dev).bfloat16() for _ in range(P)]
    vs = [torch.randn(b, h, n, d, device=dev).bfloat16() for _ in range(P)]
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=1)
    full_o, full_l = ja.core_forward(q, torch.cat(ks, 2), torch.cat(vs, 2), scale)
    assert rel_l2(out, full_o) < 1e-2
    assert rel_l2(lse, full_l) < 1e-5
    out2, lse2 = ja.ring_forward(q, ks[::-1], vs[::-1], scale, rank=0)
    assert rel_l2(out2, out) < 1e-2 and rel_l2(lse2, lse) < 1e-5
    rows = torch.arange(0, n, 32)
    qs = q[:, :, rows].double().cpu()
    K, V = torch.cat(ks, 2).double().cpu(), torch.cat(vs, 2).double().cpu()
    s = (qs @ K.mT) * scale
    want = torch.softmax(s, -1) @ V
    assert rel_l2(out[:, :, rows], want) < 2e-2
    assert rel_l2(lse[:, :, rows], torch.logsumexp(s, -1)) < 1e-4


def test_config4_shape_in_fp32_on_the_matrix_cores(dev):
    """Config 4's ring at full size with fp32 inputs (8 heads, 4096 queries, 4 chunks of 4096 keys, d = 64):
    ring of fused steps == one core call over the concatenated K/V, forward and backward; sampled
    rows against fp64; and the bf16 kernels' result within bf16's tolerance of it."""
    torch.manual_seed(6)
    b, h, n, d, P = 1, 8, 4096, 64, 4
    scale = d**-0.5
    q = torch.randn(b, h, n, d, device=dev) / 8
    ks = [torch.randn(b, h, n, d, device=dev) for _ in range(P)]
    vs = [torch.randn(b, h, n, d, device=dev) for _ in range(P)]
    dout = torch.randn(b, h, n, d, device=dev)
    Kc, Vc = torch.cat(ks, 2), torch.cat(vs, 2)
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=1)
    full_o, full_l = ja.core_forward(q, Kc, Vc, scale)
    assert out.dtype == torch.float32 and rel_l2(out, full_o) < 1e-5 and rel_l2(lse, full_l) < 1e-6
    rows = torch.arange(5, n, 64)
    qs = q[:, :, rows].double().cpu()
    s = (qs @ Kc.double().cpu().mT) * scale
    assert rel_l2(out[:, :, rows], torch.softmax(s, -1) @ Vc.double().cpu()) < 1e-5
    assert rel_l2(lse[:, :, rows], torch.logsumexp(s, -1)) < 1e-6
    o16, l16 = ja.ring_forward(q.bfloat16(), [t.bfloat16() for t in ks], [t.bfloat16() for t in vs], scale, rank=1)
    assert rel_l2(o16, out) < 2e-2 and rel_l2(l16, lse) < 1e-3

    dq, dks, dvs = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    fdq, fdk, fdv = ja.core_backward(dout, q, Kc, Vc, out, lse, scale)
    assert rel_l2(dq, fdq) < 1e-5 and rel_l2(torch.cat(dks, 2), fdk) < 1e-5 and rel_l2(torch.cat(dvs, 2), fdv) < 1e-5
    # sampled keys of one chunk against fp64 (every query takes part)
    keys = torch.arange(3, n, 128)
    Q, O, dO, L = q.double().cpu(), out.double().cpu(), dout.double().cpu(), lse.double().cpu()
    Kj, Vj = ks[2][:, :, keys].double().cpu(), vs[2][:, :, keys].double().cpu()
    p = torch.exp((Q @ Kj.mT) * scale - L.unsqueeze(-1))
    delta = (dO * O).sum(-1, keepdim=True)
    ds = p * (dO @ Vj.mT - delta) * scale
    assert rel_l2(dvs[2][:, :, keys], p.mT @ dO) < 1e-5
    assert rel_l2(dks[2][:, :, keys], ds.mT @ Q) < 1e-5


def test_config4_backward_shape_properties(dev):
    """Config 4 backward at full size (8 heads, 4096 queries, 4 chunks of 4096 keys, d = 64,
    bf16), from the GLOBAL out / lse as the ring holds them (backward.py:176-270).
    Size-independent checks against fp64 on samples: the rows of ``sum_j dq_j`` for 128
    sampled queries (each needs all 16384 keys), and the rows of ``dk_j`` / ``dv_j`` for 128
    sampled keys of every chunk (each needs all 4096 queries); plus ``sum_j dq_j`` == dq of
    one core call over the concatenated K/V."""
    torch.manual_seed(5)
    b, h, n, d, P = 1, 8, 4096, 64, 4
    scale = d**-0.5
    q = (torch.randn(b, h, n, d, device=dev) / 8).bfloat16()
    ks = [torch.randn(b, h, n, d, device=dev).bfloat16() for _ in range(P)]
    vs = [torch.randn(b, h, n, d, device=dev).bfloat16() for _ in range(P)]
    dout = torch.randn(b, h, n, d, device=dev).bfloat16()
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=0)
    dq, dks, dvs = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    assert dq.dtype == torch.bfloat16 and len(dks) == P and len(dvs) == P

    Kc, Vc = torch.cat(ks, 2), torch.cat(vs, 2)
    dq_full, dk_full, dv_full = ja.backward(dout, q, Kc, Vc, out, lse, scale, n, P * n)
    assert rel_l2(dq, dq_full) < 1e-2
    assert rel_l2(torch.cat(dks, 2), dk_full) < 1e-2 and rel_l2(torch.cat(dvs, 2), dv_full) < 1e-2

    # fp64 on the host from the same bf16 inputs and the same (rounded) global out / lse
    Q, K, V = q.double().cpu(), Kc.double().cpu(), Vc.double().cpu()
    dO, O, L = dout.double().cpu(), out.double().cpu(), lse.double().cpu()
    D = (dO * O).sum(-1)  # (b, h, n)
    rows = torch.arange(5, n, 32)
    s = (Q[:, :, rows] @ K.mT) * scale
    p = torch.exp(s - L[:, :, rows, None])
    dp = dO[:, :, rows] @ V.mT
    ds = p * (dp - D[:, :, rows, None]) * scale
    assert rel_l2(dq[:, :, rows], ds @ K) < 2e-2, f"dq rows {rel_l2(dq[:, :, rows], ds @ K):.3e}"
    keys = torch.arange(3, n, 32)
    for j in range(P):
        kj, vj = K[:, :, j * n + keys], V[:, :, j * n + keys]
        s = (Q @ kj.mT) * scale  # (b, h, n, 128)
        p = torch.exp(s - L[..., None])
        want_dv = p.mT @ dO
        ds = p * (dO @ vj.mT - D[..., None]) * scale
        want_dk = ds.mT @ Q
        assert rel_l2(dvs[j][:, :, keys], want_dv) < 2e-2, f"dv chunk {j}: {rel_l2(dvs[j][:, :, keys], want_dv):.3e}"
        assert rel_l2(dks[j][:, :, keys], want_dk) < 2e-2, f"dk chunk {j}: {rel_l2(dks[j][:, :, keys], want_dk):.3e}"


@pytest.mark.parametrize("b,h,n,nk,P", [(1, 2, 256, 128, 3), (2, 3, 128, 384, 1), (1, 8, 512, 256, 5), (1, 1, 128, 128, 16)])
def test_backward_over_resident_chunks_in_one_pass(b, h, n, nk, P, dev):
    """``backward_chunks`` (one dQ launch over all chunks, the chunk as a grid dimension of the dK/dV
    kernel): dK / dV of every chunk have the bits of the per-chunk ``core_backward`` (same kernel, same
    arithmetic per chunk), dQ is the fp32 sum of the chunks rounded once, checked against fp64
    (backward.py:176-277 visits chunk s at step s and adds the steps' dq)."""
    torch.manual_seed(11)
    d = 64
    scale = d**-0.5
    q = (torch.randn(b, h, n, d, device=dev) / 4).bfloat16()
    ks = [torch.randn(b, h, nk, d, device=dev).bfloat16() for _ in range(P)]
    vs = [torch.randn(b, h, nk, d, device=dev).bfloat16() for _ in range(P)]
    dout = torch.randn(b, h, n, d, device=dev).bfloat16()
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=0)
    res = ja.backward_chunks(dout, q, out, lse, ks, vs, scale)
    assert res is not None, "bf16 at head size 64 with lengths in multiples of 128 is what the one-pass kernels cover"
    dq, dks, dvs = res
    want_dq = torch.zeros(q.shape, dtype=torch.float64)
    for j in range(P):
        dq_j, dk_j, dv_j = ja.core_backward(dout, q, ks[j], vs[j], out, lse, scale)
        assert torch.equal(dks[j], dk_j) and torch.equal(dvs[j], dv_j), f"chunk {j}"
        ref = oa.core_backward(dout.double().cpu(), q.double().cpu(), ks[j].double().cpu(), vs[j].double().cpu(),
                                        out.double().cpu(), lse.double().cpu(), scale)
        want_dq += ref[0]
        assert rel_l2(dk_j, ref[1]) < 2e-2 and rel_l2(dv_j, ref[2]) < 2e-2
    assert rel_l2(dq, want_dq) < 2e-2, f"dq {rel_l2(dq, want_dq):.3e}"
    # and through ring_backward, which takes this route by itself
    dq2, dks2, dvs2 = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    assert torch.equal(dq2, dq) and all(torch.equal(a, c) for a, c in zip(dks2, dks))


@pytest.mark.parametrize("heads", [2, 150], ids=["32-query workgroups", "128-query workgroups"])
@pytest.mark.parametrize("n,nk,P", [(64, 128, 1), (65, 129, 1), (128, 192, 1), (127, 257, 1), (33, 320, 1), (96, 383, 1), (130, 448, 1), (64, 640, 1), (100, 1100, 1),
                                    (64, 128, 2), (70, 190, 3), (128, 256, 5)], ids=str)
def test_query_gradient_at_the_ends_of_its_key_tiles(heads, n, nk, P, dev):
    """One to eighteen tiles of a key half (four a round, then one by one), chunks that end inside a tile, workgroups of 32 queries (the kernel
    of any head size) and of 128. dS is rounded to bf16,
    half of 2^-8, and so is the result; twice that leaves room for the exponential and the sums."""
    torch.manual_seed(n + nk)
    d, scale = 64, 0.125
    q, dout = (torch.randn(1, heads, n, d, device=dev).bfloat16() for _ in range(2))
    ks, vs = ([torch.randn(1, heads, nk, d, device=dev).bfloat16() for _ in range(P)] for _ in range(2))
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=0)
    dq, _, _ = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    Q, K, V, dO, O, L = (t[0].double().cpu() for t in (q, torch.cat(ks, 2), torch.cat(vs, 2), dout, out, lse))
    dS = torch.exp(Q @ K.mT * scale - L[..., None]) * (dO @ V.mT - (dO * O).sum(-1, keepdim=True)) * scale
    off = (dq[0].double().cpu() - dS @ K).abs() - 2.0**-8 * (dS.abs() @ K.abs() + (dS @ K).abs())
    assert off.max() <= 0, off.max()


@pytest.mark.parametrize("heads,n,nk,P", [(100, 65, 129, 1), (100, 96, 383, 1), (100, 127, 257, 1), (100, 128, 192, 1), (100, 128, 640, 1), (100, 128, 256, 5),
                                          (100, 70, 190, 3), (60, 130, 448, 1), (60, 150, 1100, 2), (60, 192, 128, 1)], ids=str)
def test_query_gradient_in_workgroups_of_64_queries(heads, n, nk, P, dev):
    """The same between the two: enough rows for workgroups of 32 to fill the chip, too few for those of 128 to do so."""
    cus = _compute_units()
    assert heads * -(-n // 32) > cus and 2 * heads * -(-n // 128) <= cus
    test_query_gradient_at_the_ends_of_its_key_tiles(heads, n, nk, P, dev)


@pytest.mark.parametrize("heads,n,nk,P", [(100, 65, 257, 8), (100, 128, 130, 16), (60, 150, 683, 3), (60, 129, 1024, 2), (100, 70, 146, 14), (70, 97, 2047, 1)], ids=str)
def test_query_gradient_in_workgroups_of_64_queries_over_many_keys(heads, n, nk, P, dev):
    """Lengths that are no multiples of 128, on either side of 2048 keys: four groups of wavefronts that take tiles of all chunks in turn."""
    test_query_gradient_in_workgroups_of_64_queries(heads, n, nk, P, dev)


def test_backward_over_chunks_declines_what_it_does_not_cover(dev):
    q = torch.randn(1, 1, 128, 64, device=dev)
    k = [torch.randn(1, 1, 128, 64, device=dev)]
    assert ja.backward_chunks(q, q, q, q[..., 0], k, k, 0.125) is None  # fp32
    qb = q.bfloat16()
    kb = [torch.randn(1, 1, 96, 64, device=dev).bfloat16()]
    assert ja.backward_chunks(qb, qb, qb, q[..., 0], kb, kb, 0.125) is None  # 96 keys
    many = [torch.randn(1, 1, 128, 64, device=dev).bfloat16() for _ in range(17)]
    assert ja.backward_chunks(qb, qb, qb, q[..., 0], many, many, 0.125) is None  # more chunks than a call takes


@pytest.mark.parametrize("b,sq,sk,d,P", [
    (1, 1, 1, 4, 1), (3, 33, 31, 32, 16), (2, 197, 70, 20, 5), (300, 100, 40, 32, 2), (513, 33, 33, 24, 2),  # 32, 64 and 128 rows a workgroup
    (2, 65, 129, 64, 3), (300, 70, 33, 40, 1), (512, 129, 20, 64, 1),
    (4, 171, 95, 80, 3), (280, 66, 32, 96, 2), (600, 32, 17, 88, 1),
    (2, 40, 64, 128, 4), (260, 96, 50, 100, 1), (512, 64, 34, 128, 1),
])
def test_fp32_ring_in_one_launch_each_way(b, sq, sk, d, P, dev):
    """fp32 rings over resident chunks against fp64: every kernel width with and without columns past the head size, every
    number of rows a workgroup takes, groups of wavefronts without a step, lengths that end inside a step."""
    torch.manual_seed(8)
    scale = d**-0.5
    q, dout = torch.randn(b, 1, sq, d), torch.randn(b, 1, sq, d)
    ks, vs = ([torch.randn(b, 1, sk, d) for _ in range(P)] for _ in range(2))
    want_o, want_l = oa.ring_forward(q.double(), [t.double() for t in ks], [t.double() for t in vs], scale)
    on = lambda ts: [t.to(dev) for t in ts]  # noqa: E731
    res = ja._resident_forward(q.to(dev), on(ks), on(vs), scale)
    assert res is not None
    out, lse = res
    assert out.dtype == lse.dtype == torch.float32 and rel_l2(out, want_o) < 1e-5 and rel_l2(lse, want_l) < 1e-5
    dq, dks, dvs = ja.ring_backward(dout.to(dev), q.to(dev), want_o.float().to(dev), want_l.float().to(dev), on(ks), on(vs), scale)
    total = torch.zeros_like(q, dtype=torch.float64)
    for k, v, dk, dv in zip(ks, vs, dks, dvs):
        a, b_, c = oa.core_backward(dout.double(), q.double(), k.double(), v.double(), want_o, want_l, scale)
        total += a
        # with one key to attend the true dK is 0: what is left are roundings of the products that cancel
        floor = 1e-6 * float((dout.double().unsqueeze(-2) * v.double().mean(-2, keepdim=True).unsqueeze(-2)).norm())
        assert rel_l2(dv, c) < 1e-5 and float((dk.cpu().double() - b_).norm()) < 1e-5 * float(b_.norm()) + floor
    assert float((dq.cpu().double() - total).norm()) < 1e-5 * float(total.norm()) + floor


@pytest.mark.parametrize("h,n,d,P", [(256, 256, 32, 16), (128, 256, 64, 12), (16, 700, 96, 16)])
def test_fp32_rings_of_many_chunks_stay_as_exact_as_one_chunk(h, n, d, P, dev):
    """Output and dQ are sums over the keys of all chunks. A sum of n terms of either sign, whose partial sums grow as the square root of their
    number, is sqrt(n / 2) roundings off: with the steps of 32 keys summed by themselves sqrt((32 + n / 32) / 2), here up to
    16.3 of 2^-24 = 9.7e-7 at 16000 keys; in one chain 5.3e-6 (1.1e-6 to 2.0e-6 seen, a rounding is off by less than its bound)."""
    torch.manual_seed(13)
    nk, scale, some = 1000, d**-0.5, slice(0, h, h // 3)
    q, dout = (torch.randn(1, h, n, d, device=dev) for _ in range(2))
    ks, vs = ([torch.randn(1, h, nk, d, device=dev) for _ in range(P)] for _ in range(2))
    out, lse = ja.ring_forward(q, ks, vs, scale)
    Q, G, K, V = q[0, some].double(), dout[0, some].double(), torch.cat([k[0, some] for k in ks], -2).double(), torch.cat([v[0, some] for v in vs], -2).double()
    S = Q @ K.mT.contiguous() * scale
    L = S.logsumexp(-1)
    assert rel_l2(out[0, some], (S - L[..., None]).exp() @ V) < 1e-6 and rel_l2(lse[0, some], L) < 2.0**-23
    dq, _, _ = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    P_, O = (S - lse[0, some, :, None].double()).exp(), out[0, some].double()
    assert rel_l2(dq[0, some], P_ * (G @ V.mT.contiguous() - (G * O).sum(-1, keepdim=True)) * scale @ K) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [4, 20, 32, 40, 96, 128])
def test_gradient_of_a_bias_that_was_not_given(d, dtype, dev):
    """``want_dbias`` without a bias at any head size: the gradient that a bias of zeros gets."""
    torch.manual_seed(12)
    q, k, v, dout = (torch.randn(2, 2, n, d, device=dev).to(dtype) for n in (37, 41, 41, 37))
    out, lse = ja.core_forward(q, k, v, 0.125)
    zeros = torch.zeros(2, 37, 41, device=dev)
    for a, b in zip(ja.core_backward(dout, q, k, v, out, lse, 0.125, want_dbias=True),
                    ja.core_backward(dout, q, k, v, out, lse, 0.125, bias=zeros, want_dbias=True)):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("b", [3, 300, 520])  # 32, 64 and 128 rows a workgroup
@pytest.mark.parametrize("dead", [(0, 32), (32, 64), (0, 70), (64, 70)])
def test_fp32_steps_without_a_finite_score_weigh_nothing(b, dead, dev):
    """Keys whose scores are all -inf, by whole steps of a wavefront or a whole chunk: the others' softmax, in whichever
    group of wavefronts and at whichever place of the walk they fall (fp64 reference; the bar of the other fp32 tests)."""
    torch.manual_seed(9)
    q = torch.randn(b, 1, 33, 32).abs()
    ks, vs = ([torch.randn(b, 1, 70, 32) for _ in range(2)] for _ in range(2))
    ks[0][..., dead[0] : dead[1], :] = float("-inf")
    want_o, want_l = oa.core_forward(q.double(), torch.cat(ks, -2).double(), torch.cat(vs, -2).double(), 0.125)
    out, lse = ja._resident_forward(q.to(dev), [t.to(dev) for t in ks], [t.to(dev) for t in vs], 0.125)
    assert rel_l2(out, want_o) < 1e-5 and rel_l2(lse, want_l) < 1e-5


@pytest.mark.parametrize("dtype,bar", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2), (torch.float16, 4e-3)], ids=str)
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("b", [3, 300, 520])
def test_a_chunk_without_a_finite_score_weighs_nothing_step_by_step(b, d, dtype, bar, dev):
    """The same with the chunks arriving one by one, the dead one before, between and behind the others: the merge inside the
    core's launch and the one of its own agree with the resident route. Where no key is left the row is 0 and its lse
    -inf, and a NaN stays one."""
    torch.manual_seed(9)
    q = torch.randn(b, 1, 33, d).abs().to(dtype)
    ks, vs = ([torch.randn(b, 1, 70, d).to(dtype) for _ in range(2)] for _ in range(2))
    want_o, want_l = oa.core_forward(q.double(), torch.cat(ks, -2).double(), torch.cat(vs, -2).double(), 0.125)
    q, dead, vd = q.to(dev), torch.full((b, 1, 70, d), float("-inf"), dtype=dtype, device=dev), torch.ones(b, 1, 70, d, dtype=dtype, device=dev)
    live = [(k.to(dev), v.to(dev)) for k, v in zip(ks, vs)]
    nothing = (torch.zeros(q.shape, device=dev), torch.full(q.shape[:-1], float("-inf"), device=dev))
    merged = lambda k, v, out, lse: ja.fused_online_softmax_merge_(out, lse, *ja.core_forward(q, k, v, 0.125), "bhsd")  # noqa: E731
    for step in (lambda k, v, out, lse: ja.attend_step_(q, k, v, 0.125, out, lse), merged):

        def ring(chunks):
            out, lse = (t.clone() for t in nothing)
            for k, v in chunks:
                out, lse = step(k, v, out, lse)
            return out, lse

        for at in range(3):
            out, lse = ring([*live[:at], (dead, vd), *live[at:]])
            assert rel_l2(out, want_o) < bar and rel_l2(lse, want_l) < bar
        out, lse = ring([(dead, vd), (dead, vd)])
        assert torch.equal(out, nothing[0]) and torch.equal(lse, nothing[1])
        # a score that is NaN in the first row of the first entry
        sick = live[0][0].clone()
        sick[0, 0, 3, 1] = float("nan")
        out, lse = ring([(sick, live[0][1]), live[1]])
        assert out[0].isnan().all() and lse[0].isnan().all() and not out[1:].isnan().any() and not lse[1:].isnan().any()


@pytest.mark.parametrize("dtype,bar", [(torch.float32, 1e-5), (torch.bfloat16, 4e-3), (torch.float16, 5e-4)], ids=str)
@pytest.mark.parametrize("b,sq,sk,d,P", [
    # one launch: groups without a tile, one row in the last tile, chunks of fewer than 128 keys, workgroups of 32, 64 and 128 rows
    (3, 33, 130, 64, 2), (3, 1, 150, 64, 1), (3, 70, 70, 32, 2), (71, 132, 95, 24, 3), (68, 80, 141, 32, 1), (5, 66, 150, 96, 1), (13, 102, 130, 128, 2),
    # two launches, of both kernels of heads of 64
    (18, 1000, 300, 64, 2), (300, 70, 140, 64, 1), (80, 300, 150, 32, 4), (60, 200, 200, 96, 2), (60, 200, 100, 128, 2), (3, 128, 128, 64, 2),
])
def test_keys_without_a_finite_score_get_no_gradient(b, sq, sk, d, P, dtype, bar, dev):
    """dK and dV of keys whose scores are all -inf are 0, and the others' are those of the formula, against float64 (tolerances as
    in :func:`test_backward_in_one_launch`; dQ is NaN by the formula: 0 x -inf). A whole block of dead keys and single ones. No
    query is 0, which makes a score of NaN. A probability that is kept in three bf16 parts is 2^-126 where it is 0."""
    gen = torch.Generator().manual_seed(b + sq)
    q, g = (torch.randn(1, b, sq, d, generator=gen).abs() + 0.01).to(dtype), torch.randn(1, b, sq, d, generator=gen).to(dtype)
    ks, vs = ([torch.randn(1, b, sk, d, generator=gen).to(dtype) for _ in range(P)] for _ in range(2))
    dead = torch.zeros(sk, dtype=torch.bool)
    dead[:32] = dead[sk - 1] = dead[sk // 2] = True
    ks[0][..., dead, :] = float("-inf")
    out, lse = ja.ring_forward(q.to(dev), [t.to(dev) for t in ks], [t.to(dev) for t in vs], d**-0.5)
    _, dk, dv = ja.ring_backward(g.to(dev), q.to(dev), out, lse, [t.to(dev) for t in ks], [t.to(dev) for t in vs], d**-0.5)
    k, v = torch.cat(ks, 2).double(), torch.cat(vs, 2).double()
    _, wk, wv = oa.core_backward(g.double(), q.double(), k, v, out.cpu().double(), lse.cpu().double(), d**-0.5)
    for got, want in ((dk, wk), (dv, wv)):
        assert (got[0][..., dead, :].abs() <= sq * 2.0**-120).all()
        got = torch.cat(got, 2).cpu().double()
        assert (got - want).norm() <= bar * want.norm()


@pytest.mark.parametrize("d,n,nk", [(64, 192, 160), (32, 100, 70), (128, 64, 96)])
def test_fp32_ring_step_takes_the_fused_merge(d, n, nk, dev):
    """``attend_step_`` on fp32 tensors at the head sizes of the fp32 matrix-core kernel: one launch that merges in
    its epilogue, against the core followed by the separate merge (forward.py:64-96) and the fp64 oracle."""
    torch.manual_seed(3)
    scale = d**-0.5
    q = torch.randn(1, 2, n, d, device=dev)
    ks = [torch.randn(1, 2, nk, d, device=dev) for _ in range(3)]
    vs = [torch.randn(1, 2, nk, d, device=dev) for _ in range(3)]
    assert ja._fused_ok(q, ks[0])
    out = torch.zeros_like(q)
    lse = torch.full(q.shape[:-1], float("-inf"), device=dev)
    out2, lse2 = out.clone(), lse.clone()
    for kj, vj in zip(ks, vs):
        out, lse = ja.attend_step_(q, kj, vj, scale, out, lse)
        o_j, l_j = ja.core_forward(q, kj, vj, scale)
        out2, lse2 = ja.fused_online_softmax_merge_(out2, lse2, o_j, l_j, "bhsd")
    want_o, want_l = oa.ring_forward(q.double().cpu(), [t.double().cpu() for t in ks], [t.double().cpu() for t in vs], scale)
    assert rel_l2(out, want_o) < 1e-5 and rel_l2(lse, want_l) < 1e-5
    assert rel_l2(out, out2) < 1e-6 and rel_l2(lse, lse2) < 1e-6


def test_window_attention_with_bias_and_mask(dev):
    """Swin-style windows: (B, nW, heads, N, d) with a (nW, heads, N, N) bias that
    holds -inf entries (shift mask), forward and backward incl. the bias gradient."""
    torch.manual_seed(4)
    B, nW, heads, N, d = 2, 6, 4, 64, 32
    q, k, v = (torch.randn(B, nW, heads, N, d) for _ in range(3))
    bias = torch.randn(nW, heads, N, N) * 0.5
    mask = torch.zeros(nW, 1, N, N)
    mask[1, :, :32, 32:] = float("-inf")
    mask[1, :, 32:, :32] = float("-inf")
    bias = bias + mask
    qd, kd, vd = (t.double().requires_grad_() for t in (q, k, v))
    bd = bias.double().requires_grad_()
    want = oa.window_attention(qd, kd, vd, bd)
    g = torch.randn_like(want)
    want.backward(g)
    qg, kg, vg, bg = (t.to(dev).requires_grad_() for t in (q, k, v, bias))
    out = ja.window_attention(qg, kg, vg, bg)
    assert rel_l2(out, want.detach()) < 1e-5
    out.backward(g.float().to(dev))
    assert rel_l2(qg.grad, qd.grad) < 1e-5 and rel_l2(kg.grad, kd.grad) < 1e-5 and rel_l2(vg.grad, vd.grad) < 1e-5
    assert rel_l2(bg.grad, torch.nan_to_num(bd.grad)) < 1e-5
    # broadcast bias (heads, N, N), bf16 inputs
    out_b = ja.window_attention(qg.detach().bfloat16(), kg.detach().bfloat16(), vg.detach().bfloat16(), bg.detach()[0])
    want_b = oa.window_attention(q.bfloat16().double(), k.bfloat16().double(), v.bfloat16().double(), bias[0].double())
    assert rel_l2(out_b, want_b) < 2e-2


@pytest.mark.parametrize("with_bias", [True, False])
def test_window_kernels_bf16(with_bias, dev):
    """64-token windows, head size 32, bf16: the dedicated window kernels (one wavefront
    per window and head), forward and backward with the bias gradient, against the
    oracle in fp64 on the same bf16 inputs. 15 entries: the last workgroup is ragged."""
    torch.manual_seed(11)
    B, nW, heads, N, d = 1, 5, 3, 64, 32
    q, k, v = (torch.randn(B, nW, heads, N, d).bfloat16() for _ in range(3))
    bias = None
    if with_bias:
        bias = torch.randn(nW, heads, N, N) * 0.5
        bias[2, :, :24, 24:] = float("-inf")
        bias[2, :, 24:, :24] = float("-inf")
    qd, kd, vd = (t.double().requires_grad_() for t in (q, k, v))
    bd = bias.double().requires_grad_() if with_bias else None
    want = oa.window_attention(qd, kd, vd, bd if with_bias else torch.zeros(N, N, dtype=torch.float64))
    g = torch.randn_like(want).bfloat16()
    want.backward(g.double())
    qg, kg, vg = (t.to(dev).requires_grad_() for t in (q, k, v))
    bg = bias.to(dev).requires_grad_() if with_bias else None
    out = ja.window_attention(qg, kg, vg, bg)
    assert out.dtype == torch.bfloat16
    assert rel_l2(out, want.detach()) < 2e-2
    out.backward(g.to(dev))
    assert rel_l2(qg.grad, qd.grad) < 2e-2 and rel_l2(kg.grad, kd.grad) < 2e-2 and rel_l2(vg.grad, vd.grad) < 2e-2
    if with_bias:
        assert rel_l2(bg.grad, torch.nan_to_num(bd.grad)) < 2e-2
        assert (bg.grad[2, :, :24, 24:] == 0).all()
    # lse of the same call through the core interface
    out2, lse = ja.core_forward(qg.detach(), kg.detach(), vg.detach(), d ** -0.5, bias=bg.detach() if with_bias else None)
    s = torch.einsum("bwhqd,bwhkd->bwhqk", q.double(), k.double()) * d ** -0.5
    if with_bias:
        s = s + bias.double()
    assert rel_l2(lse, torch.logsumexp(s, -1)) < 1e-4
    assert torch.equal(out2, out.detach())


def test_core_argument_errors(dev):
    q = torch.zeros(1, 2, 8, 16, device=dev)
    with pytest.raises(NotImplementedError):
        ja.forward(q, q, q, 0.25, 0.0, layout="bshd")
    with pytest.raises(NotImplementedError):
        ja.forward(q, q, q, 0.25, 0.1)
    with pytest.raises(RuntimeError):
        ja.forward(q, q.bfloat16(), q, 0.25)
    with pytest.raises(ValueError):
        ja.forward(q, q[:, :1], q, 0.25)
    wide = torch.zeros(1, 2, 8, 136, device=dev)  # beyond the largest head size the kernels are built for
    with pytest.raises(NotImplementedError):
        ja.forward(wide, wide, wide, 0.25)


@pytest.mark.parametrize("d", [5, 40, 72])
def test_head_sizes_between_the_kernel_sizes_are_zero_padded(d, dev):
    q, k, v = _qkv(1, 2, 33, 47, d, torch.float32)
    scale = d**-0.5
    want_o, want_l = oa.core_forward(q.double(), k.double(), v.double(), scale)
    out, lse, _ = ja.forward(q.to(dev), k.to(dev), v.to(dev), scale)
    assert out.shape == q.shape and rel_l2(out, want_o) < 1e-5 and rel_l2(lse, want_l) < 1e-5
    dout = torch.randn(1, 2, 33, d)
    want = oa.core_backward(dout.double(), q.double(), k.double(), v.double(), want_o, want_l, scale)
    got = ja.backward(dout.to(dev), q.to(dev), k.to(dev), v.to(dev), want_o.float().to(dev), want_l.float().to(dev), scale, 33, 47)
    for g, w in zip(got, want):
        assert g.shape == w.shape and rel_l2(g, w) < 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,sq,sk,d,P", [
    (1, 2, 1, 1, 64, 1), (1, 1, 129, 31, 64, 3), (2, 3, 127, 33, 64, 2), (1, 4, 300, 257, 64, 5), (1, 2, 128, 4097, 64, 1),
    (1, 2, 1, 1, 32, 2), (1, 3, 130, 65, 8, 3), (2, 2, 100, 97, 40, 2), (1, 2, 257, 129, 80, 3), (1, 1, 33, 31, 96, 16),
    (1, 2, 200, 300, 128, 2), (1, 40, 300, 260, 128, 2), (3, 90, 130, 100, 96, 1), (3, 90, 130, 100, 32, 1), (1, 5, 640, 513, 128, 1),
], ids=str)
def test_ring_of_any_lengths_in_one_pass(b, h, sq, sk, d, P, dtype, dev):
    """Lengths at and beside the tile edges (32 keys, 64 rows, 128 resident rows), head sizes between the kernels' widths,
    few and many workgroups (which split a workgroup's tiles over 1, 2 or 4 groups of wavefronts): forward and backward
    over resident chunks against the oracle, and the fused merge of the same step against core + merge."""
    torch.manual_seed(sq + sk + d)
    q = (torch.randn(b, h, sq, d, device=dev) / d**0.5).to(dtype)
    ks = [torch.randn(b, h, sk, d, device=dev).to(dtype) for _ in range(P)]
    vs = [torch.randn(b, h, sk, d, device=dev).to(dtype) for _ in range(P)]
    dout = torch.randn(b, h, sq, d, device=dev).to(dtype)
    scale = d**-0.5
    dbl = lambda t: t.double().cpu()  # noqa: E731
    assert ja._resident(q, ks, vs)
    out, lse = ja.ring_forward(q, ks, vs, scale, rank=P // 2)
    want_o, want_l = oa.ring_forward(dbl(q), [dbl(t) for t in ks], [dbl(t) for t in vs], scale)
    assert rel_l2(out, want_o) < 1e-2 and rel_l2(lse, want_l) < 1e-3
    dq, dks, dvs = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    parts = [oa.core_backward(dbl(dout), dbl(q), dbl(k), dbl(v), dbl(out), dbl(lse), scale) for k, v in zip(ks, vs)]
    want_dq = sum(p[0] for p in parts)
    if sk * P > 1:  # one key: dq and dk are zero in exact arithmetic
        assert rel_l2(dq, want_dq) < 2e-2
        assert rel_l2(torch.stack(dks), torch.stack([p[1] for p in parts])) < 2e-2
    assert rel_l2(torch.stack(dvs), torch.stack([p[2] for p in parts])) < 2e-2
    acc1, l1 = torch.randn(b, h, sq, d, device=dev), torch.randn(b, h, sq, device=dev)
    acc2, l2 = acc1.clone(), l1.clone()
    assert ja._fused_ok(q, ks[0])
    acc1, l1 = ja.attend_step_(q, ks[0], vs[0], scale, acc1, l1)
    o_j, l_j = ja.core_forward(q, ks[0], vs[0], scale)
    acc2, l2 = ja.fused_online_softmax_merge_(acc2, l2, o_j, l_j, "bhsd")
    assert rel_l2(acc1, acc2) < 1e-5 and rel_l2(l1, l2) < 1e-5


def _differ(a, b) -> float:
    return (a != b).double().mean().item()


# Two fp32 evaluations differ by about 4e-6 of a value, and 16-bit values lie 2^-8 (bf16) and 2^-11 (fp16) of it apart, so up
# to 0.2 % and 1.6 % of the rounded results may differ; with probabilities rounded to 16 bits more than a third do.
_STRAYS = {torch.bfloat16: 0.005, torch.float16: 0.02}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 88, 128])
@pytest.mark.parametrize("h,sq,sk,P", [
    # workgroups of 32, 64 and 128 queries and, apart from them, keys; key groups with fewer tiles than others, none at all, one key
    (2, 33, 40, 2), (3, 65, 300, 1), (60, 150, 70, 3), (70, 65, 290, 1), (100, 130, 140, 2), (140, 130, 64, 1), (300, 70, 33, 1), (5, 64, 1025, 2), (260, 1, 130, 1),
])
def test_workgroups_of_every_width(h, sq, sk, P, d, dtype, dev):
    test_ring_of_any_lengths_in_one_pass(1, h, sq, sk, d, P, dtype, dev)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,sq,sk,d,P", [
    # workgroups of 128 rows on 256 compute units, up to 64 columns: two blocks of 32 rows a wavefront where the keys are many; blocks and
    # wavefronts without a row, key groups with fewer tiles, chunks shorter than 128 keys; four wavefronts, then eight
    (780, 1, 129, 24, 16), (780, 33, 600, 32, 1), (400, 97, 161, 32, 13), (520, 33, 600, 32, 1), (520, 33, 90, 32, 1), (260, 65, 2049, 64, 1), (257, 128, 100, 64, 16), (260, 33, 257, 48, 4), (300, 31, 33, 40, 3),
    (120, 130, 4100, 64, 1), (125, 129, 293, 56, 14),
])
def test_workgroups_that_fill_the_chip(h, sq, sk, d, P, dtype, dev):
    test_ring_of_any_lengths_in_one_pass(1, h, sq, sk, d, P, dtype, dev)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,sq,sk,d,P", [(4, 100, 100, 64, 2), (4, 300, 127, 64, 3), (3, 64, 31, 64, 1), (4, 100, 65, 40, 2), (3, 130, 97, 32, 5),
                                         (3, 130, 97, 96, 2), (3, 200, 127, 128, 2), (300, 130, 100, 80, 1)], ids=str)
def test_short_key_ranges_keep_probabilities_in_fp32(h, sq, sk, d, P, dtype, dev):
    """Fewer than 128 keys a chunk: the same results as the one-thread-per-row kernels (a bias of zeros selects them), which
    hold probabilities and dS in fp32, forward and backward, and over the chunks of a ring."""
    torch.manual_seed(sk + d)
    mk = lambda n: torch.randn(1, h, n, d, device=dev).to(dtype)  # noqa: E731
    q, dout, ks, vs, scale = mk(sq), mk(sq), [mk(sk) for _ in range(P)], [mk(sk) for _ in range(P)], d**-0.5
    out, lse = ja.ring_forward(q, ks, vs, scale)
    k, v = torch.cat(ks, -2), torch.cat(vs, -2)
    zeros = torch.zeros(sq, sk * P, device=dev)
    want_o, want_l = ja.core_forward(q, k, v, scale, bias=zeros)
    assert _differ(out, want_o) < _STRAYS[dtype] and rel_l2(lse, want_l) < 1e-6
    dq, dks, dvs = ja.ring_backward(dout, q, want_o, want_l, ks, vs, scale)
    want = ja.core_backward(dout, q, k, v, want_o, want_l, scale, bias=zeros)
    for got, w in zip((dq, torch.cat(dks, -2), torch.cat(dvs, -2)), want):
        assert _differ(got, w) < _STRAYS[dtype]


@pytest.mark.parametrize("h,sq,sk,d,P,dtype", [
    (3, 130, 300, 64, 1, torch.bfloat16), (3, 256, 1000, 64, 3, torch.bfloat16), (30, 256, 1000, 128, 2, torch.bfloat16),
    (3, 130, 255, 96, 3, torch.bfloat16), (30, 256, 1000, 128, 2, torch.float16), (3, 130, 255, 96, 3, torch.float16),
    # workgroups of 128 queries, at bf16 and head size 64 the kernel of that size
    (100, 130, 300, 64, 1, torch.bfloat16), (70, 256, 1000, 64, 3, torch.bfloat16), (70, 256, 1000, 128, 2, torch.bfloat16), (100, 130, 255, 96, 3, torch.float16),
], ids=str)
def test_keys_behind_the_last_whole_tile_keep_probabilities_in_fp32(h, sq, sk, d, P, dtype, dev):
    """Forward at a head size that fills a kernel: the keys of a chunk behind its last multiple of 128. The whole tiles
    have probabilities near 0 here, so that the last keys alone make the result."""
    torch.manual_seed(sk + d)
    mk = lambda n: torch.randn(1, h, n, d, device=dev).to(dtype)  # noqa: E731
    q, k, vs, scale = mk(sq), mk(sk), [mk(sk) for _ in range(P)], d**-0.5
    q[..., 0], k[..., 0] = 16, 0
    k[:, :, : sk // 128 * 128, 0] = -8 * d**0.5  # scores of -128 and below
    out, lse = ja.ring_forward(q, [k] * P, vs, scale)
    want_o, want_l = ja.core_forward(q, torch.cat([k] * P, -2), torch.cat(vs, -2), scale, bias=torch.zeros(sq, sk * P, device=dev))
    assert _differ(out, want_o) < _STRAYS[dtype] and rel_l2(lse, want_l) < 1e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h", [2, 140], ids=["workgroups of 32 queries", "workgroups of 128 queries"])
@pytest.mark.parametrize("sq,sk,d", [(70, 100, 64), (70, 1000, 64), (70, 100, 128), (70, 200, 96), (70, 33, 32)], ids=str)
def test_infinite_values_stay_infinite_where_probabilities_are_kept_in_fp32(sq, sk, d, h, dtype, dev):
    """A value that is infinite makes its output column infinite, not NaN, also as the last key of a range."""
    torch.manual_seed(sk)
    q, k, v = (torch.randn(1, h, n, d, device=dev).to(dtype) for n in (sq, sk, sk))
    v[..., sk - 1, 3], v[..., sk // 2, 5] = float("inf"), float("-inf")
    out, _ = ja.core_forward(q, k, v, d**-0.5)
    want, _ = ja.core_forward(q, k, v, d**-0.5, bias=torch.zeros(sq, sk, device=dev))
    assert torch.isinf(want[..., 3]).all() and torch.isinf(want[..., 5]).all()
    assert torch.equal(out[..., (3, 5)], want[..., (3, 5)]) and torch.isfinite(out[..., 6:]).all()


@pytest.mark.parametrize("sk", [100, 200, 256])
def test_misaligned_heads_of_64_run_the_kernels_that_take_any_alignment(sk, dev):
    """The C entry points on tensors that start 2 bytes off a 16-byte boundary: the one-thread-per-row kernels."""
    from jigsaw_amd import _lib

    torch.manual_seed(sk)
    lib, h, sq, d, scale = _lib.load(), 2, 130, 64, 0.125
    off = lambda *s: torch.randn(h * s[0] * s[1] + 1, device=dev).bfloat16()[1:].view(h, *s)  # noqa: E731
    q, dout, k, v, out, dq, dk, dv = off(sq, d), off(sq, d), off(sk, d), off(sk, d), off(sq, d), off(sq, d), off(sk, d), off(sk, d)
    lse = torch.empty(h, sq, device=dev)
    ws = torch.empty(int(lib.jg_attn_bwd_workspace_bytes(h, sq, sk, d)), dtype=torch.uint8, device=dev)
    p, bf16, stream = _lib.ptr, _lib.dtype_code(torch.bfloat16), _lib.stream_ptr(q.device)
    _lib.check(lib.jg_attn_fwd(p(out), p(lse), p(q), p(k), p(v), h, sq, sk, d, scale, None, 0, None, None, bf16, stream))
    _lib.check(lib.jg_attn_bwd(p(dq), p(dk), p(dv), p(dout), p(q), p(k), p(v), p(out), p(lse), h, sq, sk, d, scale, None, 0, None, bf16,
                               p(ws), ws.numel(), stream))
    want_o, want_l = ja.core_forward(q.clone(), k.clone(), v.clone(), scale, bias=torch.zeros(sq, sk, device=dev))
    want = ja.core_backward(dout, q, k, v, want_o, want_l, scale, bias=torch.zeros(sq, sk, device=dev))
    assert torch.equal(out, want_o) and torch.equal(lse, want_l)
    for got, w in zip((dq, dk, dv), want):
        assert torch.equal(got, w)
    acc = torch.zeros(h, sq, d, device=dev)
    rc = lib.jg_attn_fwd(None, None, p(q), p(k), p(v), h, sq, sk, d, scale, None, 0, p(acc), p(lse), bf16, stream)
    assert rc == -2


@pytest.mark.parametrize("h,sq,sk,P,d", [(2, 2048, 2048, 2, 40), (1, 2050, 4097, 1, 16), (1, 2048, 1400, 3, 56), (8, 4096, 4096, 1, 32), (2, 2048, 4096, 1, 36)], ids=str)
def test_narrow_heads_on_long_sequences_run_as_64_columns(h, sq, sk, P, d, dev):
    """bf16 heads of fewer than 64 columns where the 64-column kernels with zero columns are the faster ones: the ring, the
    core and the step that merges, against 64 bits; results keep their own width."""
    torch.manual_seed(sk + d)
    mk = lambda n: (torch.randn(1, h, n, d, device=dev)).bfloat16()  # noqa: E731
    q, dout, ks, vs, scale = mk(sq), mk(sq), [mk(sk) for _ in range(P)], [mk(sk) for _ in range(P)], d**-0.5
    assert ja._as_64_columns(q, ks[0], P) and not ja._as_64_columns(q.half(), ks[0], P) and not ja._as_64_columns(q[..., :1024, :], ks[0], P)
    leaves = [t.double().requires_grad_() for t in (q, torch.cat(ks, -2), torch.cat(vs, -2))]
    scores = leaves[0] @ leaves[1].transpose(-1, -2) * scale
    want_l = torch.logsumexp(scores, -1)
    want_o = torch.exp(scores - want_l[..., None]) @ leaves[2]
    want = torch.autograd.grad(want_o, leaves, dout.double())
    out, lse = ja.ring_forward(q, ks, vs, scale)
    assert out.shape == q.shape and out.is_contiguous() and rel_l2(out, want_o) < 1e-2 and rel_l2(lse, want_l) < 1e-3
    dq, dks, dvs = ja.ring_backward(dout, q, out, lse, ks, vs, scale)
    assert all(t.shape == ks[0].shape and t.is_contiguous() for t in (*dks, *dvs)) and dq.shape == q.shape
    for got, w in zip((dq, torch.cat(dks, -2), torch.cat(dvs, -2)), want):
        assert rel_l2(got, w) < 2e-2
    acc, l_acc = torch.zeros(q.shape, device=dev), torch.full(q.shape[:-1], float("-inf"), device=dev)
    for k, v in zip(ks, vs):
        acc, l_acc = ja.attend_step_(q, k, v, scale, acc, l_acc)
    assert rel_l2(acc, want_o) < 1e-2 and rel_l2(l_acc, want_l) < 1e-3
    if P == 1:
        got = ja.core_backward(dout, q, ks[0], vs[0], out, lse, scale)
        for g, w in zip(got, want):
            assert g.shape == w.shape and rel_l2(g, w) < 2e-2


@pytest.mark.parametrize("h,d", [(17, 16), (33, 56)])
def test_narrow_heads_with_many_rows_keep_their_width(h, d, dev):
    """Beyond 2^16 rows the kernels of the heads' own width are the faster ones: their results against those of the same heads
    with zero columns up to 64, which add nothing. Both round probabilities and results to bf16, twice 2^-8 apart at most."""
    torch.manual_seed(d)
    mk = lambda: torch.randn(1, h, 4096, d, device=dev).bfloat16()  # noqa: E731
    q, k, v, dout = mk(), mk(), mk(), mk()
    assert not ja._as_64_columns(q, k) and ja._as_64_columns(q[:, :16], k[:, :16])
    wide = [torch.nn.functional.pad(t, (0, 64 - d)) for t in (q, k, v, dout)]
    out, lse = ja.ring_forward(q, [k], [v], d**-0.5)
    out64, lse64 = ja.ring_forward(wide[0], [wide[1]], [wide[2]], d**-0.5)
    assert rel_l2(out, out64[..., :d]) < 2.0**-7 and rel_l2(lse, lse64) < 1e-5
    got = ja.ring_backward(dout, q, out, lse, [k], [v], d**-0.5)
    want = ja.ring_backward(wide[3], wide[0], torch.nn.functional.pad(out, (0, 64 - d)), lse, [wide[1]], [wide[2]], d**-0.5)
    for g, w in zip((got[0], got[1][0], got[2][0]), (want[0], want[1][0], want[2][0])):
        assert rel_l2(g, w[..., :d]) < 2.0**-7


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,sq,sk,d,P", list(ONE_LAUNCH))
def test_backward_in_one_launch(h, sq, sk, d, P, dtype, dev):
    """dQ, dK and dV of small rings, one launch with delta formed twice, against float64: one rounding to 16 bits of dS and P (none in short
    chunks) and one of the result, 2^-9 (bf16) and 2^-12 (fp16) each at most, of terms of both signs."""
    if _compute_units() == 256:
        assert one_launch_rows(h, sq, sk, d, P, dtype) == ONE_LAUNCH[h, sq, sk, d, P][dtype == torch.float16]
    gen = torch.Generator().manual_seed(h + sq)
    q, g = ((torch.randn(1, h, sq, d, generator=gen) * f).to(dtype) for f in (d**-0.5, 1.0))
    ks, vs = ([torch.randn(1, h, sk, d, generator=gen).to(dtype) for _ in range(P)] for _ in range(2))
    out, lse = ja.ring_forward(q.to(dev), [t.to(dev) for t in ks], [t.to(dev) for t in vs], 0.7)
    dq, dk, dv = ja.ring_backward(g.to(dev), q.to(dev), out, lse, [t.to(dev) for t in ks], [t.to(dev) for t in vs], 0.7)
    k, v = torch.cat(ks, 2).double(), torch.cat(vs, 2).double()
    wq, wk, wv = oa.core_backward(g.double(), q.double(), k, v, out.cpu().double(), lse.cpu().double(), 0.7)
    tol = {torch.bfloat16: 4e-3, torch.float16: 5e-4}[dtype]
    for got, want in ((dq, wq), (torch.cat(dk, 2), wk), (torch.cat(dv, 2), wv)):
        # (a single key: P is 1, dS and with it dQ and dK are what rounding leaves of 0)
        assert (got.cpu().double() - want).norm() <= tol * (want.norm() if sk * P > 2 else g.double().norm() * 3)
