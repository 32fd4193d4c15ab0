"""Ring-attention step on the GPU: attention core, log-sum-exp merge, ring loops.

Host-side mirror of

* the attention-core contract ``forward(q, k, v, scale, dropout_p, seed=None, *,
  layout) -> (out, logsumexp, rng_state)`` and ``backward(grad_out, q, k, v, out,
  logsumexp, scale, *extra, ...) -> (dq, dk, dv)``
  (jigsaw/modules/attention/_functional/cores/__init__.py:1-15), i.e. what
  ``RingAttentionConfig.attn_core_forward_fn / attn_core_backward_fn`` hold
  (jigsaw/modules/attention/_config.py:459-464);
* the fused merge hook ``fused_online_softmax_merge_``
  (jigsaw/modules/attention/_functional/_merge_kernel.py:88-172);
* the per-rank loops of ``ring_forward`` / ``ring_backward``
  (jigsaw/modules/attention/_functional/forward.py:160-199, backward.py:176-270)
  over K/V chunks that are already local. Circulating the chunks between ranks is
  outside this module.
"""

from __future__ import annotations

import ctypes
import math
from collections.abc import Sequence

import torch

from . import _lib
from ._autograd import saved_rows

_SUPPORTED_O = (torch.float16, torch.bfloat16, torch.float32)


# --------------------------------------------------------------------------- #
# merge hook
# --------------------------------------------------------------------------- #
def fused_online_softmax_merge_(o1, l1, o2, l2, layout):
    """HIP stand-in for the Triton merge: mutates ``o1``, returns ``(o1, l_new)``.

    Returns ``None`` for anything the kernel does not cover, exactly where the
    reference's hook does (_merge_kernel.py:117-138), so the caller's eager
    fallback stays reachable.
    """
    if not o1.is_cuda:
        return None
    if layout not in ("bhsd", "bshd"):
        return None
    if o1.dtype not in _SUPPORTED_O or o2.dtype not in _SUPPORTED_O:
        return None
    if o1.shape != o2.shape or not o1.is_contiguous() or not o2.is_contiguous():
        return None
    if l1.shape != l2.shape or l1.dim() != 3 or not l1.is_contiguous() or not l2.is_contiguous():
        return None
    if o1.dtype != torch.float32 and o1.dtype != o2.dtype:
        return None
    is_bshd = layout == "bshd"
    b, s1, s2, d = o1.shape
    n = s1 if is_bshd else s2
    h = s2 if is_bshd else s1
    if l1.shape != (b, h, n) or l1.dtype != torch.float32:
        return None
    l2f = l2 if l2.dtype == torch.float32 else l2.to(torch.float32)
    l_new = torch.empty_like(l1, dtype=torch.float32)
    rc = _lib.load().jg_lse_merge(
        _lib.ptr(o1), _lib.ptr(l1), _lib.ptr(o2), _lib.ptr(l2f), _lib.ptr(l_new), b, h, n, d, int(is_bshd),
        _lib.dtype_code(o1.dtype), _lib.dtype_code(o2.dtype), _lib.stream_ptr(o1.device),
    )
    _lib.check(rc, "jg_lse_merge")
    return o1, l_new


# --------------------------------------------------------------------------- #
# attention core
# --------------------------------------------------------------------------- #
def _flat(t: torch.Tensor) -> tuple[int, int, int]:
    if t.dim() < 3:
        raise ValueError(f"expected (..., s, d), got shape {tuple(t.shape)}")
    batch = 1
    for s in t.shape[:-2]:
        batch *= int(s)
    return batch, int(t.shape[-2]), int(t.shape[-1])


def _check_qkv(q, k, v):
    _lib.require_gpu(q, k, v)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError(f"q, k, v must share a dtype, got {q.dtype}, {k.dtype}, {v.dtype}")
    if k.shape != v.shape or q.shape[:-2] != k.shape[:-2] or q.shape[-1] != k.shape[-1]:
        raise ValueError(f"shape mismatch: q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)}")


def _bias_args(bias, batch, sq, sk):
    if bias is None:
        return None, 0
    bias = bias.to(torch.float32).contiguous()
    if bias.dim() < 2 or tuple(bias.shape[-2:]) != (sq, sk):
        raise ValueError(f"bias must end in ({sq}, {sk}), got {tuple(bias.shape)}")
    period = bias.numel() // (sq * sk)
    if period == 0 or batch % period:
        raise ValueError(f"bias with {period} matrices does not tile a batch of {batch}")
    return bias, period


# --------------------------------------------------------------------------- #
# The 16-bit matrix-core kernels take any lengths and any head size that is a multiple of 8 up to
# 128, the fp32 ones any lengths at multiples of 4 up to 128, the one-thread-per-row kernels (bias, more
# batch entries than a grid dimension holds) a few head sizes. Other head sizes get zero columns:
# they add nothing to the scores and give zero output columns, which are dropped. Narrow bf16 heads on
# long sequences get them too, by a rule of the time when the kernels of 64 columns were the faster ones (_as_64_columns).
# --------------------------------------------------------------------------- #
_KERNEL_HEAD_SIZES = (8, 16, 32, 64, 96, 128)
_F32_MFMA_HEAD_SIZES = (32, 64, 128)
_MOST_BATCH = 65535
_MOST_ROWS = 1 << 23  # rows of one head: the kernels address them by 32-bit byte offsets


def _mfma16(q, k, bias=None) -> bool:
    """Whether the 16-bit matrix-core kernels take q against the keys k (their head size padded to a multiple of 8)."""
    return (bias is None and q.dtype in (torch.bfloat16, torch.float16) and q.shape[-1] <= 128
            and max(q.shape[-2], k.shape[-2]) <= _MOST_ROWS and math.prod(q.shape[:-2]) <= _MOST_BATCH)


def _mfma32(q, k) -> bool:
    """Whether the fp32 matrix-core kernels take q against the keys k (their head size padded to a multiple of 4)."""
    return (q.dtype == torch.float32 and q.shape[-1] <= 128 and max(q.shape[-2], k.shape[-2]) <= _MOST_ROWS
            and math.prod(q.shape[:-2]) <= _MOST_BATCH)


def _kernel_head_size(d: int, dtype=None, has_bias: bool = False) -> int:
    """Smallest head size the kernels beside the 16-bit matrix-core ones are built for that holds ``d`` columns;
    ``d`` itself beyond the largest. fp32 without a bias goes to the widths of its matrix-core kernels,
    everything else to the sizes of the one-thread-per-row kernels."""
    sizes = _F32_MFMA_HEAD_SIZES if dtype == torch.float32 and not has_bias else _KERNEL_HEAD_SIZES
    return next((n for n in sizes if n >= d), d)


def _as_64_columns(q, k, chunks: int = 1) -> bool:
    """Whether bf16 heads of fewer than 64 columns against ``chunks`` chunks like ``k`` run with zero columns up to 64, copies there
    and back included, on the kernels of that size. The line was drawn when those were the faster ones there: forward / backward, us, own width and
    as 64 columns, 8 heads x 4096 x 4096 keys, 16 columns 89/170 and 76/172, 32 85/159 and 73/164, 48 105/206 and 81/180; 2 x 8192 x 8192, 32
    100/205 and 96/206; 8 x 8192 x 4096, 40 117/317 and 118/288. With two blocks of rows a wavefront and one launch backward the kernels of any width are now as
    fast or faster at every one of them: 43/93 and 68/144, 39/92 and 67/152, 67/166 and 75/164; 48/119 and 86/201; 98/280 and 111/267. More rows were
    always better off there: 32 heads x 4096, 16 columns 125/297 and 193/455, 48 180/474 and 214/528, 64 heads, 56 354/952 and 435/1081. The rule stands
    until it is taken out together with the tests that ask for its answers."""
    # (host.cpp's may_want_64_columns asks here about the rows, keys and widths that it names: no others may get a yes)
    *lead, sq, d = q.shape
    if sq < 2048 or d >= 64 or q.dtype != torch.bfloat16:
        return False
    keys, rows = k.shape[-2] * chunks, math.prod(lead) * sq
    if keys < 4096:
        return False
    if 24 < d <= 32:
        return rows * keys >= 1 << 27 and sq >= 4096 and rows <= 1 << 15
    return rows <= 1 << 16


def _padded_head_size(q, k, bias, want_dbias: bool = False) -> int:
    d = q.shape[-1]
    if want_dbias:  # the gradient of a bias comes from the one-thread-per-row kernels, also where there is none to add
        return _kernel_head_size(d, q.dtype, True)
    if bias is None and _mfma32(q, k):
        return (d + 3) // 4 * 4
    if not _mfma16(q, k, bias):
        return _kernel_head_size(d, q.dtype, bias is not None)
    return 64 if _as_64_columns(q, k) else (d + 7) // 8 * 8


def _pad_last(t: torch.Tensor, to: int) -> torch.Tensor:
    return t if t.shape[-1] == to else torch.nn.functional.pad(t, (0, to - t.shape[-1]))


def _dense(t: torch.Tensor) -> torch.Tensor:
    """``t`` contiguous on a 16-byte boundary (a view into a larger tensor may start anywhere)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def core_forward(q, k, v, scale, bias=None, out_acc=None, lse_acc=None, want_out=True):
    """One attention core call; optionally merges into ``(out_acc, lse_acc)`` in place.

    Returns ``(out, lse)`` (``None`` each when ``want_out`` is false).
    """
    _check_qkv(q, k, v)
    d, dp = q.shape[-1], _padded_head_size(q, k, bias)
    if dp != d and out_acc is None and lse_acc is None:
        out, lse = _core_forward(_pad_last(q, dp), _pad_last(k, dp), _pad_last(v, dp), scale, bias, None, None, want_out)
        return (out[..., :d].contiguous() if want_out else None), lse
    return _core_forward(q, k, v, scale, bias, out_acc, lse_acc, want_out)


def _core_forward(q, k, v, scale, bias=None, out_acc=None, lse_acc=None, want_out=True):
    q, k, v = _dense(q), _dense(k), _dense(v)
    batch, sq, d = _flat(q)
    sk = int(k.shape[-2])
    bias_t, period = _bias_args(bias, batch, sq, sk)
    out = torch.empty_like(q) if want_out else None
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device=q.device) if want_out else None
    rc = _lib.load().jg_attn_fwd(
        _lib.ptr(out), _lib.ptr(lse), _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), batch, sq, sk, d, float(scale),
        _lib.ptr(bias_t), period, _lib.ptr(out_acc), _lib.ptr(lse_acc), _lib.dtype_code(q.dtype),
        _lib.stream_ptr(q.device),
    )
    _lib.check(rc, "jg_attn_fwd")
    return out, lse


def forward(q, k, v, scale=0.0, dropout_p=0.0, seed=None, *, layout="bhsd"):
    """Attention core forward with the reference's signature
    (cores/math.py:31-78, cores/sdpa.py:17-85): ``(out, logsumexp, rng_state)``."""
    if layout != "bhsd":
        raise NotImplementedError(f"the HIP core is bhsd-only; got layout={layout!r}")
    if dropout_p != 0.0:
        raise NotImplementedError("attention dropout is not supported by the HIP core")
    scale = scale or (q.size(-1) ** -0.5)
    out, lse = core_forward(q, k, v, scale)
    return out, lse, None


def core_backward(grad_out, q, k, v, out, logsumexp, scale, bias=None, want_dbias=False):
    """``(dq, dk, dv[, dbias])`` of one chunk from the global ``out`` / ``logsumexp``."""
    _check_qkv(q, k, v)
    _lib.require_gpu(grad_out, out, logsumexp)
    d, dp = q.shape[-1], _padded_head_size(q, k, bias, want_dbias)
    if dp != d:
        res = _core_backward(_pad_last(grad_out, dp), _pad_last(q, dp), _pad_last(k, dp), _pad_last(v, dp),
                             _pad_last(out, dp), logsumexp, scale, bias, want_dbias)
        return tuple(t[..., :d].contiguous() for t in res[:3]) + tuple(res[3:])
    return _core_backward(grad_out, q, k, v, out, logsumexp, scale, bias, want_dbias)


def _core_backward(grad_out, q, k, v, out, logsumexp, scale, bias=None, want_dbias=False):
    dt = q.dtype
    grad_out, out = _dense(grad_out.to(dt)), _dense(out.to(dt))
    q, k, v = _dense(q), _dense(k), _dense(v)
    lse = logsumexp.to(torch.float32).contiguous()
    batch, sq, d = _flat(q)
    sk = int(k.shape[-2])
    bias_t, period = _bias_args(bias, batch, sq, sk)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    dbias = torch.empty(q.shape[:-1] + (sk,), dtype=torch.float32, device=q.device) if want_dbias else None
    lib = _lib.load()
    nbytes = int(lib.jg_attn_bwd_workspace_bytes(batch, sq, sk, d))
    ws = torch.empty(max(nbytes, 4), dtype=torch.uint8, device=q.device)
    rc = lib.jg_attn_bwd(
        _lib.ptr(dq), _lib.ptr(dk), _lib.ptr(dv), _lib.ptr(grad_out), _lib.ptr(q), _lib.ptr(k), _lib.ptr(v),
        _lib.ptr(out), _lib.ptr(lse), batch, sq, sk, d, float(scale), _lib.ptr(bias_t), period, _lib.ptr(dbias),
        _lib.dtype_code(dt), _lib.ptr(ws), nbytes, _lib.stream_ptr(q.device),
    )
    _lib.check(rc, "jg_attn_bwd")
    if want_dbias:
        return dq, dk, dv, dbias
    return dq, dk, dv


def backward(grad_out, q, k, v, out, logsumexp, scale, *args, dropout_p=0.0, seed=None, rng_state=None,
             layout="bhsd", **kwargs):
    """Attention core backward with the reference's signature
    (cores/math.py:81-149, cores/sdpa.py:88-165): ``(dq, dk, dv)`` in ``grad_out.dtype``."""
    if layout != "bhsd":
        raise NotImplementedError(f"the HIP core is bhsd-only; got layout={layout!r}")
    if dropout_p != 0.0:
        raise NotImplementedError("attention dropout is not supported by the HIP core")
    dq, dk, dv = core_backward(grad_out, q, k, v, out, logsumexp, scale)
    gd = grad_out.dtype
    return dq.to(gd), dk.to(gd), dv.to(gd)


# --------------------------------------------------------------------------- #
# per-rank ring loops over local chunks
# --------------------------------------------------------------------------- #
def _fused_ok(q, k) -> bool:
    """Whether one launch attends the chunk AND merges into the running accumulators: the 16-bit matrix-core
    kernels at head sizes that are multiples of 8, the fp32 one at multiples of 4 (any lengths,
    16-byte aligned tensors)."""
    d = q.shape[-1]
    if any(t.data_ptr() % 16 for t in (q, k)):
        return False
    if _as_64_columns(q, k):  # the merge is a kernel of its own then
        return False
    return d % 4 == 0 and _mfma32(q, k) if q.dtype == torch.float32 else d % 8 == 0 and _mfma16(q, k)


def attend_step_(q, kj, vj, scale, out, lse):
    """One ring step: attend chunk ``(kj, vj)`` and merge into the running fp32
    ``(out, lse)`` in place (``_attend_step``, forward.py:64-96). Uses the fused
    kernel when it covers the shape, the core + merge kernels otherwise."""
    kj, vj = kj.contiguous(), vj.contiguous()
    if (_fused_ok(q, kj) and q.is_contiguous() and vj.data_ptr() % 16 == 0 and out.dtype == torch.float32
            and out.is_contiguous() and lse.is_contiguous() and out.data_ptr() % 16 == 0):
        core_forward(q, kj, vj, scale, out_acc=out, lse_acc=lse, want_out=False)
        return out, lse
    out_j, l_j = core_forward(q, kj, vj, scale)
    fused = fused_online_softmax_merge_(out, lse, out_j, l_j, "bhsd")
    if fused is None:
        raise NotImplementedError("merge of these dtypes / layouts is not covered by the HIP kernel")
    return fused


def ring_forward(q, k_chunks: Sequence[torch.Tensor], v_chunks: Sequence[torch.Tensor], scale, rank: int = 0):
    """``(out, lse)`` of one rank's queries over all P chunks, visited in ring order
    ``(rank + step) % P`` (forward_chunk_provider.py:190-192). The accumulator is
    fp32 and cast to ``q.dtype`` once at the end (forward.py:160-167, 199). Chunks that are all
    resident here go through one launch that keeps it in registers (a step's output is then not
    rounded before it is merged, as it is step by step)."""
    P = len(k_chunks)
    order = [(rank + step) % P for step in range(P)]
    ks, vs = [k_chunks[j] for j in order], [v_chunks[j] for j in order]
    one_pass = _native("ring_forward", q, ks, vs, scale) or _resident_forward(q, ks, vs, scale)
    if one_pass is not None:
        return one_pass
    acc = torch.promote_types(q.dtype, torch.float32)
    out = torch.zeros(q.shape, device=q.device, dtype=acc)
    lse = torch.full(q.shape[:-1], float("-inf"), device=q.device, dtype=acc)
    for j in order:
        out, lse = attend_step_(q, k_chunks[j].to(q.dtype), v_chunks[j].to(q.dtype), scale, out, lse)
    return out.to(q.dtype), lse


_MAX_CHUNKS_PER_CALL = 16


def _resident(q, k_chunks, v_chunks) -> bool:
    """Whether the one-pass kernels take q against these chunks."""
    k0 = k_chunks[0]
    covered = q.shape[-1] % 4 == 0 and _mfma32(q, k0) or q.shape[-1] % 8 == 0 and _mfma16(q, k0)
    return (covered and len(k_chunks) == len(v_chunks) <= _MAX_CHUNKS_PER_CALL and q.is_cuda
            and k0.shape[:-2] == q.shape[:-2] and k0.shape[-1] == q.shape[-1]
            and all(t.shape == k0.shape and t.device == q.device for t in (*k_chunks, *v_chunks)))


def _pointers(tensors) -> ctypes.Array:
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def _chunks_as_64_columns(chunks) -> list:
    """The chunks with zero columns up to 64: three launches for all of them."""
    return list(_pad_last(torch.stack(tuple(chunks)), 64).unbind(0))


def _native(name, *args):
    """The native host module's version of a resident call (``csrc/host.cpp``): 16-bit chunks on the GPU that need no copy,
    conversion or zero columns. ``None`` for all others, and without the module."""
    host = _lib.host() if args[0].is_cuda else None
    return None if host is None else getattr(host, name)(*args, _lib.stream_handle(args[0].device))


def _resident_forward(q, k_chunks, v_chunks, scale):
    """``(out, lse)`` over resident chunks in ONE launch (``jg_attn_fwd_chunks``), ``None`` where that does not cover them."""
    if not k_chunks or not _resident(q, k_chunks, v_chunks):
        return None
    if _as_64_columns(q, k_chunks[0], len(k_chunks)):
        kv = _chunks_as_64_columns(t.to(q.dtype) for t in (*k_chunks, *v_chunks))
        out, lse = _resident_forward(_pad_last(q, 64), kv[:len(k_chunks)], kv[len(k_chunks):], scale)
        return out[..., :q.shape[-1]].contiguous(), lse
    if q.shape[-1] < 64:  # the module leaves narrow heads on long sequences to the rule above
        done = _native("ring_forward_at_own_width", q, list(k_chunks), list(v_chunks), scale)
        if done is not None:
            return done
    q = _dense(q)
    ks, vs = [_dense(t.to(q.dtype)) for t in k_chunks], [_dense(t.to(q.dtype)) for t in v_chunks]
    batch, sq, d = _flat(q)
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device=q.device)
    rc = _lib.load().jg_attn_fwd_chunks(
        _lib.ptr(out), _lib.ptr(lse), _lib.ptr(q), _pointers(ks), _pointers(vs), len(ks), batch, sq, int(ks[0].shape[-2]), d,
        float(scale), _lib.dtype_code(q.dtype), _lib.stream_ptr(q.device),
    )
    _lib.check(rc, "jg_attn_fwd_chunks")
    return out, lse


def _resident_backward(dout, q, out, lse, k_chunks, v_chunks, scale):
    """``(dq, [dk_j], [dv_j])`` over resident chunks in one pass (``jg_attn_bwd_chunks``), ``None`` where that does not
    cover them: the dQ kernel walks every chunk with dQ in its registers (one launch, one rounding), the dK/dV
    kernel takes the chunk as a grid dimension."""
    if not k_chunks or not _resident(q, k_chunks, v_chunks):
        return None
    _lib.require_gpu(dout, q, out, lse)
    if _as_64_columns(q, k_chunks[0], len(k_chunks)):
        d, P = q.shape[-1], len(k_chunks)
        kv = _chunks_as_64_columns(t.to(q.dtype) for t in (*k_chunks, *v_chunks))
        padded = [_pad_last(t.to(q.dtype), 64) for t in (dout, q, out)]
        dq, dkv = _backward_over(*padded, lse, kv[:P], kv[P:], scale)[:2]
        dk, dv = dkv[..., :d].contiguous().unbind(0)
        return dq[..., :d].contiguous(), list(dk.unbind(0)), list(dv.unbind(0))
    if q.shape[-1] < 64:  # as in the forward
        done = _native("ring_backward_at_own_width", dout, q, out, lse, list(k_chunks), list(v_chunks), scale)
        if done is not None:
            return done
    dq, _, dks, dvs = _backward_over(dout, q, out, lse, k_chunks, v_chunks, scale)
    return dq, dks, dvs


def _backward_over(dout, q, out, lse, k_chunks, v_chunks, scale):
    """``(dq, dkv, dks, dvs)`` of ``jg_attn_bwd_chunks``: ``dks``, ``dvs`` are the chunks' views of the one allocation ``dkv``."""
    dout, out, q = _dense(dout.to(q.dtype)), _dense(out.to(q.dtype)), _dense(q)
    lse = lse.to(torch.float32).contiguous()
    ks, vs = [_dense(t.to(q.dtype)) for t in k_chunks], [_dense(t.to(q.dtype)) for t in v_chunks]
    P = len(ks)
    batch, sq, d = _flat(q)
    sk = int(ks[0].shape[-2])
    dq = torch.empty_like(q)
    dkv = torch.empty((2, P) + tuple(ks[0].shape), dtype=q.dtype, device=q.device)
    dks, dvs = list(dkv[0].unbind(0)), list(dkv[1].unbind(0))
    lib = _lib.load()
    nbytes = int(lib.jg_attn_bwd_workspace_bytes(batch, sq, sk, d))
    ws = torch.empty(max(nbytes, 4), dtype=torch.uint8, device=q.device)
    rc = lib.jg_attn_bwd_chunks(
        _lib.ptr(dq), _pointers(dks), _pointers(dvs), _lib.ptr(dout), _lib.ptr(q), _pointers(ks), _pointers(vs), P,
        _lib.ptr(out), _lib.ptr(lse), batch, sq, sk, d, float(scale), _lib.dtype_code(q.dtype), _lib.ptr(ws), nbytes,
        _lib.stream_ptr(q.device),
    )
    _lib.check(rc, "jg_attn_bwd_chunks")
    return dq, dkv, dks, dvs


def backward_chunks(dout, q, out, lse, k_chunks, v_chunks, scale):
    """``(dq, [dk_j], [dv_j])`` over resident chunks in ONE pass, a hook for a caller with a loop of its own to fall back to:
    ``None`` for anything but bf16 at head size 64 with lengths that are multiples of 128 and up to 16 chunks of one
    shape, where its results have the bits of that loop's. :func:`ring_backward` and the ring's seat take every
    type, head size and length the kernels cover."""
    if not 1 <= len(k_chunks) <= _MAX_CHUNKS_PER_CALL or len(v_chunks) != len(k_chunks):
        return None
    if q.dtype != torch.bfloat16 or q.shape[-1] != 64 or q.shape[-2] % 128 or k_chunks[0].shape[-2] % 128:
        return None
    if any(t.dtype != q.dtype for t in (*k_chunks, *v_chunks)):
        return None
    return _resident_backward(dout, q, out, lse, k_chunks, v_chunks, scale)


def ring_backward(dout, q, out, lse, k_chunks, v_chunks, scale):
    """``(dq, [dk_j], [dv_j])``: this rank's contribution to every chunk's gradient.

    ``dq`` accumulates over the chunks (backward.py:184, 269; here in fp32, cast to
    ``q.dtype`` at the end — the reference accumulates in ``q.dtype``); the sum of
    dK/dV over the ranks that attended a chunk is the caller's collective. Chunks that are all
    resident go through one pass (``jg_attn_bwd_chunks``) where it covers them."""
    core = q.dtype
    one_pass = (_native("ring_backward", dout, q, out, lse, list(k_chunks), list(v_chunks), scale)
                or _resident_backward(dout, q, out, lse, k_chunks, v_chunks, scale))
    if one_pass is not None:
        return one_pass
    dout, out = dout.to(core), out.to(core)
    dq = torch.zeros(q.shape, device=q.device, dtype=torch.float32)
    dks, dvs = [], []
    for kj, vj in zip(k_chunks, v_chunks):
        dq_j, dk_j, dv_j = core_backward(dout, q, kj.to(core), vj.to(core), out, lse, scale)
        dq += dq_j
        dks.append(dk_j)
        dvs.append(dv_j)
    return dq.to(core), dks, dvs


# --------------------------------------------------------------------------- #
# windowed attention with an additive bias (Swin block)
# --------------------------------------------------------------------------- #
class _BiasedAttention(torch.autograd.Function):
    """``F.scaled_dot_product_attention(q, k, v, attn_mask=bias)`` as the Swin example
    calls it (examples/swin.py:146-151), differentiable in q, k, v and bias."""

    @staticmethod
    def forward(ctx, q, k, v, bias):  # noqa: D102
        scale = q.shape[-1] ** -0.5
        out, lse = core_forward(q, k, v, scale, bias=bias)
        ctx.save_for_backward(q, k, v, bias, out, lse)
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, grad_out):  # noqa: D102
        q, k, v, bias, out, lse = saved_rows(ctx)
        need_bias = bias is not None and ctx.needs_input_grad[3]
        res = core_backward(grad_out, q, k, v, out, lse, ctx.scale, bias=bias, want_dbias=need_bias)
        dq, dk, dv = res[:3]
        dbias = None
        if need_bias:
            # sum the per-batch-entry gradient over the entries that share a bias matrix
            sq, sk = q.shape[-2], k.shape[-2]
            period = bias.numel() // (sq * sk)
            per_entry = res[3].reshape(-1, period, sq, sk)
            dbias = (per_entry[0] if per_entry.shape[0] == 1 else per_entry.sum(0)).reshape(bias.shape).to(bias.dtype)
        return dq, dk, dv, dbias


def window_attention(q, k, v, bias=None):
    """softmax(q k^T / sqrt(d) + bias) v over the last two axes."""
    return _BiasedAttention.apply(q, k, v, bias)


SWIN_WINDOW, SWIN_HEAD_SIZE = 8, 32


def swin_grid_supported(q: torch.Tensor, grid: tuple, window: int) -> bool:
    """Whether :func:`swin_grid_attention` has a kernel for these tensors: bf16, head size 32,
    8 x 8 windows tiling the token grid."""
    return (
        q.dtype == torch.bfloat16 and q.shape[-1] == SWIN_HEAD_SIZE and window == SWIN_WINDOW
        and grid[0] % window == 0 and grid[1] % window == 0 and grid[0] * grid[1] == q.shape[-2]
    )


class _SwinGridAttention(torch.autograd.Function):
    """Attention inside the 8 x 8 windows of a token grid. ``qkv`` is (3, B, heads, gh * gw, 32), the
    tokens in grid order, as the qkv projection writes it; relative-position bias from ``table``
    (225, heads) and the shift mask from the per-token codes ``side`` (windows, 64) are formed inside
    the kernel (examples/swin.py:99-170). ``shift``: the windows lie on the grid rolled by minus this
    along both axes (the grid wraps inside this rank). Differentiable in qkv and table; the gradient comes
    back as one (3, ...) tensor, so that nothing is stacked or split on the way to the projection."""

    @staticmethod
    def forward(ctx, qkv, table, side, grid, shift=0):  # noqa: D102
        lib = _lib.load()
        qkv = qkv.contiguous()
        table = table.detach().float().contiguous()
        _, images, heads, tokens, d = qkv.shape
        gh, gw = grid
        scale = d ** -0.5
        out = torch.empty(qkv.shape[1:], dtype=qkv.dtype, device=qkv.device)
        lse = torch.empty(images * heads * tokens, dtype=torch.float32, device=qkv.device)
        q, part = qkv.data_ptr(), out.numel() * qkv.element_size()
        rc = lib.jg_attn_swin_shifted_fwd(
            _lib.ptr(out), _lib.ptr(lse), q, q + part, q + 2 * part, _lib.ptr(table),
            _lib.ptr(side), images, heads, gh, gw, shift % gh, shift % gw, d, float(scale), _lib.dtype_code(qkv.dtype),
            _lib.stream_ptr(qkv.device),
        )
        _lib.check(rc, "jg_attn_swin_shifted_fwd")
        ctx.save_for_backward(qkv, table, side, out, lse)
        ctx.grid, ctx.scale, ctx.shift = (gh, gw), scale, shift
        return out

    @staticmethod
    def backward(ctx, grad_out):  # noqa: D102
        lib = _lib.load()
        qkv, table, side, out, lse = saved_rows(ctx)
        _, images, heads, tokens, d = qkv.shape
        gh, gw = ctx.grid
        grad_out = grad_out.contiguous()
        dqkv = torch.empty_like(qkv)
        dtable = ws = None
        ws_bytes = 0
        if ctx.needs_input_grad[1]:
            dtable = torch.empty_like(table)
            ws_bytes = lib.jg_attn_swin_bwd_workspace_bytes(images, heads, gh, gw)
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=qkv.device)
        q, dq, part = qkv.data_ptr(), dqkv.data_ptr(), out.numel() * qkv.element_size()
        rc = lib.jg_attn_swin_shifted_bwd(
            dq, dq + part, dq + 2 * part, _lib.ptr(dtable), _lib.ptr(grad_out),
            q, q + part, q + 2 * part, _lib.ptr(out), _lib.ptr(lse), _lib.ptr(table),
            _lib.ptr(side), images, heads, gh, gw, ctx.shift % gh, ctx.shift % gw, d, float(ctx.scale),
            _lib.dtype_code(qkv.dtype), _lib.ptr(ws), ws_bytes, _lib.stream_ptr(qkv.device),
        )
        _lib.check(rc, "jg_attn_swin_shifted_bwd")
        return dqkv, dtable, None, None, None


def swin_grid_attention_packed(qkv, table, side, grid, shift=0):
    """:func:`swin_grid_attention` on the (3, B, heads, tokens, 32) tensor of the qkv projection; ``shift``: on
    the windows of the grid rolled by ``-shift`` along both axes, for a grid that is not split over ranks."""
    if qkv.dim() != 5 or qkv.shape[0] != 3 or not swin_grid_supported(qkv[0], grid, SWIN_WINDOW):
        raise NotImplementedError("swin_grid_attention: (3, B, heads, tokens, 32) bf16 and 8 x 8 windows only")
    if side is not None and (side.dtype != torch.uint8 or side.numel() != qkv.shape[-2]):
        raise ValueError("side must be a uint8 code per token, (windows, 64)")
    if table.shape != (225, qkv.shape[2]):
        raise ValueError(f"table must be (225, heads = {qkv.shape[2]}), got {tuple(table.shape)}")
    return _SwinGridAttention.apply(qkv, table, side, grid, int(shift))


def swin_grid_attention(q, k, v, table, side, grid):
    """Attention inside the 8 x 8 windows of a token grid for separate ``q, k, v`` of shape
    (B, heads, gh * gw, 32) (stacked here; see :func:`swin_grid_attention_packed`). ``side`` is a uint8
    tensor (windows, 64) or ``None``."""
    if not swin_grid_supported(q, grid, SWIN_WINDOW):
        raise NotImplementedError("swin_grid_attention: bf16, head size 32 and 8 x 8 windows only")
    return swin_grid_attention_packed(torch.stack((q, k, v)), table, side, grid)


__all__ = [
    "attend_step_",
    "backward",
    "backward_chunks",
    "core_backward",
    "core_forward",
    "forward",
    "fused_online_softmax_merge_",
    "ring_backward",
    "ring_forward",
    "swin_grid_attention",
    "swin_grid_attention_packed",
    "swin_grid_supported",
    "window_attention",
]
