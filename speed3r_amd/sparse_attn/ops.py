"""Torch-facing wrappers of the C-ABI entry points.

PyTorch supplies device memory and the current HIP stream; the arithmetic is done by the
hand-written gfx950 kernels behind ``include/speed3r_hip.h``.  Every function takes and
returns HIP-device tensors and raises if the library is not built -- there is no CPU or
eager fallback.

Layouts follow the reference operators: q/k/v/o are ``[B, H, L, D]`` with a contiguous last
dimension; indices are int32 ``[B, H, n_query_blocks, K]`` in block units.
"""
from __future__ import annotations

import contextlib
import ctypes
import math
import os
from typing import Optional, Tuple

import torch
from torch.utils._device import DeviceContext

from .. import _lib


_DTYPE_CODE = {torch.float32: _lib.S3R_F32, torch.bfloat16: _lib.S3R_BF16, torch.float16: _lib.S3R_F16}


def _code(t: torch.Tensor) -> int:
    try:
        return _DTYPE_CODE[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}; expected float32, bfloat16 or float16") from None


def _need_device(*ts: torch.Tensor) -> None:
    for t in ts:
        if not t.is_cuda:
            raise RuntimeError("speed3r_amd operators run on HIP device tensors only (got a CPU tensor)")


# A short call is bound by the host: a stream object and a device guard per launch were 20 of the 280 us of two views
# through the layer and 16 of the 137 us of one view through the operators.  The raw stream is asked for directly, and the
# guard is entered only where another device is current.
def _stream(t: torch.Tensor) -> int:
    return torch._C._cuda_getCurrentRawStream(t.device.index)


_HERE = contextlib.nullcontext()


def _on(device: torch.device):
    """Makes ``device`` the current one for a launch."""
    return _HERE if torch.cuda.current_device() == device.index else torch.cuda.device(device)


def _last_contig(t: torch.Tensor) -> torch.Tensor:
    return t if t.stride(-1) == 1 else t.contiguous()


def _forward_only(*ts: torch.Tensor) -> None:
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        raise RuntimeError("speed3r_amd operators are forward-only; call them under torch.no_grad()")


def pool_mean(x: torch.Tensor, block: int) -> torch.Tensor:
    """Mean over non-overlapping runs of ``block`` tokens: [B,H,N,D] -> [B,H,ceil(N/block),D].

    ``x`` may be any strided view with a contiguous last dimension (e.g. a head-major view of
    the packed qkv projection).  A ragged tail block is a mean over its valid tokens.
    """
    _need_device(x)
    _forward_only(x)
    x = _last_contig(x)
    b, h, n, d = x.shape
    nc = -(-n // block)
    y = torch.empty((b, h, nc, d), dtype=x.dtype, device=x.device)
    with _on(x.device):
        rc = _lib.lib().s3r_pool_mean(x.data_ptr(), y.data_ptr(), b, h, n, d, block,
                                      x.stride(0), x.stride(1), x.stride(2),
                                      y.stride(0), y.stride(1), y.stride(2), _code(x), _stream(x))
    _lib.check(rc, "s3r_pool_mean")
    return y


def _pool_means(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, block: int):
    """:func:`pool_mean` of q, k and v, in one launch where they share shape, type and device (the same bits)."""
    if not (q.shape == k.shape == v.shape and q.dtype == k.dtype == v.dtype and q.device == k.device == v.device):
        return pool_mean(q, block), pool_mean(k, block), pool_mean(v, block)
    _need_device(q, k, v)
    _forward_only(q, k, v)
    q, k, v = (_last_contig(t) for t in (q, k, v))
    b, h, n, d = q.shape
    y = torch.empty((3, b, h, -(-n // block), d), dtype=q.dtype, device=q.device)
    with _on(q.device):
        rc = _lib.lib().s3r_pool_means3(q.data_ptr(), k.data_ptr(), v.data_ptr(), y.data_ptr(), b, h, n, d, block, q.stride(0), q.stride(1),
                                        q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
                                        _code(q), _stream(q))
    _lib.check(rc, "s3r_pool_means3")
    return y.unbind(0)


def pool_qkv_packed(qkv: torch.Tensor, num_heads: int, block: int) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Pool the packed projection ``[B, N, 3*H*D]`` (layout ``(qkv h d)``) in one launch.

    Returns pooled q, k, v as ``[B, H, Nc, D]`` views of one ``[B, 3H, Nc, D]`` buffer.
    """
    b, n, c3 = qkv.shape
    d = c3 // (3 * num_heads)
    view = qkv.view(b, n, 3 * num_heads, d).permute(0, 2, 1, 3)  # [B, 3H, N, D], strided
    y = pool_mean(view, block)
    return y[:, :num_heads], y[:, num_heads:2 * num_heads], y[:, 2 * num_heads:]


# largest fp32 score buffer compressed_attn_topk allocates for its own use (a caller that asks for the scores gets them whole)
SCORE_BUFFER_BYTES = 1 << 30
CAUSAL_SCORE_BYTES = 8 << 30   # the causal variant's score buffer is not banded


def compressed_attn_topk(q: torch.Tensor, k: torch.Tensor, v: Optional[torch.Tensor], topk: Optional[int],
                         softmax_scale: Optional[float] = None, return_scores: bool = False,
                         return_lse: bool = False, materialize_scores: Optional[bool] = None,
                         out: Optional[torch.Tensor] = None, causal: bool = False):
    """Dense attention over pooled tokens plus, if ``topk`` is given, the top-k columns of the
    raw scores per query row.

    Returns ``(o, idx)`` with optional ``scores`` ([B,H,Lq,Lk] fp32) and ``lse`` appended when
    requested.  ``materialize_scores`` forces (True) or forbids (False) the fp32 score buffer.  By
    default the selection is fused into the attention kernel wherever the library has it (bf16/fp16,
    head_dim 64, top-k a power of two up to 32): the scores never leave the chip.  Otherwise the scores
    go through HBM (attention kernel, then the row-wise top-k kernel).

    ``v=None`` asks for the indices alone (``o`` is returned as ``None``; fused selection only).  Short lists of
    keys (``s3r_topk_in_lds``) give attention output and indices in one launch; beyond, they come from two
    different kernels, and a caller with two streams runs them side by side, see :func:`sparse_global_attention`.

    ``out``: a ``[B,H,Lq,D]`` tensor (or view, any strides on the first three dimensions, e.g. the
    ``permute(0, 2, 1, 3)`` of a ``[B,Lq,H,D]`` buffer) that receives the attention output instead of a fresh one.

    ``causal``: the reference kernel's IS_CAUSAL variant (flash_attention_topk.py:71,93), never taken by the reference
    layer: query i attends the keys j <= i and ranks the keys below ``min((i // 64 + 1) * 64, Lk)``, those above i
    with the score -inf.  Generic kernels with a full ``[B,H,Lq,Lk]`` fp32 score buffer (at most
    ``CAUSAL_SCORE_BYTES``); with ``return_scores`` the columns a row does not rank are returned as NaN.
    """
    if causal:
        assert v is not None and out is None, "causal: attention output and indices come from one call, into a fresh tensor"
        _need_device(q, k, v)
        _forward_only(q, k, v)
        q, k, v = (_last_contig(t) for t in (q, k, v))
        assert q.dtype == k.dtype == v.dtype, "q, k, v must share a dtype"
        b, h, lq, d = q.shape
        lk = k.shape[2]
        assert k.shape == (b, h, lk, d) and v.shape == (b, h, lk, d), "k/v shape mismatch"
        scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
        o = torch.empty_like(q, memory_format=torch.contiguous_format)
        idx = torch.empty((b, h, lq, topk), dtype=torch.int32, device=q.device) if topk else None
        lse = torch.empty((b, h, lq), dtype=torch.float32, device=q.device) if return_lse else None
        scores = None
        if topk or return_scores:
            if 4 * b * h * lq * lk > CAUSAL_SCORE_BYTES:
                raise RuntimeError(f"causal top-k keeps all {b}x{h}x{lq}x{lk} fp32 scores in one buffer; that exceeds "
                                   f"CAUSAL_SCORE_BYTES = {CAUSAL_SCORE_BYTES}")
            scores = torch.full((b, h, lq, lk), float("nan"), dtype=torch.float32, device=q.device) if return_scores \
                else torch.empty((b, h, lq, lk), dtype=torch.float32, device=q.device)
        st3 = lambda t: (t.stride(0), t.stride(1), t.stride(2))
        with _on(q.device):
            rc = _lib.lib().s3r_compressed_attn_topk_causal(
                q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr() if lse is not None else None,
                idx.data_ptr() if idx is not None else None, scores.data_ptr() if scores is not None else None,
                b, h, lq, lk, d, topk or 0, *st3(q), *st3(k), *st3(v), *st3(o), scale, _code(q), _stream(q))
        _lib.check(rc, "s3r_compressed_attn_topk_causal")
        res = [o, idx]
        if return_scores:
            res.append(scores)
        if return_lse:
            res.append(lse)
        return tuple(res)
    indices_only = v is None
    if indices_only:
        assert topk and not return_scores and not return_lse and materialize_scores is not True, \
            "v=None (indices only) needs top-k without a score buffer"
        v = k
        materialize_scores = False
    _need_device(q, k, v)
    _forward_only(q, k, v)
    q, k, v = (_last_contig(t) for t in (q, k, v))
    assert q.dtype == k.dtype == v.dtype, "q, k, v must share a dtype"
    b, h, lq, d = q.shape
    lk = k.shape[2]
    assert k.shape == (b, h, lk, d) and v.shape == (b, h, lk, d), "k/v shape mismatch"
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    if out is not None:
        assert not indices_only and out.shape == q.shape and out.dtype == q.dtype and out.device == q.device \
            and out.stride(-1) == 1, "out must be a [B,H,Lq,D] tensor of q's dtype and device, last dimension contiguous"
    o = None if indices_only else out if out is not None else torch.empty_like(q, memory_format=torch.contiguous_format)
    idx = torch.empty((b, h, lq, topk), dtype=torch.int32, device=q.device) if topk else None
    fused_ok = (q.dtype != torch.float32 and d == 64 and topk in (1, 2, 4, 8, 16, 32) and lk <= (1 << 21)
                and _lib.lib_has_fused_topk())
    want_scores = return_scores or (materialize_scores is True) or (
        bool(topk) and materialize_scores is None and not fused_ok)
    if materialize_scores is False and topk and not fused_ok:
        raise RuntimeError("fused top-k is not available for this dtype/shape; allow a score buffer")
    lse = torch.empty((b, h, lq), dtype=torch.float32, device=q.device) if return_lse else None
    st3 = lambda t: (t.stride(0), t.stride(1), t.stride(2))

    def launch(q_, o_, lse_, idx_, scores_, rows):
        with _on(q.device):
            rc = _lib.lib().s3r_compressed_attn_topk(
                q_.data_ptr(), k.data_ptr(), None if indices_only else v.data_ptr(), None if indices_only else o_.data_ptr(),
                lse_.data_ptr() if lse_ is not None else None,
                idx_.data_ptr() if idx_ is not None else None,
                scores_.data_ptr() if scores_ is not None else None,
                b, h, rows, lk, d, topk or 0, *st3(q_), *st3(k), *st3(v),
                *((0, 0, 0) if indices_only else st3(o_)), scale, _code(q), _stream(q))
        _lib.check(rc, "s3r_compressed_attn_topk")

    rows_per_pass = max(128, (SCORE_BUFFER_BYTES // (4 * b * h * lk)) // 128 * 128)
    if want_scores and not return_scores and lq > rows_per_pass:
        # top-k values without a fused kernel (fp32, top-k 64, ...) on many pooled tokens: the score buffer holds a
        # band of query rows at a time instead of the whole [Lq, Lk] matrix (16.9 GB at a million tokens)
        scores = torch.empty((b, h, rows_per_pass, lk), dtype=torch.float32, device=q.device)
        for r0 in range(0, lq, rows_per_pass):
            r1 = min(lq, r0 + rows_per_pass)
            idx_c = torch.empty((b, h, r1 - r0, topk), dtype=torch.int32, device=q.device) if topk else None
            lse_c = torch.empty((b, h, r1 - r0), dtype=torch.float32, device=q.device) if return_lse else None
            launch(q[:, :, r0:r1], o[:, :, r0:r1], lse_c, idx_c, scores, r1 - r0)
            if idx_c is not None:
                idx[:, :, r0:r1] = idx_c
            if lse_c is not None:
                lse[:, :, r0:r1] = lse_c
        scores = None
    else:
        scores = torch.empty((b, h, lq, lk), dtype=torch.float32, device=q.device) if want_scores else None
        launch(q, o, lse, idx, scores, lq)
    out = [o, idx]
    if return_scores:
        out.append(scores)
    if return_lse:
        out.append(lse)
    return tuple(out)


def topk_rows(scores: torch.Tensor, k: int) -> torch.Tensor:
    """Exact top-k columns of each row of an fp32 matrix ``[..., rows, cols]`` -> int32 ``[..., rows, k]``.

    Order: descending score, equal scores lowest column first, +0.0 above -0.0; if
    ``cols < k`` the trailing slots hold ``cols - 1``.
    """
    _need_device(scores)
    assert scores.dtype == torch.float32, "scores must be float32"
    scores = scores.contiguous()
    cols = scores.shape[-1]
    rows = scores.numel() // cols
    idx = torch.empty((*scores.shape[:-1], k), dtype=torch.int32, device=scores.device)
    with _on(scores.device):
        rc = _lib.lib().s3r_topk_rows(scores.data_ptr(), idx.data_ptr(), rows, cols, cols, k, _stream(scores))
    _lib.check(rc, "s3r_topk_rows")
    return idx


def _as_64_token_blocks(idx: torch.Tensor, block: int, n: int) -> torch.Tensor:
    """Index lists over blocks of 128 or 256 tokens rewritten for the 64-token kernels.

    A query block of ``r * 64`` rows is ``r`` consecutive 64-row blocks with the same list, and a listed key block is
    the run of its ``r`` 64-token blocks in order, so the rewritten tensor is ``[B,H,ceil(N/64),K*r]``: the same keys
    in the same order for every query row (entries below zero stay -1; runs reaching beyond ``N`` are cut by the
    kernels' own ``start >= N`` rule)."""
    r = block // 64
    b, h, nqb, kk = idx.shape
    sub = torch.arange(r, device=idx.device, dtype=torch.int32)
    fine = torch.where(idx[..., None] >= 0, idx[..., None] * r + sub, idx.new_full((), -1))
    return fine.reshape(b, h, nqb, kk * r).repeat_interleave(r, dim=2)[:, :, :-(-n // 64)].contiguous()


def select_attn(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, idx: torch.Tensor, block: int,
                softmax_scale: Optional[float] = None, return_lse: bool = False):
    """Attention of each ``block``-row query block over the key blocks listed in ``idx``."""
    _need_device(q, k, v, idx)
    _forward_only(q, k, v)
    q, k, v, idx = (_last_contig(t) for t in (q, k, v, idx))
    assert q.dtype == k.dtype == v.dtype, "q, k, v must share a dtype"
    assert idx.dtype == torch.int32, "topk_idx must be int32"
    b, h, n, d = q.shape
    assert k.shape == q.shape and v.shape == q.shape, "q, k, v must share a shape"
    nqb = -(-n // block)
    assert idx.shape[:3] == (b, h, nqb), f"topk_idx shape {tuple(idx.shape)} does not match {(b, h, nqb, 'K')}"
    if block in (128, 256):
        idx, block = _as_64_token_blocks(idx, block, n), 64
    kk = idx.shape[3]
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    o = torch.empty_like(q, memory_format=torch.contiguous_format)
    lse = torch.empty((b, h, n), dtype=torch.float32, device=q.device) if return_lse else None
    with _on(q.device):
        rc = _lib.lib().s3r_select_attn(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr(), o.data_ptr(),
            lse.data_ptr() if lse is not None else None,
            b, h, n, d, block, kk,
            q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
            v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(1), o.stride(2),
            idx.stride(0), idx.stride(1), idx.stride(2), scale, _code(q), _stream(q))
    _lib.check(rc, "s3r_select_attn")
    return (o, lse) if return_lse else o


def gated_merge(o_cmp: torch.Tensor, o_sel: torch.Tensor, gate: torch.Tensor, block: int) -> torch.Tensor:
    """``out[b,n,h*D+d] = gate[b,h,n,0]*o_cmp[b,h,n//block,d] + gate[b,h,n,1]*o_sel[b,h,n,d]`` -> [B,N,H*D].

    ``gate`` is ``[B,H,N,2]`` in any strided form with a contiguous pair (the reference's
    ``'b n (h g) -> b h n g'`` view of the gate projection qualifies).
    """
    _need_device(o_cmp, o_sel, gate)
    _forward_only(o_cmp, o_sel, gate)
    o_cmp, o_sel, gate = (_last_contig(t) for t in (o_cmp, o_sel, gate))
    assert o_cmp.dtype == o_sel.dtype == gate.dtype, "o_cmp, o_sel, gate must share a dtype"
    b, h, n, d = o_sel.shape
    nc = -(-n // block)
    assert o_cmp.shape == (b, h, nc, d), f"o_cmp shape {tuple(o_cmp.shape)} != {(b, h, nc, d)}"
    assert gate.shape == (b, h, n, 2), f"gate shape {tuple(gate.shape)} != {(b, h, n, 2)}"
    out = torch.empty((b, n, h * d), dtype=o_sel.dtype, device=o_sel.device)
    with _on(o_sel.device):
        rc = _lib.lib().s3r_gated_merge(
            o_cmp.data_ptr(), o_sel.data_ptr(), gate.data_ptr(), out.data_ptr(), b, h, n, d, block,
            o_cmp.stride(0), o_cmp.stride(1), o_cmp.stride(2), o_sel.stride(0), o_sel.stride(1), o_sel.stride(2),
            gate.stride(0), gate.stride(1), gate.stride(2), _code(o_sel), _stream(o_sel))
    _lib.check(rc, "s3r_gated_merge")
    return out


def norm_rope(x: torch.Tensor, positions: Optional[torch.Tensor], cos_tab: Optional[torch.Tensor],
              sin_tab: Optional[torch.Tensor], ln_weight: Optional[torch.Tensor] = None,
              ln_bias: Optional[torch.Tensor] = None, eps: float = 1e-5) -> Optional[torch.Tensor]:
    """``RoPE2D(LayerNorm(x), positions)`` for one ``[B,H,N,64]`` tensor in one pass -> contiguous ``[B,H,N,64]``.

    ``positions``: integer ``[B,N,2]`` (or None: no rotation); ``cos_tab``/``sin_tab``: ``[P,16]`` tables in x's dtype
    (``RoPE2D.tables``); ``ln_weight``/``ln_bias``: LayerNorm(64) parameters (None: no normalisation).
    Returns None when the library has no kernel for the shape (head_dim other than 64)."""
    _need_device(x)
    _forward_only(x)
    x = _last_contig(x)
    b, h, n, d = x.shape
    if d != 64:
        return None
    pos32 = None
    p = 0
    if positions is not None:
        assert positions.shape == (b, n, 2), f"positions shape {tuple(positions.shape)} != {(b, n, 2)}"
        assert cos_tab is not None and sin_tab is not None and cos_tab.shape == sin_tab.shape and cos_tab.shape[1] == 16
        assert cos_tab.dtype == x.dtype and sin_tab.dtype == x.dtype, "tables must have x's dtype"
        pos32 = positions.to(device=x.device, dtype=torch.int32).contiguous()
        cos_tab, sin_tab = cos_tab.contiguous(), sin_tab.contiguous()
        p = cos_tab.shape[0]
    w = ln_weight.detach().to(x.dtype).contiguous() if ln_weight is not None else None
    bias = ln_bias.detach().to(x.dtype).contiguous() if (ln_bias is not None and w is not None) else None
    y = torch.empty((b, h, n, d), dtype=x.dtype, device=x.device)
    with _on(x.device):
        rc = _lib.lib().s3r_norm_rope(
            x.data_ptr(), y.data_ptr(), pos32.data_ptr() if pos32 is not None else None,
            cos_tab.data_ptr() if pos32 is not None else None, sin_tab.data_ptr() if pos32 is not None else None, p,
            w.data_ptr() if w is not None else None, bias.data_ptr() if bias is not None else None, float(eps),
            b, h, n, d, x.stride(0), x.stride(1), x.stride(2),
            pos32.stride(0) if pos32 is not None else 0, pos32.stride(1) if pos32 is not None else 0,
            _code(x), _stream(x))
    _lib.check(rc, "s3r_norm_rope")
    return y


def prepass_takes(qkv: torch.Tensor, num_heads: int) -> bool:
    """Whether the passes over the packed projection are built for it: heads of 64, rows of adjacent values that do not overlap."""
    return qkv.shape[-1] == 192 * num_heads and qkv.stride(-1) == 1 and qkv.stride(1) >= qkv.shape[-1]


def _prepass_args(qkv: torch.Tensor, h: int, block: int, positions, cos_tab, sin_tab, q_ln, k_ln, eps: float, inv_freq=None, signed=False):
    """Argument block of the passes over the packed projection, with its inputs filled in, and the tensors it points to."""
    b, n = qkv.shape[:2]
    es = qkv.element_size()
    base = qkv.data_ptr()
    a = _lib.PrepassArgs(q=base, k=base + h * 64 * es, v=base + 2 * h * 64 * es, N=n, stride_b=qkv.stride(0), stride_h=64,
                         stride_n=qkv.stride(1), B=b, H=h, head_dim=64, block=block, eps=eps, dtype=_code(qkv))
    keep = []
    if positions is not None:
        assert positions.shape == (b, n, 2), f"positions shape {tuple(positions.shape)} != {(b, n, 2)}"
        assert cos_tab is not None and sin_tab is not None and cos_tab.shape == sin_tab.shape and cos_tab.shape[1] == 16
        assert cos_tab.dtype == qkv.dtype and sin_tab.dtype == qkv.dtype, "tables must have the tokens' dtype"
        if positions.dtype not in (torch.int64, torch.int32) or positions.device != qkv.device or positions.stride(2) != 1:
            positions = positions.to(device=qkv.device, dtype=torch.int32).contiguous()
        cos_tab, sin_tab = cos_tab.contiguous(), sin_tab.contiguous()
        keep += [positions, cos_tab, sin_tab]
        a.positions, a.positions_int64 = positions.data_ptr(), positions.dtype == torch.int64
        a.pos_stride_b, a.pos_stride_n = positions.stride(0), positions.stride(1)
        a.cos_table, a.sin_table, a.table_rows = cos_tab.data_ptr(), sin_tab.data_ptr(), cos_tab.shape[0]
        if inv_freq is not None:
            a.inv_freq, a.signed_positions = inv_freq.data_ptr(), signed
    if q_ln is not None:
        params = [*q_ln, *k_ln]
        # fp32 parameters of 16-bit tokens (autocast) are used as they are, any others in the tokens' dtype
        as_fp32 = all(t is None or t.dtype == torch.float32 for t in params)
        dtype = torch.float32 if as_fp32 else qkv.dtype
        params = [t.detach().to(dtype).contiguous() if t is not None else None for t in params]
        keep += params
        a.norm_fp32 = as_fp32
        a.q_norm_weight, a.q_norm_bias, a.k_norm_weight, a.k_norm_bias = (t.data_ptr() if t is not None else None for t in params)
    return a, keep


def qkv_prepass(qkv: torch.Tensor, num_heads: int, block: int, positions: Optional[torch.Tensor],
                cos_tab: Optional[torch.Tensor], sin_tab: Optional[torch.Tensor],
                q_ln: Optional[Tuple[torch.Tensor, Optional[torch.Tensor]]] = None,
                k_ln: Optional[Tuple[torch.Tensor, Optional[torch.Tensor]]] = None, eps: float = 1e-5, *,
                tokens: bool = True, pooled: Optional[str] = "raw", keep_raw: bool = False, inv_freq: Optional[torch.Tensor] = None,
                signed: bool = False):
    """The layer's pre-pass over the packed projection ``[B, N, 3*H*64]`` (layout ``(qkv h d)``) in one kernel:
    returns ``(q, k, v, q_c, k_c, v_c)`` -- q, k ``[B,H,N,64]`` contiguous after LayerNorm (``q_ln``/``k_ln`` = (weight,
    bias) or None) and RoPE2D at ``positions`` (None: no rotation), v the strided view of the projection, and the
    block means of the RAW q, k, v ``[B,H,ceil(N/block),64]``.  Same bits as :func:`pool_qkv_packed` followed by
    :func:`norm_rope` on q and k.  Returns None where the library has no kernel for it (:func:`prepass_takes`).

    ``pooled="final"``: q_c and k_c are normalised and rotated too, at the truncated mean position of their block
    (:func:`norm_rope` at ``block_positions``); ``keep_raw`` then appends their raw values to the result.
    ``pooled=None``: q, k, v only; ``tokens=False``: the block means only.  ``inv_freq`` ([16] fp32): positions beyond the
    tables are rotated by their own angles instead of being clamped to the last row, with ``signed`` those below zero too
    (else: row 0)."""
    _need_device(qkv)
    _forward_only(qkv)
    b, n = qkv.shape[:2]
    h = num_heads
    if not prepass_takes(qkv, h):
        return None
    assert (q_ln is None) == (k_ln is None), "q and k are normalised together or not at all"
    assert pooled in ("raw", "final", None) and (tokens or pooled)
    a, keep = _prepass_args(qkv, h, block, positions, cos_tab, sin_tab, q_ln, k_ln, float(eps), inv_freq, signed)
    out = ()
    if tokens:
        q_out, k_out = qkv.new_empty((2, b, h, n, 64)).unbind(0)
        a.q_out, a.k_out = q_out.data_ptr(), k_out.data_ptr()
        out = (q_out, k_out, qkv.as_strided((b, h, n, 64), (qkv.stride(0), 64, qkv.stride(1), 1), qkv.storage_offset() + 2 * h * 64))
    if pooled:
        means = qkv.new_empty((5 if keep_raw else 3, b, h, -(-n // block), 64)).unbind(0)
        a.q_pool, a.k_pool, a.v_pool = (t.data_ptr() for t in means[:3])
        a.finish_pooled = pooled == "final"
        if keep_raw:
            a.q_raw, a.k_raw = means[3].data_ptr(), means[4].data_ptr()
        out += means
    with _on(qkv.device):
        rc = _lib.lib().s3r_layer_prepass(ctypes.byref(a), _stream(qkv))
    _lib.check(rc, "s3r_layer_prepass")
    return out


def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float) -> Optional[torch.Tensor]:
    """``F.layer_norm(x, (C,), weight, bias, eps)`` over the last dimension of token rows in one pass (inference).

    Returns None when the library has no kernel for the shape (rows that are not a multiple of 16 bytes or longer
    than 512 16-byte chunks, a tensor whose leading dimensions do not collapse to one row stride)."""
    _need_device(x)
    _forward_only(x)
    c = x.shape[-1]
    vec = 16 // x.element_size()
    if x.dtype not in (torch.bfloat16, torch.float16, torch.float32) or c % vec or c // vec > 512 or x.numel() == 0:
        return None
    x2 = x.reshape(-1, c) if x.is_contiguous() else None
    if x2 is None:
        return None
    w = weight.detach().to(x.dtype).contiguous()
    b = bias.detach().to(x.dtype).contiguous() if bias is not None else None
    y = torch.empty_like(x2)
    with _on(x.device):
        rc = _lib.lib().s3r_layer_norm(x2.data_ptr(), y.data_ptr(), w.data_ptr(), b.data_ptr() if b is not None else None,
                                       float(eps), x2.shape[0], c, x2.stride(0), y.stride(0), _code(x), _stream(x))
    _lib.check(rc, "s3r_layer_norm")
    return y.view(x.shape)


def add_layer_norm(x: torch.Tensor, a: torch.Tensor, gamma: Optional[torch.Tensor], weight: torch.Tensor, bias: Optional[torch.Tensor],
                   eps: float) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """``(s, layer_norm(s))`` of ``s = x + gamma * a`` (``gamma=None``: ``x + a``) in one pass (inference); the bits of the sum
    followed by :func:`layer_norm`.  Returns None where that has no kernel, or where the tensors' types or forms differ."""
    _need_device(x)
    _forward_only(x, a)
    c = x.shape[-1]
    vec = 16 // x.element_size()
    if x.dtype not in (torch.bfloat16, torch.float16, torch.float32) or c % vec or c // vec > 512 or x.numel() == 0:
        return None
    params = [t for t in (gamma, weight, bias) if t is not None]
    if x.shape != a.shape or any(t.shape != (c,) or not t.is_contiguous() for t in params) or not (x.is_contiguous() and a.is_contiguous()):
        return None
    if any(t.dtype != x.dtype or t.device != x.device or t.data_ptr() % 16 for t in (x, a, *params)):
        return None
    s, y = torch.empty_like(x), torch.empty_like(x)
    with _on(x.device):
        rc = _lib.lib().s3r_add_layer_norm(x.data_ptr(), a.data_ptr(), gamma.data_ptr() if gamma is not None else None, s.data_ptr(),
                                           y.data_ptr(), weight.data_ptr(), bias.data_ptr() if bias is not None else None,
                                           float(eps), x.numel() // c, c, _code(x), _stream(x))
    _lib.check(rc, "s3r_add_layer_norm")
    return s, y


# Where the layers leave a product to the library (us on the device, library / kernel).  Inputs of 1024 and fewer: nowhere; few rows are no
# faster here on the device (256 x 1024 x 1024 5.5 / 8.7, 1 041 9.0 / 9.2, 2 016 10.4 / 9.7) but on the host, which they wait for.  More
# inputs: the library splits them where tiles are few (2 016 x 1024 x 4096 26 / 39) and reaches 1.4 to 1.5 PFLOP/s where they are many
# (32 256 x 2048 x 8192 705 / 795, 16 128 x 1536 x 6144 230 / 244, 8 064 x 3072 x 12288 435 / 528, 8 064 x 4608 x 1536 97 / 101), except
# where one round of 128-wide tiles, two per CU, is full (8 064 x 1024 x 4096 58 / 55, 6 000 x 1280 x 5120 69 / 67, 4 032 x 2048 x 2048 33 / 30);
# with GELU in the epilogue there is a pass less (8 064 x 5120 x 1280 145 / 107, 2 016 x 8192 x 2048 73 / 57, 400 x 12288 x 3072 45 / 39).
def linear_pays(rows: int, n: int, k: int, gelu: bool = False) -> bool:
    if k <= 1024:
        return True
    tiles = -(-rows // 128) * -(-n // 128)
    return tiles >= 256 if gelu else 400 < tiles <= 512


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], gelu: bool = False) -> Optional[torch.Tensor]:
    """``F.linear(x, weight, bias)``, with ``gelu`` followed by ``F.gelu``, in one kernel (inference).

    Returns None where the library has no kernel (bf16/fp16, inputs a multiple of 128, outputs of 8, 16-byte aligned tensors
    of one dtype with adjacent values and rows of one stride)."""
    _need_device(x)
    _forward_only(x, weight)
    k, n = x.shape[-1], weight.shape[0]
    if x.dtype not in (torch.bfloat16, torch.float16) or k % 128 or n % 8 or x.numel() == 0 or weight.shape != (n, k) or k > 1 << 20 or n > 1 << 20 \
            or (bias is not None and bias.shape != (n,)):
        return None
    for t in (x, weight, bias):
        if t is not None and (t.dtype != x.dtype or t.device != x.device or not t.is_contiguous() or t.data_ptr() % 16):
            return None
    out = x.new_empty((*x.shape[:-1], n))
    with _on(x.device):
        rc = _lib.lib().s3r_linear(x.data_ptr(), weight.data_ptr(), bias.data_ptr() if bias is not None else None, out.data_ptr(),
                                   x.numel() // k, n, k, k, k, n, 1 if gelu else 0, _code(x), _stream(x))
    _lib.check(rc, "s3r_linear")
    return out


def unchanged_here(x: torch.Tensor) -> bool:
    """Whether a call on ``x`` is seen by nobody but torch itself: a tensor on the GPU, without a transform (vmap, forward-mode
    derivatives) or a mode (``make_fx``, flop counters, selective checkpointing, function modes) that has to see the torch
    operations; ``torch.device`` as a context and the default device concern factory functions only."""
    c = torch._C
    return x.is_cuda and c._len_torch_dispatch_stack() == 0 and c._functorch.peek_interpreter_stack() is None \
        and c._has_storage(x) and torch.autograd.forward_ad._current_level < 0 \
        and (c._len_torch_function_stack() == 0
             or all(type(c._get_function_stack_at(i)) is DeviceContext for i in range(c._len_torch_function_stack())))


def ordinary(x: torch.Tensor) -> bool:
    """Whether a call on ``x`` is an ordinary one: :func:`unchanged_here`, and neither traced nor compiled."""
    return type(x) is torch.Tensor and unchanged_here(x) and not torch.jit.is_tracing() and not torch.compiler.is_compiling()


# Gradients of weight and bias, kernel / library, us on the device: 2 048 rows x 3072 x 1024 36 / 44, x 1024 x 1024 30 / 30 (no
# faster with their launches), 4 096 rows 42 / 64 and 32 / 50, 24 000 rows 125 / 262 and 61 / 185.
def linear_wgrad_pays(rows: int) -> bool:
    return rows >= 4096


def linear_wgrad_takes(n: int, c: int) -> bool:
    """Whether the kernel is built for ``n`` outputs and ``c`` inputs."""
    return n % 8 == 0 and c % 8 == 0 and 0 < n <= 1 << 20 and 0 < c <= 1 << 20


class _LinearFn(torch.autograd.Function):
    """``F.linear`` whose parameters' gradients come from :func:`linear_wgrad`; keeps what ``F.linear`` keeps."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x if ctx.needs_input_grad[1] else None, weight if ctx.needs_input_grad[0] else None)
        # The product alone, us on the device, library / kernel: 1024 inputs, 3 072 outputs, 8 104 rows 49.8 / 44.1, 24 192 129 / 127, 33 345 213 / 172, 50 016
        # 301 / 251; 4 096: 8 104 54 / 57, 10 240 95 / 78, 24 192 182 / 159; 2 048: 6 096 27.3 / 28.3, 12 192 51.5 / 47.8, 24 192 91 / 80; 1 024: 8 192 21.9 /
        # 18.1, 9 760 24.0 / 25.8, 24 192 45.9 / 47.2, 33 345 63.9 / 69.7, 41 008 95.3 / 79.6, 80 000 150 / 130; the gate's 32: 24 192 21.7 / 15.1.  Where the
        # library is the faster one alone, a whole step is not with it: a layer's output projection of 16 128 to 33 312 rows by the library / here, 24 192 rows
        # under autocast 1 645 / 1 647, 16 128 without 1 121 / 1 115, 22 settings 0.02 % apart on average.
        out = None
        if ordinary(x) and x.numel() != 0 and weight.dim() == 2 and linear_pays(x.numel() // x.shape[-1], *weight.shape):
            out = linear(x, weight, bias)
        if out is None:
            out = torch.nn.functional.linear(x, weight, bias)
        # (of a batch it is a view of the product's rows: views that are made in here may not be changed in place)
        return torch.ops.aten._unsafe_view(out, out.shape) if out._is_view() else out

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        dx = dw = db = None
        dy2 = dy.reshape(-1, dy.shape[-1])
        if ctx.needs_input_grad[0]:
            dx = (dy2 @ weight).view(*dy.shape[:-1], weight.shape[1])
        if ctx.needs_input_grad[1] and not torch.is_grad_enabled() and ordinary(dy):   # (a derivative of the backward itself: torch's)
            want_db = ctx.needs_input_grad[2]
            inside = want_db and x.shape[-1] > 768   # (the kernel sums dy beside enough inputs only)
            got = linear_wgrad(dy2, x.reshape(-1, x.shape[-1]), inside)
            if got is not None:
                return dx, got[0], dy2.sum(0) if want_db and not inside else got[1]
        if ctx.needs_input_grad[1]:
            dw = dy2.t() @ x.reshape(-1, x.shape[-1])
        if ctx.needs_input_grad[2]:
            db = dy2.sum(0)
        return dx, dw, db


def _cast(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """``t`` as autocast hands it to a product: the copy that it keeps for a leaf in this region, else a new one.  (Autocast casts
    the operands of einsum too; of one operand in its own order einsum makes a view.)"""
    if t is None or t.dtype == torch.get_autocast_dtype("cuda"):
        return t
    return torch.einsum("...i->...i", t) if t.is_leaf and t.requires_grad else t.to(torch.get_autocast_dtype("cuda"))


def autocast_once(x: torch.Tensor) -> torch.Tensor:
    """``x`` as autocast hands it to several products: one copy in its dtype where it keeps the copy (of a leaf that wants a
    gradient) or no gradient tells one copy from several."""
    if torch.is_autocast_enabled("cuda") and x.dtype == torch.float32 and (
            not x.requires_grad or (x.is_leaf and not x._is_view() and torch.is_autocast_cache_enabled())):
        return _cast(x)
    return x


def linear_autograd(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """``F.linear(x, weight, bias)`` with autocast's casts, differentiable, with the parameters' gradients from one kernel."""
    if torch.is_autocast_enabled("cuda"):
        x, weight, bias = _cast(x), _cast(weight), _cast(bias)
    return _LinearFn.apply(x, weight, bias)


def linear_wgrad(dy: torch.Tensor, x: torch.Tensor, bias: bool):
    """``(dy^T x, dy.sum(0) or None)`` of dy ``[M,N]`` and x ``[M,C]``: gradients of a linear layer's parameters, summed in fp32.

    Returns None where the library has no kernel (bf16/fp16, N and C multiples of 8, with the bias C > 768, rows of
    adjacent values, 16-byte aligned)."""
    (m, n), c = dy.shape, x.shape[1]
    if dy.dtype not in (torch.bfloat16, torch.float16) or x.dtype != dy.dtype or x.device != dy.device or x.shape[0] != m or m == 0 \
            or not linear_wgrad_takes(n, c) or (bias and c <= 768):
        return None
    for t in (dy, x):
        if t.stride(1) != 1 or t.stride(0) % 8 or not t.shape[1] <= t.stride(0) < 1 << 21 or t.data_ptr() % 16:
            return None
    ld = max(dy.stride(0), x.stride(0))
    if m > 64 * (0x7f000000 // (2 * ld) - 128):
        return None
    dw, db = dy.new_empty((n, c)), dy.new_empty((n,)) if bias else None
    with _on(dy.device):
        lib = _lib.lib()
        ws = torch.empty((lib.s3r_linear_wgrad_workspace(m, n, c, dy.stride(0), x.stride(0)),), dtype=torch.float32, device=dy.device)
        rc = lib.s3r_linear_wgrad(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr() if bias else None, ws.data_ptr(), m, n, c,
                                  dy.stride(0), x.stride(0), _code(dy), _stream(dy))
    _lib.check(rc, "s3r_linear_wgrad")
    return dw, db


def qkv_project_takes(x: torch.Tensor, num_heads: int, block: int, pooled: bool, norms: bool) -> bool:
    """Whether the library has a kernel for :func:`qkv_project` of these tokens (``norms``: with them)."""
    b, n, c = x.shape
    return x.dtype in (torch.bfloat16, torch.float16) and c == 64 * num_heads and num_heads % 2 == 0 and 0 < c <= 1 << 18 and 0 < b * n <= 1 << 30 \
        and x.is_contiguous() and (not pooled or (norms and block in (16, 64))) \
        and (b == 1 or (n >= 256 and num_heads * n * 128 <= 0x70000000 and not (pooled and n % block)))


def qkv_project(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], num_heads: int, block: int, positions: torch.Tensor,
                cos_tab: torch.Tensor, sin_tab: torch.Tensor, q_ln=None, k_ln=None, eps: float = 1e-5, *, pooled: bool,
                inv_freq: Optional[torch.Tensor] = None, gate: Optional[Tuple[torch.Tensor, Optional[torch.Tensor]]] = None, takes: Optional[bool] = None):
    """:func:`linear` with the weights of the packed projection and :func:`qkv_prepass` of its result (``pooled``: with
    ``pooled="final"``, else without means) in one kernel: ``(q, k, v[, q_c, k_c, v_c][, gates])``, all contiguous.  The projection
    is rounded, then once at the end (the pass rounds after the norm and inside the rotation too).  ``gate``: (weight, bias) of
    :func:`gate`, whose result ``[B,N,O]`` is then the last one, or None where its outputs are not a multiple of 4 up to 32 or
    the kernel has no idle time for it.  ``takes``: what :func:`qkv_project_takes` says, where the caller has asked.

    Returns None where the library has no kernel (:func:`qkv_project_takes`): bf16/fp16, head_dim 64, an even number of heads, contiguous 16-byte
    aligned tensors of one dtype; means with norms and over blocks of 16 or 64 tokens only; several sequences of 256 tokens or
    more each, with means a multiple of the block."""
    _need_device(x)
    _forward_only(x, weight)
    b, n, c = x.shape
    h = num_heads
    if takes is None:
        takes = qkv_project_takes(x, h, block, pooled, q_ln is not None)
    if not takes or weight.shape != (3 * c, c) or (bias is not None and bias.shape != (3 * c,)):
        return None
    for t in (x, weight, bias):
        if t is not None and (t.dtype != x.dtype or t.device != x.device or not t.is_contiguous() or t.data_ptr() % 16):
            return None
    a, keep = _prepass_args(x, h, block, positions, cos_tab, sin_tab, q_ln, k_ln, float(eps), inv_freq)
    q, k, v = x.new_empty((3, b, h, n, 64)).unbind(0)
    a.q_out, a.k_out = q.data_ptr(), k.data_ptr()
    means = ()
    if pooled:
        means = x.new_empty((3, b, h, -(-n // block), 64)).unbind(0)
        a.q_pool, a.k_pool, a.v_pool = (t.data_ptr() for t in means)
        a.finish_pooled = True
    gates, gate_args = (), (None, None, None, 0)
    if gate is not None:
        gw, gb = gate
        gts = [t for t in gate if t is not None]
        rides = _lib.lib().s3r_qkv_project_gate_rides(b * n, h) and gw.shape[0] % 4 == 0 and gw.shape[0] <= 32 and gw.shape[1:] == (c,) \
            and (gb is None or gb.shape == gw.shape[:1]) \
            and all(t.dtype == x.dtype and t.device == x.device and t.is_contiguous() for t in gts) and gw.data_ptr() % 16 == 0
        gates = (x.new_empty((b, n, gw.shape[0])) if rides else None,)
        if rides:
            gate_args = (gw.data_ptr(), gb.data_ptr() if gb is not None else None, gates[0].data_ptr(), gw.shape[0])
    with _on(x.device):
        rc = _lib.lib().s3r_qkv_project(x.data_ptr(), weight.data_ptr(), bias.data_ptr() if bias is not None else None, c, c, v.data_ptr(),
                                        ctypes.byref(a), *gate_args, _stream(x))
    _lib.check(rc, "s3r_qkv_project")
    return (q, k, v, *means, *gates)


def attention_layer(x: torch.Tensor, qkv, gate, proj, num_heads: int, block: int, topk: int, positions: torch.Tensor, cos_tab: torch.Tensor,
                    sin_tab: torch.Tensor, q_ln, k_ln, eps: float, inv_freq: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """The layer's inference in one call of the library: :func:`qkv_project` with means and the gate, :func:`compressed_attn_topk`,
    :func:`gate` where it does not ride, :func:`select_attn_merge` and, unless ``proj`` is None, :func:`linear`: the same kernels in the
    same order, the same results.  ``qkv``, ``gate``, ``proj``: (weight, bias).  For tokens that :func:`qkv_project_takes` (with means and
    norms), on the calling stream alone (not where :func:`_side_stream_pays`, unless two waves of the index kernel share a row's keys:
    at most 512 workgroups of 64 pooled rows.  These leave no LDS for a kernel beside them: 16 heads, us, two streams / this: 2 016
    blocks of 16 tokens 618 / 585, 1 260 387 / 379; 1 627 of 64 1 539 / 1 537, 1 302 1 220 / 1 224; beyond, 4 164 4 295 / 4 360, 6 489 of
    16 2 368 / 2 415).

    Returns None where the library has no kernels: top-k a power of two up to 32, contiguous 16-byte aligned weights of one dtype,
    a gate of 2 outputs per head that one of its kernels takes."""
    b, n, c = x.shape
    h = num_heads
    blocks = -(-n // block)
    if topk not in (1, 2, 4, 8, 16, 32) or (b * h * -(-blocks // 64) > 512 and _side_stream_pays(b * h, blocks, topk)):
        return None
    dtype, device = x.dtype, x.device
    for lin, rows in ((qkv, 3 * c), (gate, 2 * h), (proj, c)):
        if lin is None:
            continue
        w, bias = lin
        if w.shape != (rows, c) or w.dtype != dtype or w.device != device or not w.is_contiguous() or w.data_ptr() % 16:
            return None
        if bias is not None and (bias.shape != (rows,) or bias.dtype != dtype or bias.device != device or not bias.is_contiguous()
                                 or bias.data_ptr() % 16):
            return None
    if x.data_ptr() % 16 or c % 256 or c > 1024:
        return None
    a, keep = _prepass_args(x, h, block, positions, cos_tab, sin_tab, q_ln, k_ln, float(eps), inv_freq)
    lib = _lib.lib()
    out = torch.empty_like(x)
    size = lib.s3r_attention_layer_workspace(b, h, n, block, topk, proj is not None)
    with _on(device):
        ws = torch.empty((size,), dtype=torch.uint8, device=device)
        rc = lib.s3r_attention_layer(x.data_ptr(), *(t.data_ptr() if t is not None else None for t in (*qkv, *gate, *(proj or (None, None)))),
                                     out.data_ptr(), ws.data_ptr(), size, ctypes.byref(a), topk, 0.125, _stream(x))
    _lib.check(rc, "s3r_attention_layer")
    return out


def gate(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """``sigmoid(F.linear(x, weight, bias))`` for the few outputs of the layer's gate, in one pass over ``x`` (inference).

    Returns None where the library has no kernel (bf16/fp16, channels a multiple of 256 up to 1024, an even number of
    outputs up to 32, contiguous 16-byte aligned tensors of one dtype)."""
    _need_device(x)
    _forward_only(x, weight)
    c, o = x.shape[-1], weight.shape[0]
    ts = [t for t in (x, weight, bias) if t is not None]
    if x.dtype not in (torch.bfloat16, torch.float16) or c % 256 or c > 1024 or o > 32 or o % 2 or x.numel() == 0 or weight.shape != (o, c) \
            or (bias is not None and bias.shape != (o,)):
        return None
    if any(t.dtype != x.dtype or t.device != x.device or not t.is_contiguous() or t.data_ptr() % 16 for t in ts):
        return None
    out = x.new_empty((*x.shape[:-1], o))
    with _on(x.device):
        rc = _lib.lib().s3r_gate(x.data_ptr(), weight.data_ptr(), bias.data_ptr() if bias is not None else None, out.data_ptr(),
                                 x.numel() // c, c, o, _code(x), _stream(x))
    _lib.check(rc, "s3r_gate")
    return out


def select_attn_merge(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, idx: torch.Tensor, o_cmp: torch.Tensor,
                      gate: torch.Tensor, block: int, softmax_scale: Optional[float] = None) -> Optional[torch.Tensor]:
    """``select_attn`` with ``gated_merge`` in its epilogue -> ``[B,N,H*D]``, without the round trip of the selection output
    through memory: the bits of the two calls for 16-token blocks; for 64-token blocks (and 128, 256) the expression is evaluated
    in fp32 and rounded once.  Returns ``None`` when the library has no fused kernel for the shape (the caller then runs the two
    operators), and for fp32, which it has always left to them: programs and tests rely on that answer, and the bits are the
    same (the whole path and the layer, which run either way themselves, use the kernel's fp32 merge)."""
    return _select_attn_merge(q, k, v, idx, o_cmp, gate, block, softmax_scale, (torch.bfloat16, torch.float16))


def _select_attn_merge(q, k, v, idx, o_cmp, gate, block, softmax_scale=None, dtypes=(torch.bfloat16, torch.float16, torch.float32)):
    """:func:`select_attn_merge` in fp32 too (the bits of the two operators), for this package's own paths."""
    _need_device(q, k, v, idx, o_cmp, gate)
    _forward_only(q, k, v, o_cmp, gate)
    q, k, v, idx, o_cmp, gate = (_last_contig(t) for t in (q, k, v, idx, o_cmp, gate))
    assert q.dtype == k.dtype == v.dtype == o_cmp.dtype == gate.dtype, "q, k, v, o_cmp, gate must share a dtype"
    assert idx.dtype == torch.int32, "topk_idx must be int32"
    b, h, n, d = q.shape
    assert k.shape == q.shape and v.shape == q.shape, "q, k, v must share a shape"
    nqb = -(-n // block)
    assert idx.shape[:3] == (b, h, nqb), f"topk_idx shape {tuple(idx.shape)} does not match {(b, h, nqb, 'K')}"
    assert o_cmp.shape == (b, h, nqb, d), f"o_cmp shape {tuple(o_cmp.shape)} != {(b, h, nqb, d)}"
    assert gate.shape == (b, h, n, 2), f"gate shape {tuple(gate.shape)} != {(b, h, n, 2)}"
    if block in (128, 256):  # 64-row query blocks share their parent's list and its row of the compressed output
        o_cmp = o_cmp.repeat_interleave(block // 64, dim=2)[:, :, :-(-n // 64)].contiguous()
        idx, block = _as_64_token_blocks(idx, block, n), 64
    if q.dtype not in dtypes or d != 64 or block not in ((64, 32, 16) if q.dtype == torch.float32 else (64, 16)) or idx.shape[3] > 64:
        return None
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    out = torch.empty((b, n, h * d), dtype=q.dtype, device=q.device)
    with _on(q.device):
        rc = _lib.lib().s3r_select_attn_merge(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr(), o_cmp.data_ptr(), gate.data_ptr(), out.data_ptr(),
            b, h, n, d, block, idx.shape[3],
            q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
            v.stride(0), v.stride(1), v.stride(2), idx.stride(0), idx.stride(1), idx.stride(2),
            o_cmp.stride(0), o_cmp.stride(1), o_cmp.stride(2), gate.stride(0), gate.stride(1), gate.stride(2),
            scale, _code(q), _stream(q))
    if rc == _lib.S3R_ERR_UNSUPPORTED:
        return None
    _lib.check(rc, "s3r_select_attn_merge")
    return out


# ---- backward of the two attention operators --------------------------------------------------------------------

def bwd_supported(q: torch.Tensor, block: int = 64) -> bool:
    """The backward kernels are built for bf16/fp16, head_dim 64, blocks of 64 or 16 tokens."""
    return q.dtype in (torch.bfloat16, torch.float16) and q.shape[-1] == 64 and block in (64, 16)


def key_block_lists(idx: torch.Tensor, n_key_blocks: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """Key-centric view of the index tensor ``[B,H,Nq_blocks,K]``: for every (b, h) the query-block ids grouped by
    the key block they list, one entry per occurrence, ascending within a group, ``[B,H,Nq_blocks*K]`` int32, and the
    group offsets ``[B,H,n_key_blocks+1]``; entries < 0 or >= n_key_blocks appear in no group (the tail of the list
    tensor behind the last offset is then unspecified).  The reference's count + stable argsort + reorder
    (topk_blocksparse_attention.py:423-554)."""
    _need_device(idx)
    assert idx.dtype == torch.int32 and idx.dim() == 4 and n_key_blocks > 0
    idx = _last_contig(idx)
    b, h, nqb, kk = idx.shape
    lists = torch.empty((b, h, nqb * kk), dtype=torch.int32, device=idx.device)
    off = torch.empty((b, h, n_key_blocks + 1), dtype=torch.int32, device=idx.device)
    with _on(idx.device):
        rc = _lib.lib().s3r_key_block_lists(idx.data_ptr(), lists.data_ptr(), off.data_ptr(), b, h, nqb, kk, n_key_blocks,
                                            idx.stride(0), idx.stride(1), idx.stride(2), nqb * kk, _stream(idx))
    _lib.check(rc, "s3r_key_block_lists")
    return lists, off


def key_lists_ascending(lists: torch.Tensor, offs: torch.Tensor) -> bool:
    """Whether every group of ``lists`` ([B,H,L] int32, groups delimited by ``offs`` [B,H,n_key_blocks+1]) is ascending,
    as :func:`key_block_lists` builds them.  The dK/dV kernels add up in the order of a list, so that another order gives
    other roundings.  Works on CPU and GPU tensors (on the GPU: a few small kernels and one synchronisation)."""
    b, h, length = lists.shape
    if length < 2:
        return True
    dev = lists.device
    starts = torch.zeros((b, h, length + 1), dtype=torch.bool, device=dev)
    starts.scatter_(2, offs.long().clamp(0, length), True)                      # a pair that straddles a group start is free
    second = torch.arange(1, length, device=dev)
    beyond = second >= offs[..., -1:].long()                                     # so is the unspecified tail
    ok = (lists[..., 1:] >= lists[..., :-1]) | starts[..., 1:length] | beyond
    return bool(ok.all())


def attn_bwd_delta(o: torch.Tensor, dout: torch.Tensor) -> torch.Tensor:
    """``delta[b,h,n] = sum_d o * dout`` in fp32."""
    _need_device(o, dout)
    o, dout = _last_contig(o), _last_contig(dout)
    b, h, n, d = o.shape
    delta = torch.empty((b, h, n), dtype=torch.float32, device=o.device)
    with _on(o.device):
        rc = _lib.lib().s3r_attn_bwd_delta(o.data_ptr(), dout.data_ptr(), delta.data_ptr(), b, h, n, d,
                                           o.stride(0), o.stride(1), o.stride(2),
                                           dout.stride(0), dout.stride(1), dout.stride(2), _code(o), _stream(o))
    _lib.check(rc, "s3r_attn_bwd_delta")
    return delta


def attn_bwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, o: torch.Tensor, dout: torch.Tensor, lse: torch.Tensor,
             idx: Optional[torch.Tensor] = None, block: int = 64, softmax_scale: Optional[float] = None,
             need_dq: bool = True, need_dkv: bool = True, delta: Optional[torch.Tensor] = None,
             key_lists: Optional[Tuple[torch.Tensor, torch.Tensor]] = None, check_lists: Optional[bool] = None):
    """Gradients ``(dq, dk, dv)`` of an attention forward with output ``o`` and log-sum-exp ``lse``:
    selection attention over the blocks of ``idx`` ([B,H,Nq_blocks,K] int32), or dense attention (``idx=None``).
    ``delta`` (:func:`attn_bwd_delta`) and ``key_lists`` (:func:`key_block_lists`) are computed here unless given.
    Caller-built ``key_lists`` must be ascending within every group (see :func:`key_lists_ascending`);
    ``check_lists=True`` (default: the environment variable
    ``S3R_CHECK_LISTS=1``) verifies that here, at the price of a device synchronisation."""
    _need_device(q, k, v, o, dout, lse)
    assert bwd_supported(q, block), "attention backward: built for bf16/fp16, head_dim 64, block 64 or 16"
    q, k, v, o, dout = (_last_contig(t) for t in (q, k, v, o, dout))
    lse = lse.contiguous()
    b, h, lq, d = q.shape
    lk = k.shape[2]
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    # (a kernel that walks the queries reads the output beside the gradient that it reads anyway)
    inside = delta is None and need_dq and o.shape == q.shape and o.dtype == dout.dtype == q.dtype and 0 < o.stride(2) < 1 << 20
    if inside:
        delta = torch.empty((b, h, lq), dtype=torch.float32, device=q.device)
    elif delta is None:
        delta = attn_bwd_delta(o, dout)
    dq = torch.empty_like(q, memory_format=torch.contiguous_format) if need_dq else None
    dk = torch.empty_like(k, memory_format=torch.contiguous_format) if need_dkv else None
    dv = torch.empty_like(v, memory_format=torch.contiguous_format) if need_dkv else None
    nkb = -(-lk // block)
    lists = offs = None
    kk = 0
    if idx is not None:
        idx = _last_contig(idx)
        assert idx.dtype == torch.int32 and idx.shape[:3] == (b, h, -(-lq // block))
        kk = idx.shape[3]
        if need_dkv:
            lists, offs = key_lists if key_lists is not None else key_block_lists(idx, nkb)
            if key_lists is not None and (check_lists if check_lists is not None else os.environ.get("S3R_CHECK_LISTS") == "1"):
                if not key_lists_ascending(lists, offs):
                    raise ValueError("attn_bwd: key_lists must be ascending within every key block's group "
                                     "(build them with key_block_lists)")

    def st(t):
        return (t.stride(0), t.stride(1), t.stride(2)) if t is not None else (0, 0, 0)

    rest = (idx.data_ptr() if idx is not None else None,
            lists.data_ptr() if lists is not None else None, offs.data_ptr() if offs is not None else None,
            lists.shape[-1] if lists is not None else 0,
            dq.data_ptr() if dq is not None else None, dk.data_ptr() if dk is not None else None,
            dv.data_ptr() if dv is not None else None,
            b, h, lq, lk, d, block, kk,
            *st(q), *st(k), *st(v), *st(dout), *st(dq), *st(dk), *st(dv), *st(idx),
            scale, _code(q), _stream(q))
    first = (q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), lse.data_ptr())
    with _on(q.device):
        if inside:
            rc = _lib.lib().s3r_attn_bwd_from_output(*first, o.data_ptr(), *st(o), delta.data_ptr(), *rest)
        else:
            rc = _lib.lib().s3r_attn_bwd(*first, delta.data_ptr(), *rest)
    _lib.check(rc, "s3r_attn_bwd")
    return dq, dk, dv


class _SelectAttnFn(torch.autograd.Function):
    """Selection attention with gradients (reference TopkBlockSparseAttention, topk_blocksparse_attention.py:1041-1090)."""

    @staticmethod
    def forward(ctx, q, k, v, idx, block, softmax_scale):
        with torch.no_grad():
            o, lse = select_attn(q, k, v, idx, block, softmax_scale, return_lse=True)
        ctx.save_for_backward(q, k, v, o, lse, idx)
        ctx.block, ctx.scale = block, softmax_scale
        return o

    @staticmethod
    def backward(ctx, dout):
        q, k, v, o, lse, idx = ctx.saved_tensors
        dq, dk, dv = attn_bwd(q, k, v, o, dout, lse, idx, ctx.block, ctx.scale,
                              need_dq=ctx.needs_input_grad[0], need_dkv=ctx.needs_input_grad[1] or ctx.needs_input_grad[2])
        return dq, dk, dv, None, None, None


class _CompressedAttnFn(torch.autograd.Function):
    """Compressed attention + top-k with gradients for the attention output (the indices carry none; reference
    FlashAttnTopkFunc, flash_attention_topk.py:633-665)."""

    @staticmethod
    def forward(ctx, q, k, v, topk, softmax_scale, causal=False):
        with torch.no_grad():
            o, idx, lse = compressed_attn_topk(q, k, v, topk, softmax_scale, return_lse=True, causal=causal)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.scale = softmax_scale
        if idx is not None:
            ctx.mark_non_differentiable(idx)
        return o, idx

    @staticmethod
    def backward(ctx, dout, _didx):
        q, k, v, o, lse = ctx.saved_tensors
        dq, dk, dv = attn_bwd(q, k, v, o, dout, lse, None, 64, ctx.scale,
                              need_dq=ctx.needs_input_grad[0], need_dkv=ctx.needs_input_grad[1] or ctx.needs_input_grad[2])
        return dq, dk, dv, None, None, None   # (the reference's backward does not know of `causal` either, :653-666)


def _at_16_bytes(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """``t`` or, where it does not start at a multiple of 16 bytes (a view of a flat buffer), a copy that does."""
    return t if t is None or t.data_ptr() % 16 == 0 else t.clone()


def gated_merge_bwd(dout: torch.Tensor, o_cmp: torch.Tensor, o_sel: torch.Tensor, gate: torch.Tensor, block: int):
    """Gradient of :func:`gated_merge` (bf16/fp16, head_dim 64): ``(d_o_cmp, d_o_sel, d_gate, delta_cmp, delta_sel)``, d_gate
    as the ``[B,H,N,2]`` view of a ``[B,N,H,2]`` tensor, the deltas as :func:`attn_bwd` takes them."""
    b, h, n, d = o_sel.shape
    dout, o_cmp, o_sel, gate = _at_16_bytes(dout.contiguous()), o_cmp.contiguous(), o_sel.contiguous(), _last_contig(gate)
    d_oc, d_os = torch.empty_like(o_cmp), torch.empty_like(o_sel)
    d_gate = gate.new_empty((b, n, h, 2))
    delta_c = torch.empty(o_cmp.shape[:3], dtype=torch.float32, device=gate.device)
    delta_s = torch.empty((b, h, n), dtype=torch.float32, device=gate.device)
    with _on(gate.device):
        rc = _lib.lib().s3r_gated_merge_bwd(
            dout.data_ptr(), o_cmp.data_ptr(), o_sel.data_ptr(), gate.data_ptr(), d_oc.data_ptr(), d_os.data_ptr(), d_gate.data_ptr(),
            delta_c.data_ptr(), delta_s.data_ptr(), b, h, n, d, block, gate.stride(0), gate.stride(1), gate.stride(2), _code(gate), _stream(gate))
    _lib.check(rc, "s3r_gated_merge_bwd")
    return d_oc, d_os, d_gate.permute(0, 2, 1, 3), delta_c, delta_s


PREPASS_BWD_ROWS = 768   # workgroups of the projection's backward pass that hold parameter sums: three per CU


def qkv_prepass_bwd(qkv: torch.Tensor, num_heads: int, block: int, positions, cos_tab, sin_tab, q_ln, k_ln, eps: float, raw, grads,
                    inv_freq=None, signed: bool = False):
    """Gradient of :func:`qkv_prepass` with ``pooled="final"``: ``raw`` = the raw (q_c, k_c), ``grads`` = the gradients of
    (q, k, v, q_c, k_c, v_c).  Returns ``(d_qkv, d_norm)``, d_norm ``[4,64]`` fp32 (q weight, q bias, k weight, k bias) or
    None without a norm."""
    a, keep = _prepass_args(qkv, num_heads, block, positions, cos_tab, sin_tab, q_ln, k_ln, float(eps), inv_freq, signed)
    a.q_raw, a.k_raw = (t.data_ptr() for t in raw)
    grads = [t.contiguous() for t in grads]
    d_qkv = torch.empty_strided(qkv.shape, qkv.stride(), dtype=qkv.dtype, device=qkv.device)
    off = [d_qkv.data_ptr() + i * num_heads * 64 * d_qkv.element_size() for i in range(3)]
    d_norm = work = None
    if q_ln is not None:
        work = torch.empty((PREPASS_BWD_ROWS, 256), dtype=torch.float32, device=qkv.device)
        d_norm = torch.empty((4, 64), dtype=torch.float32, device=qkv.device)
    with _on(qkv.device):
        rc = _lib.lib().s3r_layer_prepass_bwd(ctypes.byref(a), *(t.data_ptr() for t in grads), *off,
                                              d_norm.data_ptr() if d_norm is not None else None,
                                              work.data_ptr() if work is not None else None, PREPASS_BWD_ROWS, _stream(qkv))
    _lib.check(rc, "s3r_layer_prepass_bwd")
    return d_qkv, d_norm


def _norm_grads(d_norm: Optional[torch.Tensor], params):
    """Rows of ``d_norm`` in the types of ``params`` (None: none), tensors of their own: autograd keeps what it is given as .grad.  Those of
    its own type by one launch, not a copy each; the others' conversion is a copy."""
    same = [i for i, t in enumerate(params) if t is not None and t.dtype == d_norm.dtype]
    own = dict(zip(same, torch._foreach_mul([d_norm[i] for i in same], 1.0))) if same else {}
    return [None if t is None else own[i] if i in own else d_norm[i].to(t.dtype) for i, t in enumerate(params)]


class _LayerCoreFn(torch.autograd.Function):
    """Everything of the layer between its projections, ``(packed qkv, gate, qk-norm parameters) -> ([B,N,C], indices)``
    (pi3/models/layers/sparse_attention.py:97-136): the forward kernels of the inference route with their log-sum-exps,
    and a backward of kernels only.  Between the two the I/O-dtype tensors that a kernel reads again are kept."""

    @staticmethod
    def forward(ctx, qkv, gate, q_w, q_b, k_w, k_b, xpos, cos, sin, inv_freq, heads, block, topk, eps):
        q_ln, k_ln = ((q_w, q_b), (k_w, k_b)) if q_w is not None else (None, None)
        with torch.no_grad():
            q, k, v, q_c, k_c, v_c, q_raw, k_raw = qkv_prepass(qkv, heads, block, xpos, cos, sin, q_ln, k_ln, eps, pooled="final",
                                                               keep_raw=True, inv_freq=inv_freq, signed=True)
            o_c, idx, lse_c = compressed_attn_topk(q_c, k_c, v_c, topk, return_lse=True)
            o_s, lse = select_attn(q, k, v, idx, block, return_lse=True)
            out = gated_merge(o_c, o_s, gate, block)
        ctx.save_for_backward(qkv, gate, q_w, q_b, k_w, k_b, xpos, cos, sin, inv_freq, q, k, q_c, k_c, v_c, q_raw, k_raw, o_c, lse_c, o_s, lse, idx)
        ctx.args = heads, block, eps
        ctx.mark_non_differentiable(idx)
        return out, idx

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dout, _didx):
        qkv, gate, q_w, q_b, k_w, k_b, xpos, cos, sin, inv_freq, q, k, q_c, k_c, v_c, q_raw, k_raw, o_c, lse_c, o_s, lse, idx = ctx.saved_tensors
        heads, block, eps = ctx.args
        b, n, _ = qkv.shape
        v = qkv.as_strided((b, heads, n, 64), (qkv.stride(0), 64, qkv.stride(1), 1), qkv.storage_offset() + 2 * heads * 64)
        d_oc, d_os, d_gate, delta_c, delta_s = gated_merge_bwd(dout, o_c, o_s, gate, block)
        pooled = attn_bwd(q_c, k_c, v_c, o_c, d_oc, lse_c, delta=delta_c)
        full = attn_bwd(q, k, v, o_s, d_os, lse, idx, block, delta=delta_s)
        q_ln, k_ln = ((q_w, q_b), (k_w, k_b)) if q_w is not None else (None, None)
        d_qkv, d_norm = qkv_prepass_bwd(qkv, heads, block, xpos, cos, sin, q_ln, k_ln, eps, (q_raw, k_raw), (*full, *pooled), inv_freq, signed=True)
        return d_qkv, d_gate, *_norm_grads(d_norm, (q_w, q_b, k_w, k_b)), *([None] * 8)


def layer_core_autograd(qkv: torch.Tensor, gate: torch.Tensor, heads: int, block: int, topk: int, xpos, cos, sin, inv_freq, q_ln, k_ln, eps: float):
    """``(out [B,N,C], indices)`` of the layer between its projections, differentiable in qkv, gate and the norm parameters,
    or None where the kernels are not built (bf16/fp16, head_dim 64, blocks of 64 or 16 tokens).  Where only the gate
    wants a gradient: ``(o_cmp, o_sel, indices)``, constants of the merge, whose gradient is a product of torch."""
    if qkv.dtype not in (torch.bfloat16, torch.float16) or gate.dtype != qkv.dtype or qkv.shape[-1] != 3 * heads * 64 or block not in (64, 16) \
            or not qkv.is_contiguous() or qkv.data_ptr() % 16:
        return None
    if xpos is not None and xpos.is_inference():   # (such a tensor can't be saved for the backward)
        xpos = xpos.clone()
    params = [_at_16_bytes(t) for t in (*(q_ln or (None, None)), *(k_ln or (None, None)))]
    if not _wants_grad(qkv, *params):
        q_ln, k_ln = (params[:2], params[2:]) if q_ln is not None else (None, None)
        with torch.no_grad():
            q, k, v, q_c, k_c, v_c = qkv_prepass(qkv, heads, block, xpos, cos, sin, q_ln, k_ln, eps, pooled="final", inv_freq=inv_freq, signed=True)
            o_c, idx = compressed_attn_topk(q_c, k_c, v_c, topk)
            o_s = select_attn(q, k, v, idx, block)
            return (o_c, o_s, idx) if gate.requires_grad else (gated_merge(o_c, o_s, gate, block), idx)
    return _LayerCoreFn.apply(qkv, gate, *params, xpos, cos, sin, inv_freq, heads, block, topk, eps)


def _wants_grad(*ts: torch.Tensor) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)


def select_attn_autograd(q, k, v, idx, block, softmax_scale=None):
    """:func:`select_attn`, differentiable in q, k, v where the backward kernels are built."""
    if not _wants_grad(q, k, v):
        return select_attn(q, k, v, idx, block, softmax_scale)
    if block in (128, 256):
        assert idx.shape[2] == -(-q.shape[2] // block), "topk_idx does not match the number of query blocks"
        idx, block = _as_64_token_blocks(idx, block, q.shape[2]), 64
    if not bwd_supported(q, block):
        raise RuntimeError("speed3r_amd: the attention backward is built for bf16/fp16, head_dim 64, blocks of 64 or 16 tokens")
    return _SelectAttnFn.apply(q, k, v, idx, block, softmax_scale)


def compressed_attn_topk_autograd(q, k, v, topk, softmax_scale=None, causal=False):
    """:func:`compressed_attn_topk` (``(o, idx)``), differentiable in q, k, v where the backward kernels are built."""
    if not _wants_grad(q, k, v):
        return compressed_attn_topk(q, k, v, topk, softmax_scale, causal=causal)
    if not bwd_supported(q):
        raise RuntimeError("speed3r_amd: the attention backward is built for bf16/fp16, head_dim 64 only")
    return _CompressedAttnFn.apply(q, k, v, topk, softmax_scale, causal)


_SIDE_STREAMS = {}


def _side_stream(device: torch.device) -> "torch.cuda.Stream":
    """One extra stream per device (default priority), created on first use and kept."""
    key = torch.device(device).index if torch.device(device).index is not None else torch.cuda.current_device()
    if key not in _SIDE_STREAMS:
        _SIDE_STREAMS[key] = torch.cuda.Stream(device=key)
    return _SIDE_STREAMS[key]


def _two_kernel_compressed(q: torch.Tensor, topk: int, block: int = 1) -> bool:
    """True where the compressed branch is two independent kernels (attention, indices without a score buffer): not for short lists of
    keys, whose indices and attention are one launch.
    ``q``: the pooled queries (``block`` = 1) or the full tokens that will be pooled over ``block`` tokens."""
    blocks = -(-q.shape[2] // block)
    return (q.dtype != torch.float32 and q.shape[-1] == 64 and topk in (1, 2, 4, 8, 16, 32)
            and blocks <= (1 << 21) and _lib.lib_has_fused_topk()
            and not _lib.lib().s3r_topk_in_lds(q.shape[0] * q.shape[1], blocks, blocks, topk))


# When the index kernel goes on a stream of its own.  The two events and the change of stream cost the host up to 40 us and the kernels
# behind them a wait between queues; what there is to hide is the dense sweep (and the pooling of v, or a layer's gate).  Short lists of keys
# are one launch with the attention.  The two-sweep kernel pays from 19 456 pooled rows (B * H * blocks) on; long lists over few heads, whose
# chain is long and leaves most of the chip idle, from 8192.  Operators, us per call, two streams / one, 16 heads: 16-token blocks, top-32,
# 1 512 pooled tokens 185 / 188, 2 016 235 / 237, 3 780 438 / 441; 64-token blocks, top-16, 1 302 480 / 482, 1 952 701 / 702, 2 603 938 / 953, 4 164
# 1 532 / 1 551.  Layers, up to 512 workgroups of 64 pooled rows: see attention_layer; beyond, 6 489 blocks of 16 2 368 / 2 415, 12 600
# 5 410 / 5 630, 4 164 of 64 4 295 / 4 360, 3 x 16 heads of 1 008 of 16 798 / 812.  The line is too early for layers of 2 049 to some 5 500
# blocks of 16 (16 heads), which would be 1 to 3 % faster in one call: 2 520 798 / 792, 3 780 1 193 / 1 165, 5 040 1 711 / 1 665.
SIDE_STREAM_ROWS = 16 * 1216
SIDE_STREAM_ROWS_OF_LONG_LISTS = 8192


def _side_stream_pays(heads: int, blocks: int, topk: int) -> bool:
    """``heads``: those of all sequences; ``blocks``: pooled tokens of each."""
    rows = heads * blocks
    return (rows > SIDE_STREAM_ROWS or (topk > 8 and blocks > 2432 and rows > SIDE_STREAM_ROWS_OF_LONG_LISTS)) \
        and not _lib.lib().s3r_topk_in_lds(heads, blocks, blocks, topk)


def _indices_beside(q: torch.Tensor, topk: int, block: int = 1) -> bool:
    """True where the index kernel runs on the side stream (arguments as for :func:`_two_kernel_compressed`)."""
    return _side_stream_pays(q.shape[0] * q.shape[1], -(-q.shape[2] // block), topk) and _two_kernel_compressed(q, topk, block)


def topk_indices_on_side_stream(qc: torch.Tensor, kc: torch.Tensor, topk: int, softmax_scale: Optional[float] = None):
    """Launch the index kernel (top-k columns of the raw scores ``qc kc^T``, no score buffer) on the device's side
    stream, ordered after the work already queued on the current stream.  Returns ``(idx, join)``; call ``join()``
    on the current stream before the first use of ``idx`` there.  Needs :func:`_two_kernel_compressed`."""
    main = torch.cuda.current_stream(qc.device)
    side = _side_stream(qc.device)
    ready = torch.cuda.Event()
    ready.record(main)
    side.wait_event(ready)
    with torch.cuda.stream(side):
        _, idx = compressed_attn_topk(qc, kc, None, topk, softmax_scale)
        done = torch.cuda.Event()
        done.record(side)

    def join():
        torch.cuda.current_stream(qc.device).wait_event(done)
        idx.record_stream(torch.cuda.current_stream(qc.device))

    return idx, join


def sparse_global_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, gate: torch.Tensor,
                            block: int = 64, topk: int = 16, softmax_scale: Optional[float] = None,
                            return_parts: bool = False, materialize_scores: Optional[bool] = None,
                            fuse_merge: bool = True, overlap: Optional[bool] = None, timeline: Optional[dict] = None):
    """The whole path on post-norm/RoPE q, k, v ``[B,H,N,D]`` and gate ``[B,H,N,2]``:
    pool -> compressed attention + top-k -> selection attention -> gated merge -> ``[B,N,H*D]``.
    The merge runs in the selection kernel's epilogue where the library offers it (same bits either way but for 64-token
    blocks of 16-bit types, which are then rounded once, see :func:`select_attn_merge`);
    ``return_parts`` needs the selection output and therefore runs the two operators separately.

    ``overlap`` (default: where :func:`_side_stream_pays` says so; True: wherever it applies): the indices need pooled q and k only, the compressed attention output
    is not read before the merge.  Where the two come from different kernels (no score buffer, more keys than one launch
    takes for both: :func:`_two_kernel_compressed`), the index kernel runs on a second stream next to the pooling of v and the
    compressed attention (same kernels, same results; only the schedule differs).  Both sides measured: at
    ``SIDE_STREAM_ROWS``.  ``overlap=False`` runs the kernels one after the other on the calling stream.

    ``timeline``: a dict that receives timing events of the calling stream under "start", "pooled" (sequential
    schedule only), "select" (everything before the selection kernel is done) and "end".
    """
    def mark(name):
        if timeline is not None:
            ev = torch.cuda.Event(enable_timing=True)
            ev.record(torch.cuda.current_stream(q.device))
            timeline[name] = ev

    mark("start")
    if overlap is not False and materialize_scores is not True and not return_parts and q.is_cuda \
            and (_two_kernel_compressed if overlap else _indices_beside)(q, topk, block):
        qc, kc = pool_mean(q, block), pool_mean(k, block)
        idx, join = topk_indices_on_side_stream(qc, kc, topk, softmax_scale)
        vc = pool_mean(v, block)
        o_cmp, _ = compressed_attn_topk(qc, kc, vc, None, softmax_scale)
        join()
    else:
        qc, kc, vc = _pool_means(q, k, v, block)
        mark("pooled")
        o_cmp, idx = compressed_attn_topk(qc, kc, vc, topk, softmax_scale, materialize_scores=materialize_scores)
    mark("select")
    if fuse_merge and not return_parts:
        out = _select_attn_merge(q, k, v, idx, o_cmp, gate, block, softmax_scale)
        if out is not None:
            mark("end")
            return out
    o_sel = select_attn(q, k, v, idx, block, softmax_scale)
    mark("merge")
    out = gated_merge(o_cmp, o_sel, gate, block)
    mark("end")
    if return_parts:
        return out, dict(idx=idx, o_cmp=o_cmp, o_sel=o_sel, qc=qc, kc=kc, vc=vc)
    return out
