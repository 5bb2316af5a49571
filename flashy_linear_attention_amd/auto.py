"""``LinearAttentionAuto``: the reference's operator with the evaluation chosen by shape.

``LinearAttentionAuto.apply(q, k, v)`` takes the arguments of both ``LinearAttention`` and
``LinearAttentionSmallVHD`` (flashlinear/linear_attn.py:11-31, linear_attn_smallv_hd.py:14-36) and
returns the same ``tril(Q K^T) V``; it runs the quadratic kernels where they are faster (short
sequences, few heads) and the chunk-wise ones elsewhere, by the library's table of measured
thresholds (``fla_linear_attn_prefers_chunked``) and where that narrows no range
(:func:`chunked_keeps_range`; an infinite value is infinite or NaN in its column of the results either way, which of the
two goes by the evaluation) -- the reference lists autotuning as a to-do (README.md:68).  The
two reference-named Functions choose the same way within the reference's limits on shapes; quadratic calls of widths
that are no multiples of 8 run the fast kernels on copies (``fla_linear_attn_copies_fwd/bwd``);
``kernels.linear_flash_wrapper_*`` are the quadratic kernels whatever the shape.
"""

from __future__ import annotations

from typing import Any, Tuple

import torch
from torch.autograd import Function

from . import _lib, _native
from .chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd
from .kernels import (
    linear_flash_wrapper_bwd,
    linear_flash_wrapper_bwd_smallv_hd,
    linear_flash_wrapper_fwd,
    linear_flash_wrapper_fwd_smallv_hd,
)
from .kernels._common import call, device_guard, dtype_code, prepare, stream_handle


def prefers_chunked(q: torch.Tensor, v: torch.Tensor, grad: bool = True) -> bool:
    """Whether the chunk-wise kernels are the faster choice for (B, H, N, D_qk) q and (B, H, N, D_v) v, for forward +
    backward or (``grad`` false) forward alone."""
    b, h, n, dqk = q.shape
    return bool(_lib.query("fla_linear_attn_operator_prefers_chunked", b, h, n, dqk, v.shape[-1], int(grad)))


def rows_for_walks(t: torch.Tensor) -> bool:
    """Whether the walks' tile loads take a tensor's rows as they are (others go product by product)."""
    if t.stride(3) != 1:
        return True  # (copied for the call)
    return (all(t.stride(i) % 8 == 0 for i in range(3)) and t.data_ptr() % 16 == 0 and t.stride(2) >= t.shape[3]
            and t.shape[2] * t.stride(2) < 1 << 28)


def chunked_keeps_range(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, grad: bool) -> bool:
    """Whether the chunk-wise evaluation takes whatever the quadratic one does.  bf16: yes.  fp16: a state element may
    exceed 65504 where no score and no result does; the forward walk (head dims up to 128, multiples of 8, more than
    256 rows) scales its state's fp16 copy, and so do the walks of the backward pass (where the library says so, at lengths
    from which they are the faster ones, for rows that they take)."""
    if q.dtype == torch.bfloat16:
        return True
    dqk, dv = q.shape[-1], v.shape[-1]
    if not grad:
        return max(dqk, dv) <= 128 and dqk % 8 == 0 and dv % 8 == 0 and q.shape[2] > 256
    return bool(_lib.query("fla_linear_attn_f16_pair_prefers_chunked", *q.shape, dv)) and all(rows_for_walks(t) for t in (q, k, v))


def rounded_once(q: torch.Tensor, v: torch.Tensor) -> bool:
    """Whether the chunk-wise evaluation rounds every result once, as the quadratic one does: not for a v above 128 columns, whose
    halves' dQ and dK are added up in memory, unless q and k are above 128 columns too (multiples of 8)."""
    dqk, dv = q.shape[-1], v.shape[-1]
    return dv <= 128 or (dqk > 128 and dqk % 8 == 0 and dv % 8 == 0)


def _copies_bytes(q: torch.Tensor, v: torch.Tensor, backward: int) -> int:
    """Workspace of the quadratic evaluation on copies with aligned rows (widths that are no multiples of 8), 0 where it is not taken."""
    shape = (*q.shape, v.shape[-1], backward)
    if not _lib.query("fla_linear_attn_operator_prefers_copies", *shape):
        return 0
    return _lib.query("fla_linear_attn_copies_bytes", *shape)


def _copies_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    q, k, v = prepare(q, k, v)
    out = torch.empty_like(v, memory_format=torch.contiguous_format)
    with device_guard(q.device):
        nbytes = _copies_bytes(q, v, 0)
        work = torch.empty(nbytes, dtype=torch.uint8, device=q.device)
        call("fla_linear_attn_copies_fwd", *(t.data_ptr() for t in (q, k, v, out)), *q.shape, v.shape[-1],
             *(_lib.strides_arg(t) for t in (q, k, v, out)), dtype_code(q), work.data_ptr(), nbytes, stream_handle(q.device))
    return out


def _copies_bwd(grad_output: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> Tuple[torch.Tensor, ...]:
    tensors = prepare(grad_output, q, k, v)
    grads = tuple(torch.empty_like(t, memory_format=torch.contiguous_format) for t in tensors[1:])
    with device_guard(q.device):
        nbytes = _copies_bytes(q, v, 1)
        work = torch.empty(nbytes, dtype=torch.uint8, device=q.device)
        call("fla_linear_attn_copies_bwd", *(t.data_ptr() for t in (*tensors, *grads)), *q.shape, v.shape[-1],
             *(_lib.strides_arg(t) for t in (*tensors, *grads)), dtype_code(q), work.data_ptr(), nbytes, stream_handle(q.device))
    return grads


def evaluate_fwd(ctx: Any, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, chunked: bool, equal: bool) -> torch.Tensor:
    """Forward of an autograd Function by the evaluation `chunked` names; keeps what :func:`evaluate_bwd` needs."""
    ctx.chunked, ctx.equal = chunked, equal
    # (an fp16 pair that is chunk-wise because the walks keep the range)
    ctx.walks = chunked and q.dtype == torch.float16 and any(ctx.needs_input_grad[:3]) and chunked_keeps_range(q, k, v, True)
    state = None
    if chunked:
        if any(ctx.needs_input_grad[:3]):
            out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
        else:
            out = linear_attention_chunked_fwd(q, k, v)
    elif _copies_bytes(q, v, 0):
        out = _copies_fwd(q, k, v)
    else:
        out = linear_flash_wrapper_fwd(q, k, v) if equal else linear_flash_wrapper_fwd_smallv_hd(q, k, v)
    ctx.has_state = state is not None
    ctx.save_for_backward(*((q, k, v, state) if state is not None else (q, k, v)))
    return out


def evaluate_bwd(ctx: Any, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    if ctx.has_state:
        q, k, v, state = ctx.saved_tensors
    else:
        (q, k, v), state = ctx.saved_tensors, None
    if ctx.chunked:
        if ctx.walks:  # (a gradient whose rows they do not take is copied)
            grad_output, q, k, v = (t if rows_for_walks(t) else t.clone(memory_format=torch.contiguous_format)
                                    for t in prepare(grad_output, q, k, v))
        # (what later rows hold must not reach dQ, as in the quadratic evaluation)
        return linear_attention_chunked_bwd(grad_output, q, k, v, state, causal=True)
    if _copies_bytes(q, v, 1):
        return _copies_bwd(grad_output, q, k, v)
    if ctx.equal:
        return linear_flash_wrapper_bwd(grad_output, q, k, v)
    return linear_flash_wrapper_bwd_smallv_hd(grad_output, q, k, v)


class LinearAttentionAuto(Function):
    @classmethod
    def apply(cls, *args):
        if cls is LinearAttentionAuto and len(args) == 3:
            out = _native.product(2, *args)
            if out is not None:
                return out
        return super().apply(*args)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.bfloat16)
    def forward(ctx: Any, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        assert q.dim() == 4 and q.shape == k.shape and v.shape[:3] == q.shape[:3], "q, k: (B,H,N,D_qk); v: (B,H,N,D_v)"
        # (the quadratic wrappers keep the reference's limits: N a multiple of 64 and, with unequal head dims,
        # D_v a power of two not above D_qk -- what they refuse goes to the chunk-wise kernels)
        dqk, dv = q.shape[-1], v.shape[-1]
        equal = dqk == dv
        refused = q.shape[2] % 64 != 0 or (not equal and (dv > dqk or dv & (dv - 1)))
        grad = any(ctx.needs_input_grad)
        chunked = refused or (chunked_keeps_range(q, k, v, grad) and prefers_chunked(q, v, grad))
        return evaluate_fwd(ctx, q, k, v, chunked, equal)

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx: Any, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        return evaluate_bwd(ctx, grad_output)
