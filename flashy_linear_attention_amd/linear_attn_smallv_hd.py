"""``LinearAttentionSmallVHD``: causal linear attention whose query/key head dim
exceeds the value head dim (e.g. 256-wide Taylor features over 64-wide values).

Drop-in for the reference's autograd Function
(flashlinear/linear_attn_smallv_hd.py:14-36).
"""

from typing import Any, Tuple

import torch
from torch.autograd import Function

from . import _native
from .auto import chunked_keeps_range, evaluate_bwd, evaluate_fwd, prefers_chunked
from .kernels.linear_attn_kernels_smallv_hd import check_operands


class LinearAttentionSmallVHD(Function):
    @classmethod
    def apply(cls, *args):
        if cls is LinearAttentionSmallVHD and len(args) == 3:
            out = _native.product(1, *args)
            if out is not None:
                return out
        return super().apply(*args)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.bfloat16)
    def forward(ctx: Any, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        check_operands(q, k, v)
        # (D_v up to 128 only: see LinearAttention.  The quadratic backward wants
        # N a multiple of 64 where forward takes 32, so such a sequence stays with it)
        grad = any(ctx.needs_input_grad)
        chunked = (q.shape[2] % 64 == 0 and v.shape[-1] <= 128 and chunked_keeps_range(q, v, grad)
                   and prefers_chunked(q, v, grad))
        return evaluate_fwd(ctx, q, k, v, chunked, False)

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx: Any, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        return evaluate_bwd(ctx, grad_output)
