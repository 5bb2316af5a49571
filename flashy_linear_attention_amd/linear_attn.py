"""``LinearAttention``: un-normalised causal linear attention, O = tril(Q K^T) V.

Drop-in for the reference's autograd Function (flashlinear/linear_attn.py:11-31):
same ``apply(q, k, v)`` surface, same AMP behaviour (inputs are cast to bf16
under autocast), saves (q, k, v) for backward.  The denominator of full linear
attention stays with the caller in PyTorch (README.md:27-30).
"""

from typing import Any, Tuple

import torch
from torch.autograd import Function

from . import _native
from .auto import chunked_keeps_range, evaluate_bwd, evaluate_fwd, prefers_chunked
from .kernels.linear_attn_kernels import check_operands


class LinearAttention(Function):
    @classmethod
    def apply(cls, *args):
        if cls is LinearAttention and len(args) == 3:
            out = _native.product(0, *args)
            if out is not None:
                return out
        return super().apply(*args)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.bfloat16)
    def forward(ctx: Any, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        check_operands(q, k, v)
        # The chunk-wise kernels where the measured thresholds say so, up to 25 times faster on long sequences.
        # Head dims up to 128: beyond, dQ and dK are sums over v's column halves, each half rounded.
        grad = any(ctx.needs_input_grad)
        chunked = q.shape[-1] <= 128 and chunked_keeps_range(q, v, grad) and prefers_chunked(q, v, grad)
        return evaluate_fwd(ctx, q, k, v, chunked, True)

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx: Any, grad_output: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        return evaluate_bwd(ctx, grad_output)
