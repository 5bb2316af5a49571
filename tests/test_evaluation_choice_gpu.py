"""The reference-named Functions choose the quadratic or the chunk-wise evaluation by shape: both sides of
the thresholds against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionSmallVHD
from flashy_linear_attention_amd.auto import prefers_chunked

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


# (B, H, N, D_qk, D_v): the smallest problems, the last below and the first above each threshold, remainders of the
# chunks (N a multiple of 64 only), widths that the tiles pad
@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (1, 1, 64, 32, 32), (1, 4, 960, 64, 64), (1, 17, 1984, 64, 64), (2, 3, 4032, 48, 48), (1, 2, 5440, 128, 128),
    (1, 8, 2880, 96, 96), (3, 5, 2112, 120, 120), (1, 4, 1984, 256, 64), (1, 2, 1088, 256, 64), (1, 7, 1472, 192, 128),
    (1, 9, 832, 128, 64), (2, 2, 448, 64, 32), (1, 1, 4096, 256, 256),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_evaluations_match_the_oracle(b, h, n, dqk, dv, dtype, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(b, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = (LinearAttention if dqk == dv else LinearAttentionSmallVHD).apply(*leaves)
    assert_close(f"O (chunk-wise preferred: {prefers_chunked(q, v)})", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, leaves, do), want_g):
        assert_close(name, got, want)
