"""Backward of the chunk-wise operator with dQ by walks in forward direction (``causal``) against the fp32 oracle: one, two,
several and many segments, each with forward's states and without; unequal and narrow widths, halves of a wide q / k, ragged
lengths, (B, N, H, D) storage, both dtypes (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (1, 2, 257, 128, 128), (3, 90, 300, 96, 96), (2, 64, 513, 128, 128), (1, 40, 1000, 72, 128), (1, 2, 1999, 128, 24),
    (1, 3, 700, 64, 128), (1, 1, 1500, 40, 72), (2, 70, 321, 256, 64), (1, 66, 500, 136, 128), (1, 30, 700, 200, 96),
    (1, 3, 1100, 160, 32), (1, 2, 900, 192, 128), (1, 5, 640, 153, 64), (1, 2, 450, 91, 100), (2, 3, 1030, 64, 64),
    (1, 2, 600, 130, 200), (1, 2, 600, 100, 255),
])
@pytest.mark.parametrize("dtype,transposed", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, True)])
def test_causal_backward(b, h, n, dqk, dv, dtype, transposed, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(b, h, n, dqk, dv, dtype, seed=n + dqk))
    _, want = gpu_fp32_reference(q, k, v, do, True)
    if transposed:  # (B, N, H, D) storage
        q, k, v, do = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v, do))
    _, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    for st in (state, None):
        for name, got, w in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, st, causal=True), want):
            assert_close(f"{name}, state {st is not None}", got, w)
