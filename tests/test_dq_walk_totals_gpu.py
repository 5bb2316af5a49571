"""Backward with dQ by its own walk, three segments or more: that walk adds up the reverse walk's segment totals of Q^T dO on its way
-- both sides wide, a narrow v, both halves of a wide q / k, results in fp32 and in rows of any alignment, totals that the reverse walk
sums and ones that are scanned -- against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionAuto, LinearAttentionSmallVHD
from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


# (heads, N, columns): 3, 8, 20, 21 and 28 segments of 64-row chunks up to 128 columns, 3, 7, 8 and 13 with a wide q / k, ragged ends
@pytest.mark.parametrize("h,n,dqk,dv", [
    (80, 300, 128, 128), (24, 1500, 80, 80), (12, 20 * 64 - 5, 128, 100), (12, 21 * 64 - 5, 100, 128), (9, 1787, 72, 128),
    (32, 1000, 128, 64), (32, 1000, 91, 64), (9, 1787, 128, 32), (70, 450, 256, 64), (36, 7 * 64 - 7, 153, 64), (32, 8 * 64 - 7, 256, 64),
    (19, 820, 192, 40), (32, 8 * 64 - 7, 256, 128), (19, 820, 200, 72), (32, 500, 160, 128),
])
def test_against_the_oracle(h, n, dqk, dv, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    for kept in (state, None):
        for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, kept, True), want_g):
            assert_close(name, got, want)


@pytest.mark.parametrize("op,h,n,dqk,dv", [(LinearAttentionAuto, 24, 1500, 80, 80), (LinearAttentionSmallVHD, 32, 960, 256, 64),
                                           (LinearAttentionSmallVHD, 32, 960, 128, 64)])
def test_gradients_in_fp32(op, h, n, dqk, dv, gpu_device):
    inputs = [t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=n)]
    do, want = inputs.pop(), None
    for amp in (False, True):
        q, k, v = (t.float().requires_grad_() if amp else t.clone().requires_grad_() for t in inputs)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            out = op.apply(q, k, v)
        grads = torch.autograd.grad(out, (q, k, v), do)
        if amp:
            assert all(g.dtype == torch.float32 and torch.equal(g, w.float()) for g, w in zip(grads, want))
        want = grads


def test_late_rows_stay_out_of_early_gradients_of_q(gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, 24, 1500, 128, 128, torch.bfloat16, seed=5))
    clean = linear_attention_chunked_bwd(do, q, k, v, linear_attention_chunked_fwd(q, k, v, want_state=True)[1], True)
    for t in (q, k, v, do):
        t[..., 1400:, :] = float("nan")
    dq, _, _ = linear_attention_chunked_bwd(do, q, k, v, linear_attention_chunked_fwd(q, k, v, want_state=True)[1], True)
    assert torch.equal(dq[..., : 1400 // 64 * 64, :], clean[0][..., : 1400 // 64 * 64, :])
