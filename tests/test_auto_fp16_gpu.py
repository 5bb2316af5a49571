"""``LinearAttentionAuto`` in fp16 with gradients where a chunk-wise state would leave fp16's range and no score and no result
does (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionAuto

from helpers import assert_close, gpu_fp32_reference

pytestmark = pytest.mark.gpu


# K^T V grows to N * 40 = 81920 (or more) beyond 65504; outputs, gradients and scores stay below 5200
@pytest.mark.parametrize("b,h,n,dqk,dv", [(1, 1, 2048, 64, 64), (1, 2, 2048, 128, 64), (1, 1, 2048, 256, 64), (1, 2, 2048, 36, 36)])
def test_gradients_of_a_large_state(b, h, n, dqk, dv, gpu_device):
    q, k, v, do = (torch.full((b, h, n, d), s, dtype=torch.float16, device=gpu_device)
                   for d, s in ((dqk, 2.0**-12), (dqk, 1.0), (dv, 40.0), (dv, 2.0**-10)))
    want, grads = gpu_fp32_reference(q, k, v, do, True)
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    out = LinearAttentionAuto.apply(q, k, v)
    out.backward(do)
    assert_close("O", out, want)
    for name, got, w in zip(("dQ", "dK", "dV"), (q.grad, k.grad, v.grad), grads):
        assert_close(name, got, w)
