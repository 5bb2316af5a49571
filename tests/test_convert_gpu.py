"""fp32 operands under autocast: the one-launch copies to bf16 and of the gradients back to fp32, at lengths around the
copy kernel's eight-element and 2048-element steps, against PyTorch's own casts (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import FeatureMapLinearAttention, LinearAttentionAuto, LinearAttentionNormalised

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,n,d", [(1, 1, 1, 1), (1, 1, 3, 5), (2, 1, 64, 32), (1, 3, 129, 40), (2, 2, 333, 64)])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("op", ["auto", "normalised", "feature"])
def test_autocast_equals_casting_by_hand(b, h, n, d, transposed, op, gpu_device):
    g = torch.Generator().manual_seed(n + d)
    ins = [torch.rand(b, h, n, d, generator=g).to(gpu_device) for _ in range(4)]
    if transposed:
        ins = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in ins]
    apply = {"auto": LinearAttentionAuto.apply, "normalised": lambda *a: LinearAttentionNormalised.apply(*a, 1e-5, True),
             "feature": lambda *a: FeatureMapLinearAttention.apply(*a, "elu1")}[op]
    do = ins[3].bfloat16()
    wide = [t.clone().requires_grad_(True) for t in ins[:3]]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = apply(*wide)
    grads = torch.autograd.grad(out, wide, do)
    narrow = [t.bfloat16().requires_grad_(True) for t in ins[:3]]
    want = apply(*narrow)
    want_grads = torch.autograd.grad(want, narrow, do)
    assert out.dtype == torch.bfloat16 and torch.equal(out, want)
    for got, w in zip(grads, want_grads):
        assert got.dtype == torch.float32 and torch.equal(got, w.float())  # (one rounding, then exact)
