"""128 to 256 rows: the errors against fp64 of the evaluation chosen above the lines for padded widths that differ and for q and k above 128
columns, beside the quadratic kernels' (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionSmallVHD, kernels

from test_chosen_accuracy_gpu import _compare, _exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("positive", [False, True], ids=["signed", "positive"])
@pytest.mark.parametrize("bh,n,dqk,dv", [(257, 128, 128, 64), (203, 256, 72, 32), (300, 192, 128, 32), (60, 256, 256, 64), (256, 128, 192, 32),
                                         (64, 128, 160, 160), (48, 192, 256, 256)])
def test_no_larger_than_the_quadratic_kernels(bh, n, dqk, dv, positive, gpu_device):
    gen = torch.Generator(device=gpu_device).manual_seed(n + dqk + dv)
    q, k, v, do = (torch.randn(1, bh, n, d, generator=gen, device=gpu_device) for d in (dqk, dqk, dv, dv))
    q, k, v, do = ((t.abs() if positive else t).bfloat16() for t in (q, k, v, do))
    args = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = (LinearAttention if dqk == dv else LinearAttentionSmallVHD).apply(*args)
    chosen = (out.detach(), *torch.autograd.grad(out, args, do))
    other = ((kernels.linear_flash_wrapper_fwd(q, k, v), *kernels.linear_flash_wrapper_bwd(do, q, k, v)) if dqk == dv else
             (kernels.linear_flash_wrapper_fwd_smallv_hd(q, k, v), *kernels.linear_flash_wrapper_bwd_smallv_hd(do, q, k, v)))
    assert any(not torch.equal(a, b) for a, b in zip(chosen, other))  # (chunk-wise, at these sizes)
    _compare(chosen, other, _exact(q, k, v, do))
