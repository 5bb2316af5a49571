"""The normalised chunk-wise backward up to 64 columns forms dO = g / n where it is used when g's rows are aligned and dO is of more
than 10 MiB, and ahead of the walk otherwise (csrc/fla_chunk_walk.h, WalkParams::gn): the same bits either way (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import FeatureMapLinearAttention, LinearAttentionNormalised

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("h,n,d", [(1, 257, 64), (3, 1000, 40), (24, 900, 32), (300, 384, 64), (2, 4100, 24), (170, 1000, 40), (700, 384, 32), (500, 520, 24)])
@pytest.mark.parametrize("mapped", [False, True], ids=["plain", "elu1"])
def test_aligned_and_unaligned_rows_of_g(mapped, h, n, d, dtype, gpu_device):
    gen = torch.Generator().manual_seed(n + d)
    q, k, v = ((torch.nn.functional.softplus(t) if not mapped and i < 2 else t).to(gpu_device, dtype).requires_grad_(True)
               for i, t in enumerate(torch.randn(3, 1, h, n, d, generator=gen).unbind()))
    g = torch.randn(1, h, n, d, generator=gen).to(gpu_device, dtype)
    out = (FeatureMapLinearAttention.apply(q, k, v, "elu1", True, 1e-5) if mapped
           else LinearAttentionNormalised.apply(q, k, v, 1e-5, True))
    want = torch.autograd.grad(out, (q, k, v), g, retain_graph=True)
    odd = torch.empty(1, h, n, d + 1, dtype=dtype, device=gpu_device)[..., 1:]  # (rows that start at any element)
    strided = torch.empty(1, n, h, d, dtype=dtype, device=gpu_device).transpose(1, 2)
    for other in (odd.copy_(g), strided.copy_(g)):
        for name, a, b in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, (q, k, v), other, retain_graph=True), want):
            assert torch.equal(a, b), name
    ones = torch.autograd.grad(out, (q, k, v), torch.ones_like(g), retain_graph=True)
    for a, b in zip(torch.autograd.grad(out.sum(), (q, k, v)), ones):  # (g expanded from a number: strides of zero)
        assert torch.equal(a, b)
