"""Which workgroup takes which part of which head (csrc/fla_tri_fast.h, xcd_item): a head count that is no multiple of 8 (runs of
consecutive parts, or whole heads where no XCD gets more than 16 parts), a multiple of 8 (every eighth head) and, with rows that end
inside a 128-byte line in (B, N, H, D) storage, a multiple of 16 (pairs of neighbours) -- in every kernel that goes by it, so that a
part that no workgroup takes would show (``-m gpu``; a part taken twice leaves the same results, and the launch-plan tests
enumerate the map on the CPU)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionChunked, LinearAttentionNormalised, PolynomialLinearAttention
from oracle import naive

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


def _bnhd(t):
    return t.transpose(1, 2).contiguous().transpose(1, 2)


# (the walks at padded widths 32, 64 and 128, both sides wide, and the 256-row chunks with states in memory: 250 columns)
@pytest.mark.parametrize("width", [32, 40, 64, 96, 160, 250])
@pytest.mark.parametrize("heads", [2, 12, 16, 24, 48])
def test_every_part_of_every_head(heads, width, gpu_device):
    n = 1000 if width <= 128 else 777
    q, k, v, dy = (_bnhd(t.to(gpu_device)) for t in reference_style_inputs(1, heads, n, width, width, torch.bfloat16, seed=heads))
    want_o, want_g = gpu_fp32_reference(q, k, v, dy, True)
    qg, kg, vg = (t.detach().requires_grad_(True) for t in (q, k, v))
    out = LinearAttentionChunked.apply(qg, kg, vg)
    out.backward(dy)
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), (qg.grad, kg.grad, vg.grad), want_g):
        assert_close(name, got, want)


# (128 columns, four heads: 16 parts each, the most that stay together, and 17)
@pytest.mark.parametrize("n", [1024, 1025])
def test_either_side_of_whole_heads(n, gpu_device):
    q, k, v, dy = (_bnhd(t.to(gpu_device)) for t in reference_style_inputs(1, 4, n, 128, 128, torch.bfloat16, seed=n))
    want_o, want_g = gpu_fp32_reference(q, k, v, dy, True)
    qg, kg, vg = (t.detach().requires_grad_(True) for t in (q, k, v))
    out = LinearAttentionChunked.apply(qg, kg, vg)
    out.backward(dy)
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), (qg.grad, kg.grad, vg.grad), want_g):
        assert_close(name, got, want)


# (7 heads, nearly one per XCD: up to 20 parts of 128 columns whole, whose totals the walks add up, and 21 in runs; 9 heads over 64
# columns: a forward alone whole up to 2 x 16 parts on an XCD, and 2 x 17; 15 heads, nearly two per XCD)
@pytest.mark.parametrize("heads,n,width", [(7, 1280, 128), (7, 1281, 128), (9, 2048, 64), (9, 2049, 64), (15, 2500, 64)])
def test_either_side_of_more_parts(heads, n, width, gpu_device):
    q, k, v, dy = (_bnhd(t.to(gpu_device)) for t in reference_style_inputs(1, heads, n, width, width, torch.bfloat16, seed=n))
    want_o, want_g = gpu_fp32_reference(q, k, v, dy, True)
    assert_close("O alone", LinearAttentionChunked.apply(q, k, v), want_o)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = LinearAttentionChunked.apply(*leaves)
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, leaves, dy), want_g):
        assert_close(name, got, want)


@pytest.mark.parametrize("heads", [3, 16, 20])
def test_the_normalised_backward_and_the_polynomial_map(heads, gpu_device):
    q, k, v, dy = (_bnhd(t.to(gpu_device)) for t in reference_style_inputs(1, heads, 900, 32, 32, torch.bfloat16, seed=7))
    a = [t.detach().requires_grad_(True) for t in (q, k, v)]
    want = naive.linear_attention_normalised(*(t.float() for t in a), eps=1e-5)
    want_g = torch.autograd.grad(want, a, dy.float())
    out = LinearAttentionNormalised.apply(*a, 1e-5, True)
    assert_close("out", out, want.detach())
    # (one bf16 ulp of the normaliser's cancelling terms is 2.9e-2 of the largest gradient)
    for name, got, w in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, a, dy), want_g):
        assert_close(name, got, w, tol_max=5e-2)

    gen = torch.Generator().manual_seed(heads)
    x = [_bnhd(t.to(gpu_device).bfloat16()) for t in (0.5 * torch.randn(2, 1, heads, 900, 16, generator=gen)).unbind()]
    v, dy = (_bnhd(t.to(gpu_device).bfloat16()) for t in torch.randn(2, 1, heads, 900, 64, generator=gen).unbind())
    a = [t.detach().requires_grad_(True) for t in (*x, v)]
    out = PolynomialLinearAttention.apply(*a, 1.0, 1.0, 0.5)
    assert_close("O", out, naive.poly_causal_dot_product(*(t.detach().float() for t in a), (1.0, 1.0, 0.5)))
    want_g = naive.poly_causal_dot_product_grads(*(t.detach().float() for t in a), dy.float(), (1.0, 1.0, 0.5))
    for name, got, w in zip(("dXq", "dXk", "dV"), torch.autograd.grad(out, a, dy), want_g):
        assert_close(name, got, w)
