"""Errors against fp64 of the polynomial map over two halves of v, and of more than 16 columns of q and k, beside the quadratic kernels', over many
heads (a few rows of a few heads are a sample of roundings) (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import PolynomialLinearAttention
from flashy_linear_attention_amd.poly import (poly_attention_bwd, poly_attention_chunked_bwd, poly_attention_chunked_fwd,
                                              poly_attention_fwd)

from test_chosen_accuracy_gpu import NO_LARGER

pytestmark = pytest.mark.gpu

EPS = 1e-5


def _draw(h, n, r, dv, device):
    gen = torch.Generator(device=device).manual_seed(n + r + dv)
    return ([0.5 * torch.randn(1, h, n, r, generator=gen, device=device).bfloat16() for _ in range(2)]
            + [torch.randn(1, h, n, dv, generator=gen, device=device).bfloat16() for _ in range(2)])


def _quadratic(xq, xk, v, do, coef, normalise):
    out, denom = poly_attention_fwd(xq, xk, v, coef, normalise, EPS)
    return (out, *poly_attention_bwd(do, xq, xk, v, coef, *((out, denom) if normalise else ())))


def _ratios(got, quad, xq, xk, v, do, coef, normalise, heads):
    a, k, c = (t[:, -heads:].detach().double().requires_grad_(True) for t in (xq, xk, v))
    u = torch.matmul(a, k.transpose(-2, -1).contiguous())
    s = (coef[0] + coef[1] * u + coef[2] * u * u).tril()
    want = torch.matmul(s, c)
    if normalise:
        want = want / (s.sum(-1, keepdim=True) + EPS)
    want = (want.detach(), *torch.autograd.grad(want, (a, k, c), do[:, -heads:].double()))
    return [float(torch.linalg.norm(x[:, -heads:].double() - w) / torch.linalg.norm(y[:, -heads:].double() - w))
            for x, y, w in zip(got, quad, want)]


# Up to one chunk of 128 rows the quadratic evaluation rounds a score's gradient and the result, each once and alike (for signed data their
# errors add up to sqrt 2 of one): a half's, a partial sum, may not be rounded, and the result's rounding, 0.71 of it, is what is left.
@pytest.mark.parametrize("coef", [(1.0, 1.0, 0.5), (0.25, -0.5, 0.75)], ids=str)
@pytest.mark.parametrize("h,n,r,dv", [(1024, 2, 16, 72), (1024, 2, 8, 128), (256, 8, 16, 128), (64, 32, 8, 96), (32, 100, 16, 128), (32, 128, 24, 128),
                                      (256, 3, 32, 72)])
def test_partial_sums_are_not_rounded(h, n, r, dv, coef, gpu_device):
    xq, xk, v, do = _draw(h, n, r, dv, gpu_device)
    out, _, state = poly_attention_chunked_fwd(xq, xk, v, coef)
    got = (out, *poly_attention_chunked_bwd(do, xq, xk, v, coef, state))
    ratios = _ratios(got, _quadratic(xq, xk, v, do, coef, False), xq, xk, v, do, coef, False, h)
    assert ratios[1] <= 0.85 and ratios[2] <= 0.85, ratios


@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
@pytest.mark.parametrize("coef", [(1.0, 1.0, 0.5), (0.1, 0.3, 0.7)], ids=str)
@pytest.mark.parametrize("h,n,r,dv", [(512, 2, 16, 120), (48, 40, 8, 72), (16, 1100, 16, 128), (16, 1100, 8, 96), (8, 3000, 16, 128), (4, 4500, 32, 64),
                                      (4, 4500, 24, 128)])
def test_no_larger_than_the_quadratic_kernels(h, n, r, dv, coef, normalise, gpu_device):
    xq, xk, v, do = _draw(h, n, r, dv, gpu_device)
    args = [t.clone().requires_grad_(True) for t in (xq, xk, v)]
    out = PolynomialLinearAttention.apply(*args, *coef, normalise, EPS)
    got = (out.detach(), *torch.autograd.grad(out, args, do))
    quad = _quadratic(xq, xk, v, do, coef, normalise)
    assert any(not torch.equal(x, y) for x, y in zip(got, quad))  # (chunk-wise, at these sizes)
    for name, ratio in zip(("O", "dXq", "dXk", "dV"), _ratios(got, quad, xq, xk, v, do, coef, normalise, h)):
        assert ratio <= NO_LARGER, f"{name}: {ratio:.3f}"
