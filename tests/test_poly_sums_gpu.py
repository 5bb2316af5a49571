"""dq's walk of the polynomial map adds up the reverse walk's segment totals from three segments per head to twenty; two and twenty-one
have a kernel of their own for them: with and without the normaliser, against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import PolynomialLinearAttention
from oracle import naive

from helpers import assert_close

pytestmark = pytest.mark.gpu

COEF = (1.0, 1.0, 0.5)


# (heads, N: 256 / heads segments of one chunk of 128 rows or more, the last one ragged; r, D_v)
@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
@pytest.mark.parametrize("h,n,r,dv", [(100, 500, 16, 64), (85, 3 * 128 - 5, 16, 64), (40, 1500, 8, 40), (12, 20 * 128 - 3, 16, 64),
                                      (12, 21 * 128 - 3, 16, 32)])
def test_gradients(h, n, r, dv, normalise, gpu_device):
    gen = torch.Generator().manual_seed(n + r)
    xq, xk = (0.5 * torch.randn(2, 1, h, n, r, generator=gen)).to(gpu_device).bfloat16().unbind()
    v, do = torch.randn(2, 1, h, n, dv, generator=gen).to(gpu_device).bfloat16().unbind()
    leaves = [t.clone().requires_grad_(True) for t in (xq, xk, v)]
    out = PolynomialLinearAttention.apply(*leaves, *COEF, normalise, 1e-5)
    grads = torch.autograd.grad(out, leaves, do)
    exact = [t.float().requires_grad_(True) for t in (xq, xk, v)]
    want = naive.poly_linear_attention_normalised(*exact, COEF, 1e-5) if normalise else naive.poly_causal_dot_product(*exact, COEF)
    assert_close("O", out, want.detach())
    # (the bound of the operator's own tests where the normaliser's terms cancel: one bf16 ulp of them)
    for name, got, w in zip(("dXq", "dXk", "dV"), grads, torch.autograd.grad(want, exact, do.float())):
        assert_close(name, got, w, tol_max=5e-2 if normalise else 1e-2)
