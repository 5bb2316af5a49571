"""The polynomial score map chunk-wise (fla_poly_attn_chunked_fwd/bwd) against the CPU oracle: two rows, chunk edges, one,
a few (added up on load) and many (scanned) segments, padded widths, other strides (``-m gpu``).  Tolerances as for the
quadratic evaluation of the same operator."""

import pytest
import torch

from flashy_linear_attention_amd.poly import poly_attention_chunked_bwd, poly_attention_chunked_fwd
from oracle import naive

from helpers import assert_close

pytestmark = pytest.mark.gpu

TAYLOR = (1.0, 1.0, 0.5)
OTHER = (0.25, -0.5, 0.75)


@pytest.mark.parametrize("b,h,n,r,dv", [
    (1, 1, 2, 16, 64), (1, 2, 127, 8, 32), (1, 1, 128, 16, 64), (2, 1, 129, 16, 40), (1, 3, 300, 16, 64), (1, 1, 1000, 8, 64),
    (1, 1, 1700, 16, 64), (20, 15, 260, 16, 64),
])
@pytest.mark.parametrize("normalise,coef,transposed", [(False, OTHER, False), (True, TAYLOR, False), (True, TAYLOR, True)])
def test_poly_chunked_vs_oracle(b, h, n, r, dv, normalise, coef, transposed, gpu_device):
    g = torch.Generator().manual_seed(n + r + dv)
    xq, xk = (0.5 * torch.randn(b, h, n, r, generator=g).to(torch.bfloat16) for _ in range(2))
    v, do = (torch.randn(b, h, n, dv, generator=g).to(torch.bfloat16) for _ in range(2))
    leaves = [t.float().requires_grad_(True) for t in (xq, xk, v)]
    want = (naive.poly_linear_attention_normalised(*leaves, coef, 1e-5) if normalise
            else naive.poly_causal_dot_product(*leaves, coef))
    want.backward(do.float())
    ins = [t.to(gpu_device) for t in (xq, xk, v, do)]
    if transposed:
        ins = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in ins]
    a, k, c, d = ins
    out, denom, state = poly_attention_chunked_fwd(a, k, c, coef, normalise, 1e-5)
    grads = poly_attention_chunked_bwd(d, a, k, c, coef, state, *((out, denom) if normalise else ()))
    assert_close("O", out, want.detach())
    for name, got, leaf in zip(("dXq", "dXk", "dV"), grads, leaves):
        # (normalised: dO / n and dn pass through 16-bit storage and the two terms of the score gradient cancel)
        assert_close(name, got, leaf.grad, tol_fro=1e-2, tol_max=5e-2 if normalise else 1e-2)
