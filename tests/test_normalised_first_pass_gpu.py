"""The normalised backward's first pass (dO, dn and the segments' totals in one kernel) and the walks behind it: one segment, two,
a few whose totals the walk adds up, many that are scanned, gradients whose rows allow no 16-byte loads, backward without
forward's state -- against the fp64 recipe (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.normalised import linear_attention_normalised_bwd, linear_attention_normalised_fwd

from helpers import assert_close

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _recipe(q, k, v, g):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    out = (torch.tril(q @ k.transpose(-1, -2)) @ v) / ((q * k.cumsum(-2)).sum(-1, keepdim=True) + EPS)
    return (out, *torch.autograd.grad(out, (q, k, v), g.double()))


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16), ids=("bf16", "fp16"))
# chunks of 128 rows up to 64 columns, of 64 above; as many segments as keep 512 (256) workgroups busy
@pytest.mark.parametrize("b,h,n,d,odd_rows", [
    (1, 520, 300, 32, False), (2, 100, 600, 64, False), (1, 3, 700, 64, True), (1, 1, 4300, 48, False), (4, 60, 385, 16, False),
    (1, 260, 330, 128, False), (1, 100, 400, 96, True), (1, 20, 900, 128, False), (1, 2, 2100, 72, False), (1, 128, 257, 128, False),
])
def test_gradients(b, h, n, d, odd_rows, dtype, gpu_device):
    gen = torch.Generator().manual_seed(n + d)
    q, k = (torch.nn.functional.softplus(torch.randn(b, h, n, d, generator=gen)).to(gpu_device, dtype) for _ in range(2))
    v, g = (torch.randn(b, h, n, d, generator=gen).to(gpu_device, dtype) for _ in range(2))
    if odd_rows:  # rows of d + 1 elements, the first of them not g's
        rows = torch.zeros(b, h, n, d + 1, device=gpu_device, dtype=dtype)
        rows[..., 1:] = g
        g = rows[..., 1:]
    want = _recipe(q, k, v, g)
    out, denom, state = linear_attention_normalised_fwd(q, k, v, EPS, True, want_state=True)
    assert_close("out", out, want[0].float())
    for kept in (state, None):
        grads = linear_attention_normalised_bwd(g, q, k, v, out, denom, True, kept)
        for name, got, ref in zip(("dQ", "dK", "dV"), grads, want[1:]):
            # (the bound of the operator's own tests: one bf16 ulp of the cancelling terms is 2.9e-2 of the largest gradient)
            assert_close(name, got, ref.float(), tol_fro=1e-2, tol_max=5e-2)
