"""The polynomial score map chunk-wise with several chunks in a segment: one, two and three of them per totals workgroup, segments
that the walks add up and segments that are scanned, against fp64 (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.poly import poly_attention_chunked_bwd, poly_attention_chunked_fwd

from helpers import assert_close

pytestmark = pytest.mark.gpu
COEF, EPS = (0.25, -0.5, 0.75), 1e-5


# (B H, N): 256 workgroups at a time, chunks of 128 rows -> segments x chunks
@pytest.mark.parametrize("bh,n,r", [(64, 1536, 16), (100, 700, 16), (20, 3300, 8), (33, 1700, 16), (128, 500, 16),
                                     (12, 2500, 16), (10, 5500, 8)],
                         ids=["4x3", "2x3", "9x3", "7x2", "2x2", "20x1", "22x2, scanned"])
@pytest.mark.parametrize("normalise", [False, True])
def test_segments_of_several_chunks(bh, n, r, normalise, gpu_device):
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    xq, xk = (0.5 * torch.randn(1, bh, n, r, generator=gen, device=gpu_device).bfloat16() for _ in range(2))
    v, do = (torch.randn(1, bh, n, 64, generator=gen, device=gpu_device).bfloat16() for _ in range(2))
    coef = (1.0, 1.0, 0.5) if normalise else COEF
    out, denom, state = poly_attention_chunked_fwd(xq, xk, v, coef, normalise, EPS)
    got = (out, *poly_attention_chunked_bwd(do, xq, xk, v, coef, state, *((out, denom) if normalise else ())))
    for h in (0, bh // 2, bh - 1):
        a, b, c = (t[0, h].double().requires_grad_(True) for t in (xq, xk, v))
        u = a @ b.t()
        s = (coef[0] + coef[1] * u + coef[2] * u * u).tril()
        want = s @ c
        if normalise:
            want = want / (s.sum(-1, keepdim=True) + EPS)
        want = (want, *torch.autograd.grad(want, (a, b, c), do[0, h].double()))
        for name, x, ref in zip(("O", "dXq", "dXk", "dV"), got, want):
            # (the bounds of test_poly_chunked_gpu.py: dO / n and dn pass through 16 bits and two terms of a score gradient cancel)
            assert_close(f"{name} of head {h}", x[0, h], ref.detach().float(), tol_fro=1e-2, tol_max=5e-2 if normalise else 1e-2)
