"""The error against fp64 of the evaluation chosen by shape is that of the quadratic kernels (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionSmallVHD, PolynomialLinearAttention
from flashy_linear_attention_amd import kernels
from flashy_linear_attention_amd.poly import poly_attention_bwd, poly_attention_chunked_fwd, poly_attention_fwd

pytestmark = pytest.mark.gpu

# Both round one factor of every product to bf16 (the scores; within a chunk the scores, beyond it the running state), sum in
# fp32 and round the result, so the errors are alike: at worst the state's rounding is averaged over D terms where the
# scores' are averaged over N, 1 + 1 / D of the squared error for data of one sign (1.016 at D = 32).  The rest of the 3 %
# is the sampling of the two norms.
NO_LARGER = 1.03


def _exact(q, k, v, do):
    q, k, v, do = (t.double() for t in (q, k, v, do))
    a, m = (torch.matmul(x, y.transpose(-2, -1).contiguous()).tril() for x, y in ((q, k), (do, v)))
    return (torch.matmul(a, v), torch.matmul(m, k), torch.matmul(m.transpose(-2, -1).contiguous(), q),
            torch.matmul(a.transpose(-2, -1).contiguous(), do))


def _compare(chosen, other, want):
    for name, got, ref, w in zip(("O", "dQ", "dK", "dV"), chosen, other, want):
        err, bound = (float(torch.linalg.norm(t.double() - w) / torch.linalg.norm(w)) for t in (got, ref))
        assert err <= NO_LARGER * bound, f"{name}: {err:.3e} against {bound:.3e}"


@pytest.mark.parametrize("positive", [False, True], ids=["signed", "positive"])
@pytest.mark.parametrize("h,n,dqk,dv", [
    (4, 2048, 64, 64), (4, 4096, 32, 32), (4, 2048, 128, 128), (4, 2048, 128, 64), (4, 2048, 256, 64), (4, 2048, 256, 128),
    (4, 2048, 192, 128), (4, 2048, 153, 64), (4, 2048, 136, 128),
])
def test_no_larger_than_the_quadratic_kernels(h, n, dqk, dv, positive, gpu_device):
    gen = torch.Generator().manual_seed(dqk + dv)
    q, k, v, do = (torch.randn(1, h, n, d, generator=gen) for d in (dqk, dqk, dv, dv))
    q, k, v, do = ((t.abs() if positive else t).bfloat16().to(gpu_device) for t in (q, k, v, do))
    args = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = (LinearAttention if dqk == dv else LinearAttentionSmallVHD).apply(*args)
    chosen = (out.detach(), *torch.autograd.grad(out, args, do))
    if dqk == dv:
        other = (kernels.linear_flash_wrapper_fwd(q, k, v), *kernels.linear_flash_wrapper_bwd(do, q, k, v))
    else:
        other = (kernels.linear_flash_wrapper_fwd_smallv_hd(q, k, v), *kernels.linear_flash_wrapper_bwd_smallv_hd(do, q, k, v))
    assert any(not torch.equal(a, b) for a, b in zip(chosen, other))  # (chunk-wise, at these sizes)
    _compare(chosen, other, _exact(q, k, v, do))


# from the first lengths that forward alone takes chunk-wise: a single segment per head (257 and 129 heads), several
@pytest.mark.parametrize("positive", [False, True], ids=["signed", "positive"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("h,n,dqk,dv", [
    (257, 320, 64, 64), (129, 320, 128, 128), (520, 320, 32, 32), (2, 768, 64, 64), (4, 1024, 32, 32), (2, 1024, 128, 128), (4, 1024, 128, 64),
])
def test_forward_alone_no_larger_than_the_quadratic_kernels(h, n, dqk, dv, dtype, positive, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk + dv)
    q, k, v = (torch.randn(1, h, n, d, generator=gen) for d in (dqk, dqk, dv))
    # (in fp16 the results, up to 2e5 at 1024 rows of 128 positive columns, would leave its range)
    q, k, v = ((t.abs() if positive else t).mul(s).to(dtype).to(gpu_device) for t, s in ((q, dqk**-0.5), (k, 1.0), (v, 1.0)))
    with torch.no_grad():
        chosen = (LinearAttention if dqk == dv else LinearAttentionSmallVHD).apply(q, k, v)
    other = (kernels.linear_flash_wrapper_fwd if dqk == dv else kernels.linear_flash_wrapper_fwd_smallv_hd)(q, k, v)
    assert not torch.equal(chosen, other)  # (chunk-wise, at these sizes)
    want = torch.matmul(torch.matmul(q.double(), k.double().transpose(-2, -1).contiguous()).tril(), v.double())
    _compare((chosen,), (other,), (want,))


# (0.1 and 0.3 are no bf16 numbers; the second-order part alone; a leading constant)
@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
@pytest.mark.parametrize("coef", [(1.0, 1.0, 0.5), (0.0, 0.0, 0.5), (0.1, 0.3, 0.7)], ids=str)
@pytest.mark.parametrize("h,n,r,dv,scale", [(4, 2048, 16, 64, 1.0), (4, 2048, 16, 64, 0.5), (4, 4096, 8, 32, 1.0), (4, 512, 16, 64, 1.0), (3, 1111, 16, 40, 1.0)])
def test_polynomial_no_larger_than_the_quadratic_kernels(h, n, r, dv, scale, coef, normalise, gpu_device):
    gen = torch.Generator().manual_seed(n + r + dv)
    xq, xk, v, do = ((s * torch.randn(1, h, n, d, generator=gen)).bfloat16().to(gpu_device)
                     for d, s in ((r, scale), (r, scale), (dv, 1.0), (dv, 1.0)))
    args = [t.clone().requires_grad_(True) for t in (xq, xk, v)]
    out = PolynomialLinearAttention.apply(*args, *coef, normalise, 1e-5)
    chosen = (out.detach(), *torch.autograd.grad(out, args, do))
    o, denom = poly_attention_fwd(xq, xk, v, coef, normalise, 1e-5)
    other = (o, *poly_attention_bwd(do, xq, xk, v, coef, *((o, denom) if normalise else ())))
    assert any(not torch.equal(a, b) for a, b in zip(chosen, other))
    exact = [t.double().requires_grad_(True) for t in (xq, xk, v)]
    u = torch.matmul(exact[0], exact[1].transpose(-2, -1).contiguous())
    scores = (coef[0] + coef[1] * u + coef[2] * u * u).tril()
    want = torch.matmul(scores, exact[2])
    n_want = scores.sum(-1) + 1e-5
    if normalise:
        want = want / n_want[..., None]
        # (sums of fp32 scores, as the quadratic kernels' normaliser: a few 1e-7 where nothing cancels)
        got = poly_attention_chunked_fwd(xq, xk, v, coef, True, 1e-5)[1]
        assert float(torch.linalg.norm(got.double() - n_want.detach()) / torch.linalg.norm(n_want.detach())) <= 1e-6
    _compare(chosen, other, (want.detach(), *torch.autograd.grad(want, exact, do.double())))
