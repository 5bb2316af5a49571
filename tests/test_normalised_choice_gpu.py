"""LinearAttentionNormalised chooses the evaluation by shape when not told: both sides of the thresholds, with and without
gradients, natively and through the Python forward, against the fp64 recipe (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionNormalised, _lib
from flashy_linear_attention_amd.normalised import _prefers_chunked

from helpers import assert_close

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _recipe(q, k, v, g):
    q, k, v = (t.detach().double().requires_grad_() for t in (q, k, v))
    out = (torch.tril(q @ k.transpose(-1, -2)) @ v) / ((q * k.cumsum(-2)).sum(-1, keepdim=True) + EPS)
    return (out, *torch.autograd.grad(out, (q, k, v), g.double()))


# (B, H, N, D, chunk-wise with gradients, chunk-wise without): below and from each threshold, ragged lengths
@pytest.mark.parametrize("b,h,n,d,with_grad,without", [
    (1, 2, 1023, 64, False, False), (1, 2, 1024, 64, False, True), (1, 1, 1500, 128, False, False), (1, 1, 2049, 72, False, True),
    (2, 2, 4096, 32, True, True), (1, 30, 1500, 64, True, True), (1, 2, 257, 128, False, False),
    (1, 8, 2900, 128, True, True), (1, 1, 2100, 100, False, False),
])
def test_choice_and_results(b, h, n, d, with_grad, without, gpu_device):
    gen = torch.Generator().manual_seed(n + d)
    q, k = (torch.nn.functional.softplus(torch.randn(b, h, n, d, generator=gen)).to(gpu_device).bfloat16() for _ in range(2))
    v, g = (torch.randn(b, h, n, d, generator=gen).to(gpu_device).bfloat16() for _ in range(2))
    assert (_prefers_chunked(q, v, True), _prefers_chunked(q, v, False)) == (with_grad, without)
    assert not _lib.query("fla_normalised_prefers_chunked", b, h, n, d, d, 1, 0)  # fp16
    want = _recipe(q, k, v, g)
    assert_close("out, no gradients", LinearAttentionNormalised.apply(q, k, v, EPS), want[0].float())
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    for apply in (LinearAttentionNormalised.apply, super(LinearAttentionNormalised, LinearAttentionNormalised).apply):
        out = apply(*leaves, EPS)
        assert_close("out", out, want[0].float())
        for name, got, ref in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, leaves, g), want[1:]):
            # (the bound of the operator's own tests: one bf16 ulp of the cancelling terms is 2.9e-2 of the largest gradient)
            assert_close(name, got, ref.float(), tol_fro=1e-2, tol_max=5e-2)
