"""LinearAttentionNormalised chooses the evaluation of forward alone by shape when not told: both sides of the thresholds, with
and without gradients, natively and through the Python forward, against the fp64 recipe (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionNormalised, _lib
from flashy_linear_attention_amd.normalised import _forward_prefers_chunked

from helpers import assert_close

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _recipe(q, k, v, g):
    q, k, v = (t.detach().double().requires_grad_() for t in (q, k, v))
    out = (torch.tril(q @ k.transpose(-1, -2)) @ v) / ((q * k.cumsum(-2)).sum(-1, keepdim=True) + EPS)
    return (out, *torch.autograd.grad(out, (q, k, v), g.double()))


# (B, H, N, D, chunk-wise without gradients): below and from each threshold, ragged lengths, a single segment per head
@pytest.mark.parametrize("b,h,n,d,chunked", [
    (1, 2, 1023, 64, False), (1, 2, 1024, 64, True), (1, 1, 1500, 128, False), (1, 1, 2049, 72, True), (2, 2, 4096, 32, True),
    (1, 30, 1500, 64, True), (1, 2, 257, 128, False), (1, 8, 2900, 128, True), (1, 1, 2100, 100, False),
    (2, 65, 320, 128, True), (1, 128, 320, 128, False), (1, 260, 257, 64, True),
])
def test_choice_and_results(b, h, n, d, chunked, gpu_device):
    gen = torch.Generator().manual_seed(n + d)
    q, k = (torch.nn.functional.softplus(torch.randn(b, h, n, d, generator=gen)).to(gpu_device).bfloat16() for _ in range(2))
    v, g = (torch.randn(b, h, n, d, generator=gen).to(gpu_device).bfloat16() for _ in range(2))
    assert _forward_prefers_chunked(q, v) == chunked
    assert not _lib.query("fla_normalised_forward_prefers_chunked", b, h, n, d, d, 1)  # fp16
    want = _recipe(q, k, v, g)
    with torch.no_grad():
        out = LinearAttentionNormalised.apply(q, k, v, EPS)
    assert_close("out, no gradients", out, want[0].float())
    assert torch.equal(out, LinearAttentionNormalised.apply(q, k, v, EPS, chunked))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    for apply in (LinearAttentionNormalised.apply, super(LinearAttentionNormalised, LinearAttentionNormalised).apply):
        out = apply(*leaves, EPS)
        assert_close("out", out, want[0].float())
        for name, got, ref in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, leaves, g), want[1:]):
            # (the bound of the operator's own tests: one bf16 ulp of the cancelling terms is 2.9e-2 of the largest gradient)
            assert_close(name, got, ref.float(), tol_fro=1e-2, tol_max=5e-2)
