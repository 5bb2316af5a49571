"""The plain chunk-wise forward in fp16 where the running state leaves fp16's range and scores and results do not, and where
it is tiny; every padded width, one and several segments (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionSmallVHD
from flashy_linear_attention_amd.chunked import linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference

pytestmark = pytest.mark.gpu


# state elements grow to n * sk * sv: 2e6 in the first scale, 1e-7 in the last
@pytest.mark.parametrize("sq,sk,sv", [(2.0**-14, 30.0, 30.0), (0.05, 1.0, 1.0), (30.0, 2.0**-13, 2.0**-13)])
@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (1, 3, 2060, 32, 32), (1, 40, 2048, 64, 64), (3, 5, 1999, 128, 128), (1, 260, 513, 96, 96), (1, 2, 2048, 128, 64),
    (1, 2, 700, 64, 128), (2, 2, 1500, 64, 32), (1, 1, 300, 24, 16),
])
def test_state_beyond_the_range(b, h, n, dqk, dv, sq, sk, sv, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk)
    q, k = (torch.rand(b, h, n, dqk, generator=gen).add(0.5).mul(s).half().to(gpu_device) for s in (sq, sk))
    v = torch.rand(b, h, n, dv, generator=gen).add(0.5).mul(sv).half().to(gpu_device)
    want, _ = gpu_fp32_reference(q, k, v, None, False)
    out = linear_attention_chunked_fwd(q, k, v)
    inside = want.abs() < 6e4
    assert inside.float().mean() > 0.5
    assert_close("O", torch.where(inside, out.float(), 0.0), torch.where(inside, want, 0.0))
    op = LinearAttention if dqk == dv else LinearAttentionSmallVHD
    if n % 64 == 0 and dv & (dv - 1) == 0 and dv <= dqk:
        with torch.no_grad():
            got = op.apply(q, k, v)
        assert_close("O, evaluation chosen by shape", torch.where(inside, got.float(), 0.0), torch.where(inside, want, 0.0))


# an infinite or NaN value: the other columns' state elements, 1e5 and more beyond the range, keep their scale (widths up to 64: one
# segment and several; 128: several)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")], ids=["inf", "-inf", "nan"])
@pytest.mark.parametrize("h,n,dqk,dv", [(3, 1024, 32, 32), (2, 1024, 64, 64), (300, 512, 64, 64), (2, 1024, 128, 128), (128, 1024, 96, 96), (2, 1024, 128, 64)])
def test_a_non_finite_value_beside_a_state_beyond_the_range(h, n, dqk, dv, value, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk)
    q, k = (torch.rand(1, h, n, dqk, generator=gen).add(0.5).mul(s).half().to(gpu_device) for s in (2.0**-14, 20.0))
    v = torch.rand(1, h, n, dv, generator=gen).add(0.5).mul(20.0).half().to(gpu_device)
    want, _ = gpu_fp32_reference(q, k, v, None, False)
    v[:, :, 3, 1] = value
    with torch.no_grad():
        picked = (LinearAttention if dqk == dv else LinearAttentionSmallVHD).apply(q, k, v)
    for out in (linear_attention_chunked_fwd(q, k, v), picked):
        assert not bool(out[:, :, 3:, 1].isfinite().any())
        keep = torch.arange(dv, device=gpu_device) != 1
        assert_close("O", out[..., keep], want[..., keep])
