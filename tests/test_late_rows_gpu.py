"""Causality of dQ where late rows of k and v are infinite, NaN or merely huge: the outputs and dQ of the rows before are those
of a call without them, bit for bit, in the operators that choose their evaluation by shape (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionAuto, LinearAttentionSmallVHD

pytestmark = pytest.mark.gpu

OPERATORS = {"linear": LinearAttention, "smallv": LinearAttentionSmallVHD, "auto": LinearAttentionAuto}


def _step(op, q, k, v, do):
    q, k, v = (t.clone().requires_grad_(True) for t in (q, k, v))
    out = OPERATORS[op].apply(q, k, v)
    out.backward(do)
    return out.detach(), q.grad


# (one, two, several and many segments per head)
@pytest.mark.parametrize("late", [float("nan"), float("inf"), 1e30], ids=["nan", "inf", "huge"])
@pytest.mark.parametrize("op,b,h,n,dqk,dv", [
    ("linear", 4, 160, 512, 64, 64), ("linear", 4, 64, 1024, 64, 64), ("linear", 1, 16, 8192, 32, 32), ("linear", 1, 4, 16384, 64, 64),
    ("smallv", 1, 48, 1024, 64, 32), ("auto", 1, 30, 2200, 40, 40), ("auto", 2, 2, 2500, 36, 36),
])
def test_late_rows_do_not_reach_earlier_ones(op, b, h, n, dqk, dv, late, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk + dv)
    q, k, v, do = (torch.randn(b, h, n, d, generator=gen).bfloat16().to(gpu_device) for d in (dqk, dqk, dv, dv))
    want = _step(op, q, k, v, do)
    first = n - 40
    k[:, :, first:], v[:, :, first:] = late, late
    got = _step(op, q, k, v, do)
    rows = first // 32 * 32  # (the score blocks on the diagonal are 32 rows: a masked score times a late row)
    for name, a, w in zip(("O", "dQ"), got, want):
        assert torch.equal(a[:, :, :rows], w[:, :, :rows]), name
