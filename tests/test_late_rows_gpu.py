"""Causality of dQ where late rows of k and v are infinite, NaN or merely huge: the outputs and dQ of the rows before are those
of a call without them, bit for bit, in the operators that choose their evaluation by shape (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionAuto, LinearAttentionSmallVHD, PolynomialLinearAttention

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
    # D = 128: one, two, several and many segments; unequal widths; copies with aligned rows
    ("linear", 8, 40, 512, 128, 128), ("linear", 4, 32, 2048, 128, 128), ("linear", 1, 32, 4096, 96, 96), ("linear", 1, 4, 8192, 128, 128),
    ("smallv", 2, 16, 2048, 128, 64), ("auto", 2, 10, 1500, 72, 72), ("auto", 1, 6, 2100, 100, 100), ("smallv", 1, 12, 1024, 91, 64),
    # q and k of more than 128 columns
    ("smallv", 4, 64, 512, 256, 64), ("smallv", 4, 16, 2048, 256, 64), ("smallv", 1, 8, 2048, 160, 32), ("smallv", 1, 20, 2048, 192, 128),
    ("smallv", 2, 3, 4096, 136, 128), ("smallv", 1, 16, 2048, 153, 64), ("auto", 1, 4, 1100, 250, 250),
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


# (forward alone at lengths and head counts that take either evaluation: a single segment per head and several, two column halves)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")], ids=["inf", "-inf", "nan"])
@pytest.mark.parametrize("op,h,n,dqk,dv", [
    ("linear", 2, 512, 64, 64), ("linear", 3, 1024, 64, 64), ("linear", 300, 384, 64, 64), ("linear", 4, 1088, 32, 32),
    ("linear", 130, 320, 128, 128), ("linear", 100, 640, 128, 128), ("smallv", 3, 1024, 128, 64), ("smallv", 2, 2048, 256, 64),
])
def test_a_non_finite_value_keeps_to_its_column(op, h, n, dqk, dv, value, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk + dv)
    q, k, v = (torch.randn(1, h, n, d, generator=gen).bfloat16().to(gpu_device) for d in (dqk, dqk, dv))
    want = OPERATORS[op].apply(q, k, v)
    row, column = 70, dv - 3
    v[:, :, row, column] = value
    got = OPERATORS[op].apply(q, k, v)
    assert not bool(got[:, :, row:, column].isfinite().any())
    assert torch.equal(got[:, :, : row // 32 * 32], want[:, :, : row // 32 * 32])
    others = torch.arange(dv, device=gpu_device) != column
    assert torch.equal(got[..., others], want[..., others])


@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
@pytest.mark.parametrize("late", [float("nan"), float("inf"), 1e9], ids=["nan", "inf", "huge"])
@pytest.mark.parametrize("b,h,n,r,dv", [(4, 70, 512, 16, 64), (4, 32, 1024, 8, 32), (1, 6, 1700, 16, 64), (1, 1, 4096, 16, 48)])
def test_late_rows_do_not_reach_earlier_ones_of_the_polynomial(b, h, n, r, dv, late, normalise, gpu_device):
    gen = torch.Generator().manual_seed(n + r + dv)
    q, k, v, do = (torch.randn(b, h, n, d, generator=gen).bfloat16().to(gpu_device) for d in (r, r, dv, dv))

    def step():
        args = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = PolynomialLinearAttention.apply(*args, 1.0, 1.0, 0.5, normalise, 1e-5)
        return out.detach(), torch.autograd.grad(out, args, do)[0]

    want = step()
    first = n - 40
    k[:, :, first:], v[:, :, first:] = late, late
    rows = first // 32 * 32
    for name, a, w in zip(("O", "dXq"), step(), want):
        assert torch.equal(a[:, :, :rows], w[:, :, :rows]), name
