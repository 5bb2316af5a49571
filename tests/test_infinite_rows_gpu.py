"""Infinite, NaN and huge rows where the polynomial map runs as two halves of v or as three parts of q and k, and where odd widths run on
copies; the polynomial map's fp32 gradients under autocast over two halves (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttention, LinearAttentionSmallVHD, PolynomialLinearAttention, _lib

from helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
@pytest.mark.parametrize("late", [float("nan"), float("inf"), 1e9], ids=["nan", "inf", "huge"])
# (one chunk; several segments that are added up, a single one, many that are scanned; halves of q and k over one and two of v)
@pytest.mark.parametrize("b,h,n,r,dv", [(2, 3, 100, 16, 120), (1, 6, 1700, 16, 128), (2, 16, 900, 8, 72), (3, 100, 800, 16, 128), (1, 1, 3300, 8, 96),
                                        (1, 2, 9000, 32, 64), (1, 1, 4300, 24, 128)])
def test_late_rows_do_not_reach_earlier_ones_of_the_polynomial(b, h, n, r, dv, late, normalise, gpu_device):
    assert _lib.query("fla_poly_attn_operator_prefers_chunked", b, h, n, r, dv, 0, 1, int(normalise))
    gen = torch.Generator(device=gpu_device).manual_seed(n + r + dv)
    q, k, v, do = (torch.randn(b, h, n, d, generator=gen, device=gpu_device).bfloat16() for d in (r, r, dv, dv))

    def step():
        args = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = PolynomialLinearAttention.apply(*args, 1.0, 1.0, 0.5, normalise, 1e-5)
        return out.detach(), torch.autograd.grad(out, args, do)[0]

    want = step()
    first = n - 40
    k[:, :, first:], v[:, :, first:] = late, late
    rows = first // 32 * 32  # (the score blocks on the diagonal are 32 rows: a masked score times a late row)
    for name, a, w in zip(("O", "dXq"), step(), want):
        assert torch.equal(a[:, :, :rows], w[:, :, :rows]), name


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")], ids=["inf", "-inf", "nan"])
@pytest.mark.parametrize("h,n,r,dv", [(3, 1700, 16, 128), (2, 100, 16, 120), (1, 16384, 32, 64)])
def test_a_non_finite_value_keeps_to_its_column_of_the_polynomial(h, n, r, dv, value, gpu_device):
    gen = torch.Generator(device=gpu_device).manual_seed(n + dv)
    q, k, v = (0.5 * torch.randn(1, h, n, d, generator=gen, device=gpu_device).bfloat16() for d in (r, r, dv))
    want = PolynomialLinearAttention.apply(q, k, v, 1.0, 1.0, 0.5, False, 1e-5)
    row, column = 70, dv - 3
    v[:, :, row, column] = value
    got = PolynomialLinearAttention.apply(q, k, v, 1.0, 1.0, 0.5, False, 1e-5)
    assert not bool(got[:, :, row:, column].isfinite().any())
    assert torch.equal(got[:, :, : row // 32 * 32], want[:, :, : row // 32 * 32])
    others = torch.arange(dv, device=gpu_device) != column
    assert torch.equal(got[..., others], want[..., others])


@pytest.mark.parametrize("b,h,n,r,dv", [(1, 3, 900, 16, 128), (2, 1, 100, 8, 120), (1, 1, 4300, 32, 72)])
@pytest.mark.parametrize("normalise", [False, True], ids=["plain", "normalised"])
def test_autocast_over_two_halves(b, h, n, r, dv, normalise, gpu_device):
    """fp32 tensors: the results are those of the bf16 call, the gradients the same sums unrounded."""
    gen = torch.Generator(device=gpu_device).manual_seed(n + dv)
    wide = [0.5 * torch.randn(b, h, n, d, generator=gen, device=gpu_device) for d in (r, r, dv)]
    do = torch.randn(b, h, n, dv, generator=gen, device=gpu_device).bfloat16()

    def step(tensors, amp):
        args = [t.detach().requires_grad_(True) for t in tensors]
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            out = PolynomialLinearAttention.apply(*args, 1.0, 1.0, 0.5, normalise, 1e-5)
        return out.detach(), torch.autograd.grad(out, args, do)

    out, grads = step(wide, True)
    other, narrow = step([t.bfloat16() for t in wide], False)
    assert torch.equal(out, other)
    for name, x, y in zip(("dXq", "dXk", "dV"), grads, narrow):
        assert x.dtype == torch.float32 and y.dtype == torch.bfloat16
        assert torch.equal(x.bfloat16(), y), name
        assert_close(name, x, y.float(), tol_fro=4e-3, tol_max=4e-3)  # (one rounding to bf16)


@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("h,n,dqk,dv", [(3, 512, 100, 100), (2, 576, 20, 20), (4, 320, 153, 64), (2, 192, 250, 250)])
def test_a_non_finite_value_keeps_to_its_column_of_the_copies(h, n, dqk, dv, value, gpu_device):
    on_copies = [_lib.query("fla_linear_attn_operator_prefers_copies", 1, h, n, dqk, dv, backward) for backward in (0, 1)]
    assert on_copies == [int(dqk > 20), 1]
    op = LinearAttention if dqk == dv else LinearAttentionSmallVHD
    gen = torch.Generator(device=gpu_device).manual_seed(n + dv)
    q, k, v, do = (torch.randn(1, h, n, d, generator=gen, device=gpu_device).mul(0.3).half() for d in (dqk, dqk, dv, dv))

    def step():
        args = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
        out = op.apply(*args)
        return (out.detach(), *torch.autograd.grad(out, args, do))

    want = step()
    row, column = n - 70, dv - 3
    others = torch.arange(dv, device=gpu_device) != column
    rows = row // 128 * 128  # (row tiles of up to 128: a masked score times a late row)
    do[:, :, row, column] = value
    got = step()  # (an element of dO: its column of dV, and dQ of its own row)
    assert torch.equal(got[0], want[0]) and torch.equal(got[3][..., others], want[3][..., others])
    assert torch.equal(got[1][:, :, :rows], want[1][:, :, :rows]) and not bool(got[3][:, :, :rows, column].isfinite().any())
    do[:, :, row, column] = 0.0
    plain = step()
    v[:, :, row, column] = value
    got = step()  # (an element of v: its column of O from its row on)
    assert not bool(got[0][:, :, row:, column].isfinite().any()) and torch.equal(got[0][..., others], plain[0][..., others])
    assert torch.equal(got[1][:, :, :rows], plain[1][:, :, :rows]) and torch.equal(got[3], plain[3])
    if on_copies[0]:  # (the bounds-checked kernel multiplies masked scores by the 256 rows of its tile)
        assert torch.equal(got[0][:, :, :rows], plain[0][:, :, :rows])
