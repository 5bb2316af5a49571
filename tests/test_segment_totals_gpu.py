"""Plans whose walks add up the segments' totals as they start, around the numbers of segments where a scan takes over (20 at
128 columns and with both sides above 128, 20 or 15 with a wide q / k alone, 32 at 64, 16 at 32): both passes, with forward's state and
without, against the fp32 oracle (``-m gpu``)."""

import ctypes

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionAuto, LinearAttentionSmallVHD, _lib
from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd
from flashy_linear_attention_amd.normalised import linear_attention_normalised_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


# (heads, N, columns): the last segment ragged.  One chunk a segment (64 rows above 64 columns, 128 up to it) up to the rule
# and one beyond it, and totals in groups of three (D = 128) and eight (64): 3, 4, 5, 9, 10 segments
@pytest.mark.parametrize("h,n,dqk,dv,dtype", [
    (12, 20 * 64 - 5, 128, 128, torch.bfloat16), (12, 21 * 64 - 5, 128, 128, torch.float16), (85, 9 * 64, 80, 80, torch.bfloat16),
    (64, 1003, 96, 96, torch.float16), (50, 5 * 64 - 1, 128, 128, torch.bfloat16), (12, 1270, 128, 64, torch.bfloat16),
    (6, 20 * 64 - 3, 256, 256, torch.bfloat16), (6, 21 * 64 - 3, 160, 256, torch.bfloat16), (32, 5 * 64, 256, 160, torch.float16),
    (36, 7 * 64 - 7, 256, 64, torch.bfloat16), (32, 8 * 64 - 7, 256, 64, torch.bfloat16), (16, 900, 192, 128, torch.float16),
    (16, 32 * 128 - 9, 64, 64, torch.bfloat16), (15, 33 * 128 - 9, 64, 64, torch.bfloat16), (30, 17 * 128 - 9, 32, 32, torch.bfloat16),
    (12, 40 * 128 - 9, 64, 64, torch.bfloat16), (12, 41 * 128 - 9, 64, 64, torch.float16), (51, 9 * 128 + 1, 32, 32, torch.bfloat16),
])
def test_both_passes(h, n, dqk, dv, dtype, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    for kept in (state, None):
        for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, kept), want_g):
            assert_close(name, got, want)


# one chunk of 128 (D = 128: 64) rows a segment, and groups of eight states (six at 128 over 64 columns) that are full, begun and left over
@pytest.mark.parametrize("segments", [3, 6, 7, 8, 9, 11, 13, 16])
@pytest.mark.parametrize("dqk,dv", [(32, 32), (64, 64), (128, 64)])
def test_groups_of_states(segments, dqk, dv, gpu_device):
    rows, resident = (128, 512) if dqk <= 64 else (64, 256)
    h, n = resident // segments, segments * rows - 5
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, state), want_g):
        assert_close(name, got, want)


@pytest.mark.parametrize("h,n,dqk,dv", [(24, 1500, 80, 80), (36, 7 * 64, 256, 64), (36, 448, 153, 64), (32, 512, 256, 128)])
def test_operators_that_keep_dq_causal(h, n, dqk, dv, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    op = LinearAttentionAuto if dqk == dv else LinearAttentionSmallVHD
    out = op.apply(q, k, v)
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), torch.autograd.grad(out, (q, k, v), do), want_g):
        assert_close(name, got, want)


@pytest.mark.parametrize("h,n,d", [(12, 20 * 64 - 5, 128), (12, 21 * 64 - 5, 128), (16, 1000, 72), (12, 40 * 128, 64)])
def test_normalised_forward(h, n, d, gpu_device):
    q, k, v, _ = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, d, d, torch.bfloat16, seed=n + d))
    qd, kd = q.double(), k.double()
    want = (torch.tril(qd @ kd.transpose(-1, -2)) @ v.double()) / ((qd * kd.cumsum(-2)).sum(-1, keepdim=True) + 1e-5)
    assert_close("out", linear_attention_normalised_fwd(q, k, v, 1e-5, True)[0], want.float())


@pytest.mark.parametrize("h,n,accepted", [(16, 16 * 64, True), (20, 12 * 64, False), (10, 24 * 64, True)])
def test_a_state_buffer_and_no_workspace(h, n, accepted, gpu_device):
    """From 13 segments on a forward with a state buffer needs no workspace: the entry states are scanned in the former."""
    q, k, v, _ = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, 128, 128, torch.bfloat16, seed=n))
    want, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    out, mine, valid = torch.empty_like(want), torch.empty_like(state), ctypes.c_int32(0)
    st = _lib.strides_arg
    rc = _lib.load().fla_linear_attn_chunked_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 1, h, n, 128, 128, st(q), st(k), st(v), st(out), _lib.FLA_DTYPE_BF16,
        mine.data_ptr(), ctypes.byref(valid), None, 0, torch.cuda.current_stream().cuda_stream)
    assert (rc == 0) == accepted
    if accepted:
        assert valid.value == 1
        assert_close("O", out, want.float())


# numbers of segments whose sums leave part of a group over
@pytest.mark.parametrize("h,n,dqk,dv", [(12, 20 * 64, 128, 128), (12, 40 * 128, 64, 64), (16, 32 * 128, 64, 64), (36, 7 * 64, 256, 64), (6, 20 * 64, 256, 256)])
def test_an_infinite_value_stays_infinite(h, n, dqk, dv, gpu_device):
    """With q, k > 0 a value (an upstream gradient) of +inf gives +inf in its column of every row after (before) it, not NaN, and
    nothing in the other columns."""
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=n + dqk))
    want, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    want_dv = linear_attention_chunked_bwd(do, q, k, v, state)[2]
    v_inf, do_inf = v.clone(), do.clone()
    v_inf[:, :, 3, 1], do_inf[:, :, n - 2, 1] = float("inf"), float("inf")
    # (a row's own chunk, of up to 128 rows, multiplies masked scores of zero by it)
    got, after, before = linear_attention_chunked_fwd(q, k, v_inf, want_state=False), slice(128, n), slice(0, n - 128)
    got_dv = linear_attention_chunked_bwd(do_inf, q, k, v, state)[2]
    for x, x_want, rows in ((got, want, after), (got_dv, want_dv, before)):
        assert bool((x[:, :, rows, 1] == float("inf")).all())
        x[:, :, :, 1] = x_want[:, :, :, 1] = 0
        assert torch.equal(x, x_want)


# a wide q / k alone: up to 15 segments over a v of 64 columns, 20 over a v of 128, a scan beyond (one chunk of 64 rows a segment)
@pytest.mark.parametrize("segments,dqk,dv", [(9, 256, 64), (12, 153, 64), (15, 192, 64), (16, 256, 64), (9, 256, 128), (20, 192, 128),
                                             (21, 256, 128)])
def test_a_wide_q_k(segments, dqk, dv, gpu_device):
    test_operators_that_keep_dq_causal(256 // segments, 64 * segments, dqk, dv, gpu_device)
