"""fp32 operands under autocast whose gradients the chunk-wise kernels store in fp32 themselves (FLA_GRADS_F32): the values of a
16-bit call, widened -- ragged lengths, one and several segments, heads of fewer columns than the padded width -- and what
the flag is refused for (``-m gpu``)."""

import ctypes

import pytest
import torch

from flashy_linear_attention_amd import (FeatureMapLinearAttention, LinearAttention, LinearAttentionAuto,
                                         LinearAttentionChunked, LinearAttentionNormalised, LinearAttentionSmallVHD,
                                         PolynomialLinearAttention, _lib)
from flashy_linear_attention_amd.chunked import linear_attention_chunked_fwd
from flashy_linear_attention_amd.feature import feature_attention_fwd, feature_attention_normalised_fwd
from flashy_linear_attention_amd.normalised import linear_attention_normalised_fwd
from flashy_linear_attention_amd.poly import poly_attention_chunked_fwd

pytestmark = pytest.mark.gpu

OPS = {
    "auto": LinearAttentionAuto.apply,
    "linear": LinearAttention.apply,
    "smallv": LinearAttentionSmallVHD.apply,
    "chunked": LinearAttentionChunked.apply,
    "normalised": lambda *a: LinearAttentionNormalised.apply(*a, 1e-5, True),
    "feature": lambda *a: FeatureMapLinearAttention.apply(*a, "elu1"),
    "feature_normalised": lambda *a: FeatureMapLinearAttention.apply(*a, "softplus", True, 1e-5),
    "poly": lambda *a: PolynomialLinearAttention.apply(*a, 1.0, 1.0, 0.5, True, 1e-5),
}


@pytest.mark.parametrize("op,b,h,n,dqk,dv", [
    ("chunked", 2, 3, 333, 64, 64), ("chunked", 1, 2, 1100, 40, 40), ("auto", 2, 4, 3000, 80, 80), ("linear", 1, 64, 4096, 128, 128),
    ("smallv", 1, 8, 4096, 128, 64), ("smallv", 1, 8, 4096, 256, 64), ("chunked", 1, 3, 700, 256, 64), ("chunked", 1, 3, 700, 200, 128), ("chunked", 1, 80, 700, 128, 128), ("chunked", 1, 2, 700, 72, 64), ("auto", 1, 2, 4096, 100, 100), ("normalised", 1, 5, 700, 64, 64),
    ("normalised", 1, 130, 300, 96, 96), ("normalised", 2, 9, 1001, 128, 128), ("feature", 1, 3, 400, 32, 32), ("feature", 1, 3, 400, 128, 128),
    ("feature_normalised", 1, 3, 515, 48, 48), ("feature_normalised", 1, 3, 515, 128, 128), ("poly", 1, 3, 515, 16, 40), ("poly", 1, 300, 200, 8, 64),
    ("normalised", 1, 2, 300, 200, 64),
])
@pytest.mark.parametrize("transposed", [False, True])
def test_equals_widening_by_hand(op, b, h, n, dqk, dv, transposed, gpu_device):
    gen = torch.Generator().manual_seed(n + dqk)
    ins = [torch.rand(b, h, n, d, generator=gen).to(gpu_device) for d in (dqk, dqk, dv, dv)]
    if transposed:
        ins = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in ins]
    do = ins[3].bfloat16()
    wide = [t.clone().requires_grad_(True) for t in ins[:3]]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = OPS[op](*wide)
    grads = torch.autograd.grad(out, wide, do)
    narrow = [t.bfloat16().requires_grad_(True) for t in ins[:3]]
    want = OPS[op](*narrow)
    want_grads = torch.autograd.grad(want, narrow, do)
    assert torch.equal(out, want)
    for got, w in zip(grads, want_grads):
        assert got.dtype == torch.float32 and torch.equal(got, w.float())


F32 = 0x100  # FLA_GRADS_F32


@pytest.mark.parametrize("dtype,n,d,causal,status", [
    (torch.bfloat16, 600, 64, True, 0), (torch.bfloat16, 600, 128, True, 0), (torch.float16, 600, 64, True, -8),
    (torch.bfloat16, 600, 128, False, 0), (torch.bfloat16, 100, 64, True, -8), (torch.bfloat16, 600, 60, True, -8),
    (torch.bfloat16, 600, 256, True, -8),
])
def test_what_the_flag_is_taken_for(dtype, n, d, causal, status, gpu_device):
    lib = _lib.load()
    q, k, v, go = (torch.rand(1, 2, n, d, device=gpu_device).to(dtype) for _ in range(4))
    code = 0 if dtype is torch.bfloat16 else 1
    out = torch.empty_like(v)
    state = torch.empty(max(16, _lib.query("fla_linear_attn_chunked_state_bytes", 1, 2, n, d, d)), dtype=torch.uint8, device=gpu_device)
    work = torch.empty(max(16, _lib.query("fla_linear_attn_chunked_workspace_bytes", 1, 2, n, d, d)), dtype=torch.uint8, device=gpu_device)
    valid = ctypes.c_int32(0)
    st = _lib.strides_arg
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.fla_linear_attn_chunked_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 1, 2, n, d, d, st(q), st(k), st(v),
                                           st(out), code, state.data_ptr(), ctypes.byref(valid), work.data_ptr(), work.numel(), stream) == 0
    grads = [torch.full((1, 2, n, d), 7.0, device=gpu_device) for _ in range(3)]
    fn = lib.fla_linear_attn_chunked_bwd_causal if causal else lib.fla_linear_attn_chunked_bwd
    got = fn(go.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), *(t.data_ptr() for t in grads), 1, 2, n, d, d, st(go), st(q),
             st(k), st(v), *(st(t) for t in grads), code | F32, state.data_ptr() if valid.value else None, work.data_ptr(),
             work.numel(), stream)
    assert got == status
    torch.cuda.synchronize()
    assert all(bool((t == 7.0).all()) == (status != 0) for t in grads)


@pytest.mark.parametrize("op,b,h,n,dqk,dv,stored", [
    ("chunked", 1, 2, 100, 64, 64, False), ("auto", 1, 8, 249, 32, 32, False), ("normalised", 1, 2, 300, 256, 64, False),
    ("feature", 1, 2, 100, 64, 64, False), ("feature_normalised", 1, 2, 200, 128, 128, False), ("chunked", 1, 3, 700, 256, 128, False),
    ("chunked", 1, 2, 300, 64, 64, True), ("normalised", 1, 5, 700, 64, 64, True), ("feature", 1, 3, 400, 128, 128, True),
    ("feature_normalised", 1, 3, 515, 48, 48, True), ("smallv", 1, 8, 4096, 256, 64, True), ("poly", 1, 3, 515, 16, 40, True),
])
def test_gradients_are_allocated_once(op, b, h, n, dqk, dv, stored, gpu_device):
    """Beside what a 16-bit backward allocates, one of fp32 operands allocates nothing where the kernels store fp32, and the
    three converted gradients elsewhere -- no second set for a call that is refused."""
    def allocations(cast):
        ins = [torch.rand(b, h, n, d, device=gpu_device) for d in (dqk, dqk, dv)]
        ins = [(t if cast else t.bfloat16()).requires_grad_(True) for t in ins]
        do = torch.rand(b, h, n, dv, device=gpu_device).bfloat16()
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=cast):
            out = OPS[op](*ins)
        before = torch.cuda.memory_stats(gpu_device)["allocation.all.allocated"]
        grads = torch.autograd.grad(out, ins, do)
        assert all(g.dtype == t.dtype for g, t in zip(grads, ins))
        return torch.cuda.memory_stats(gpu_device)["allocation.all.allocated"] - before
    allocations(False), allocations(True)
    assert allocations(True) - allocations(False) == (0 if stored else 3)


def backward_call(op, n, dqk, dv, dtype, device):
    """`call(code, grads)` -> status of the operator's backward entry point, over what its forward left."""
    lib, stream, st = _lib.load(), torch.cuda.current_stream().cuda_stream, _lib.strides_arg
    b, h, gen = 1, 3, torch.Generator().manual_seed(n + dqk)
    q, k, v, go = (torch.rand(b, h, n, d, generator=gen).to(device, dtype) for d in (dqk, dqk, dv, dv))
    out = denom = None
    middle, end = (), ()  # (arguments between the strides and the dtype; between the dtype and the state)
    workspace = ("fla_linear_attn_chunked_workspace_bytes",)
    if op in ("chunked", "causal"):
        fn = lib.fla_linear_attn_chunked_bwd if op == "chunked" else lib.fla_linear_attn_chunked_bwd_causal
        _, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    elif op == "feature":
        fn, middle = lib.fla_feature_attn_bwd, (1,)
        _, q, k, state = feature_attention_fwd(q, k, v, "elu1", want_state=True)
    elif op == "poly":
        fn, middle, workspace = lib.fla_poly_attn_chunked_bwd, ((ctypes.c_float * 3)(1.0, 1.0, 0.5),), ("fla_poly_attn_chunked_workspace_bytes",)
        out, denom, state = poly_attention_chunked_fwd(q, k, v, (1.0, 1.0, 0.5), True, 1e-5)
    else:
        end, workspace = (1,), ("fla_normalised_workspace_bytes", 1)
        if op == "normalised":
            fn = lib.fla_linear_attn_normalised_bwd
            out, denom, state = linear_attention_normalised_fwd(q, k, v, 1e-5, True, want_state=True)
        else:
            fn, middle = lib.fla_feature_attn_normalised_bwd, (1,)
            out, q, k, denom, state = feature_attention_normalised_fwd(q, k, v, "elu1", 1e-5, want_state=True)
    work = torch.empty(max(16, _lib.query(workspace[0], b, h, n, dqk, dv, *workspace[1:])), dtype=torch.uint8, device=device)
    ins = [go, q, k, v] + ([out] if out is not None else [])

    def call(code, grads):
        pointers = [t.data_ptr() for t in ins] + ([denom.data_ptr()] if denom is not None else []) + [t.data_ptr() for t in grads]
        status = fn(*pointers, b, h, n, dqk, dv, *(st(t) for t in (*ins, *grads)), *middle, code, *end,
                    state.data_ptr() if state is not None else None, work.data_ptr(), work.numel(), stream)
        torch.cuda.synchronize()
        return status
    return call, [(b, h, n, d) for d in (dqk, dqk, dv)]


# one entry point after the other, ragged lengths; columns below the padded width; both halves of a wide q / k
@pytest.mark.parametrize("op,n,dqk,dv", [
    ("chunked", 601, 64, 64), ("chunked", 601, 128, 128), ("chunked", 601, 128, 40), ("chunked", 601, 256, 64), ("causal", 601, 200, 64),
    ("causal", 601, 128, 128), ("causal", 601, 80, 80), ("feature", 601, 64, 64), ("feature", 601, 104, 104), ("normalised", 601, 32, 32),
    ("normalised", 601, 128, 128), ("feature_normalised", 601, 56, 56), ("feature_normalised", 601, 128, 128), ("poly", 601, 16, 64),
    ("poly", 601, 8, 40),
])
def test_the_calls_store_every_value(op, n, dqk, dv, gpu_device):
    """Straight to the library: the flag is taken, and every element of the three buffers is the 16-bit call's, widened."""
    call, shapes = backward_call(op, n, dqk, dv, torch.bfloat16, gpu_device)
    want = [torch.full(s, float("nan"), dtype=torch.bfloat16, device=gpu_device) for s in shapes]
    got = [torch.full(s, float("nan"), device=gpu_device) for s in shapes]
    assert call(0, want) == 0 and call(0 | F32, got) == 0
    for name, g, w in zip(("dQ", "dK", "dV"), got, want):
        assert bool(w.isfinite().all()) and torch.equal(g, w.float()), name


@pytest.mark.parametrize("op,n,dqk,dv,dtype", [
    ("chunked", 601, 256, 128, torch.bfloat16), ("causal", 601, 128, 128, torch.float16), ("feature", 100, 64, 64, torch.bfloat16),
    ("normalised", 200, 128, 128, torch.bfloat16), ("normalised", 601, 64, 64, torch.float16),
    ("feature_normalised", 601, 256, 64, torch.bfloat16),
])
def test_the_calls_refuse_without_a_store(op, n, dqk, dv, dtype, gpu_device):
    """... and the sizes and types without such a kernel: refused, nothing written; the 16-bit call of the same is taken."""
    code = 0 if dtype is torch.bfloat16 else 1
    call, shapes = backward_call(op, n, dqk, dv, dtype, gpu_device)
    grads = [torch.full(s, 7.0, device=gpu_device) for s in shapes]
    assert call(code | F32, grads) == -8 and all(bool((t == 7.0).all()) for t in grads)
    assert call(code, [torch.empty(s, dtype=dtype, device=gpu_device) for s in shapes]) == 0
