"""fp16 feature-map calls without the normaliser whose rows the mapping walks do not take: forward maps in passes of its own and
runs the plain walk, which scales its saved states, and the mapping backward walk reads those.  Forward and backward agree on the scales of a
state on the CPU (launch records), and the gradients are the oracle's on the GPU."""

import ctypes

import pytest
import torch

import launch_plan as lp
from flashy_linear_attention_amd import FeatureMapLinearAttention
from test_results_plan_cpu import lib  # noqa: F401

from helpers import assert_close


# (three chunks of 128 rows, the last of one row or more, one segment per head, several)
SHAPES = [(1, 2, 257, 64, 64), (1, 2, 300, 32, 32), (2, 300, 260, 64, 48), (1, 2, 1024, 40, 64), (1, 16, 2048, 24, 16)]


def state_scales(launches):
    """whether each saved state has scales, as its writer and as its reader has it"""
    wrote, read = {}, {}
    for l in launches:
        p = l.struct("a0")
        if l.kernel == "walk_fwd_kernel" and p["saved"]:
            wrote[p["saved"]] = p["saved_scale"]
        if l.kernel == "walk_bwd_kernel":
            read[p["saved"]] = p["saved_scale"]
    return wrote, read


@pytest.mark.parametrize("b,h,n,dqk,dv", SHAPES)
@pytest.mark.parametrize("dtype", [0, 1], ids=["bf16", "f16"])
@pytest.mark.parametrize("layout", ["contiguous", "bnhd", "odd"])
@pytest.mark.parametrize("mapped_fwd,mapped_bwd", [(True, True), (False, False), (True, False), (False, True)])
def test_forward_and_backward_agree_on_a_states_scales(lib, b, h, n, dqk, dv, dtype, layout, mapped_fwd, mapped_bwd):  # noqa: F811
    """(the feature-map calls share the plain ones' state: either's backward takes either's)"""
    arena = lp.Arena()
    xq, xk = (lp.make_tensor(arena, nm, b, h, n, dqk, layout) for nm in ("xq", "xk"))
    q, k, dq, dk = (lp.make_tensor(arena, nm, b, h, n, dqk) for nm in ("q", "k", "dq", "dk"))
    v, o, g, dvv = (lp.make_tensor(arena, nm, b, h, n, dv) for nm in ("v", "out", "grad_out", "dv"))
    sbytes, wbytes = (getattr(lib, f"fla_linear_attn_chunked_{nm}_bytes")(b, h, n, dqk, dv) for nm in ("state", "workspace"))
    state, valid = arena.alloc("state", sbytes), ctypes.c_int32(0)
    work = arena.alloc("workspace", max(wbytes, 16))
    if mapped_fwd:
        st = [t.strides_arg() for t in (xq, xk, v, o, q, k)]
        assert lib.fla_feature_attn_fwd(xq.ptr, xk.ptr, v.ptr, o.ptr, q.ptr, k.ptr, b, h, n, dqk, dv, *st, 1, dtype, state,
                                        ctypes.byref(valid), work, wbytes, None) == 0
    else:
        st = [t.strides_arg() for t in (q, k, v, o)]
        assert lib.fla_linear_attn_chunked_fwd(q.ptr, k.ptr, v.ptr, o.ptr, b, h, n, dqk, dv, *st, dtype, state, ctypes.byref(valid), work,
                                               wbytes, None) == 0
    launches = lp.take_launches(lib)
    st = [t.strides_arg() for t in (g, q, k, v, dq, dk, dvv)]
    ins = (g.ptr, q.ptr, k.ptr, v.ptr, dq.ptr, dk.ptr, dvv.ptr, b, h, n, dqk, dv)
    tail = (dtype, state if valid.value else None, work, wbytes, None)
    assert (lib.fla_feature_attn_bwd(*ins, *st, 1, *tail) if mapped_bwd else lib.fla_linear_attn_chunked_bwd_causal(*ins, *st, *tail)) == 0
    launches += lp.take_launches(lib)
    lp.check_all(arena, launches, lp.Stats())
    wrote, read = state_scales(launches)
    assert wrote == read and set(wrote) == {state}
    assert bool(wrote[state]) == (dtype == 1)


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,n,dqk,dv", SHAPES)
@pytest.mark.parametrize("kind", ["elu1", "softplus"])
def test_gradients_of_rows_off_the_grid(b, h, n, dqk, dv, kind, gpu_device):
    from oracle import naive

    gen = torch.Generator().manual_seed(n + dqk + dv)
    xq, xk = (torch.randn(b, h, n, dqk + 1, generator=gen).half() for _ in range(2))
    v, do = (torch.randn(b, h, n, dv, generator=gen).half() for _ in range(2))
    part = [t[:1, -2:].float() for t in (xq[..., 1:], xk[..., 1:], v, do)]
    want = (naive.feature_causal_dot_product(*part[:3], kind), *naive.feature_causal_dot_product_grads(*part, kind))
    base = FeatureMapLinearAttention
    results = []
    for apply in (base.apply, super(base, base).apply):
        args = [t.to(gpu_device).requires_grad_(True) for t in (xq, xk, v)]
        out = apply(args[0][..., 1:], args[1][..., 1:], args[2], kind)
        grads = torch.autograd.grad(out, args, do.to(gpu_device))
        got = (out.detach(), grads[0][..., 1:], grads[1][..., 1:], grads[2])
        for name, x, w in zip(("O", "dXq", "dXk", "dV"), got, want):
            assert_close(name, x[:1, -2:], w)
        results.append(got)
    assert all(torch.equal(x, y) for x, y in zip(*results))
