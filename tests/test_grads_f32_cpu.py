"""Gradients in fp32 (FLA_GRADS_F32), on the CPU: the sizes that fla_linear_attn_chunked_grads_f32 names are those for which the
chunk-wise backward calls take the flag, and what they refuse enqueues nothing."""

import itertools

import pytest

import launch_plan as lp

F32 = 0x100  # FLA_GRADS_F32
UNSUPPORTED = -8

DIMS = [(32, 32), (40, 64), (64, 64), (64, 32), (72, 72), (128, 128), (128, 64), (64, 128), (100, 100), (136, 64), (256, 64),
        (200, 72), (256, 128), (256, 256), (128, 256), (60, 60)]


@pytest.fixture(scope="module")
def lib():
    return lp.trace_lib()


def backward(lib, op, b, h, n, dqk, dv, with_state, dtype=0, layout="contiguous", grads="contiguous", misalign=0):
    """One chunk-wise backward with the flag: its status, the launches, and the address space they name."""
    arena = lp.Arena()
    q, k = (lp.make_tensor(arena, nm, b, h, n, dqk, layout, misalign) for nm in ("q", "k"))
    v, g, o = (lp.make_tensor(arena, nm, b, h, n, dv, layout) for nm in ("v", "grad_out", "out"))
    dq, dk, dvv = (lp.make_tensor(arena, nm, b, h, n, w, grads, size=4) for nm, w in (("dq", dqk), ("dk", dqk), ("dv", dv)))
    denom = arena.alloc("denom", 4 * b * h * n)
    normalised = "normalised" in op
    wbytes = lib.fla_normalised_workspace_bytes(b, h, n, dqk, dv, 1) if normalised else \
        lib.fla_linear_attn_chunked_workspace_bytes(b, h, n, dqk, dv)
    sbytes = lib.fla_linear_attn_chunked_state_bytes(b, h, n, dqk, dv)
    state = arena.alloc("state", sbytes) if with_state and sbytes else None
    work = arena.alloc("workspace", max(int(wbytes), 16))
    outs = (dq.ptr, dk.ptr, dvv.ptr, b, h, n, dqk, dv)
    strides = [t.strides_arg() for t in (g, q, k, v)] + ([o.strides_arg()] if normalised else []) + \
        [t.strides_arg() for t in (dq, dk, dvv)]
    tail = (state, work, wbytes, None)
    ins = (g.ptr, q.ptr, k.ptr, v.ptr)
    if op == "plain":
        rc = lib.fla_linear_attn_chunked_bwd(*ins, *outs, *strides, dtype | F32, *tail)
    elif op == "causal":
        rc = lib.fla_linear_attn_chunked_bwd_causal(*ins, *outs, *strides, dtype | F32, *tail)
    elif op == "feature":
        rc = lib.fla_feature_attn_bwd(*ins, *outs, *strides, 1, dtype | F32, *tail)
    elif op == "normalised":
        rc = lib.fla_linear_attn_normalised_bwd(*ins, o.ptr, denom, *outs, *strides, dtype | F32, 1, *tail)
    else:
        rc = lib.fla_feature_attn_normalised_bwd(*ins, o.ptr, denom, *outs, *strides, 1, dtype | F32, 1, *tail)
    return rc, lp.take_launches(lib), arena, state


OPS = ("plain", "causal", "feature", "normalised", "feature_normalised")


@pytest.mark.parametrize("op", OPS)
def test_the_sizes_named_are_those_taken(lib, op):
    taken = 0
    for (dqk, dv), (h, n), with_state in itertools.product(DIMS, ((2, 100), (8, 165), (8, 249), (3, 300), (16, 1000), (64, 513),
                                                                  (300, 700)), (True, False)):
        rc, launches, _, state = backward(lib, op, 1, h, n, dqk, dv, with_state)
        named = lib.fla_linear_attn_chunked_grads_f32(1, h, n, dqk, dv, op in ("plain", "causal"), state is not None)
        assert rc == (0 if named else UNSUPPORTED), (dqk, dv, h, n, with_state)
        assert bool(launches) == bool(named), (dqk, dv, h, n, with_state)
        taken += named
    assert taken  # (and the rest are refused)


@pytest.mark.parametrize("op", OPS)
def test_operands_without_such_a_kernel_are_refused(lib, op):
    for kwargs in ({"dtype": 1}, {"layout": "odd"}, {"misalign": 8}, {"layout": "expanded"}, {"grads": "odd"}):
        rc, launches, _, _ = backward(lib, op, 1, 8, 1000, 64, 64, True, **kwargs)
        assert rc == UNSUPPORTED and not launches, kwargs
        rc, launches, _, _ = backward(lib, op, 1, 8, 1000, 128, 128, True, **kwargs)
        assert rc == UNSUPPORTED and not launches, kwargs
