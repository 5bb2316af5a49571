"""The polynomial map's chunk-wise forward asks for what it writes: the segments' totals and, above 16 columns of q and k, the sums that go
from launch to launch, 65 floats a row and half of v."""

import ctypes

import pytest

import launch_plan as lp
from test_results_plan_cpu import checked, lib  # noqa: F401

WORKSPACE = -9  # FLA_ERR_WORKSPACE


@pytest.mark.parametrize("normalised", [False, True])
@pytest.mark.parametrize("b,h,n,r,dv", [(1, 2, 130, 32, 64), (1, 40, 1100, 24, 128), (1, 1, 3200, 32, 72), (300, 1, 200, 24, 8), (1, 3, 300, 16, 128),
                                        (4, 16, 1024, 16, 64), (150, 1, 200, 8, 120)])
def test_forward_workspace(lib, b, h, n, r, dv, normalised):  # noqa: F811
    need, both = (getattr(lib, f"fla_poly_attn_chunked_{nm}workspace_bytes")(b, h, n, r, dv) for nm in ("fwd_", ""))
    halves, segments = 1 + (dv > 64), lib.fla_poly_attn_chunked_state_bytes(b, h, n, r, dv) > 16
    sums = b * h * halves * n * 65 * 4 if r > 16 else 0
    assert sums <= need <= both and (segments or need == sums)
    # (the rest is backward's: 128 floats of sums, and dXq and dXk of two halves)
    rows = b * h * halves * n * 4
    assert both - need == rows * ((128 - 65 if r > 16 else 0) + (2 * (32 if r > 16 else 16) if dv > 64 else 0))
    for nbytes in (need, need - 1):
        arena = lp.Arena()
        q, k = (lp.make_tensor(arena, nm, b, h, n, r) for nm in ("q", "k"))
        v, o = (lp.make_tensor(arena, nm, b, h, n, dv) for nm in ("v", "out"))
        denom = arena.alloc("denom", 4 * b * h * n) if normalised else None
        state = arena.alloc("state", lib.fla_poly_attn_chunked_state_bytes(b, h, n, r, dv))
        work = arena.alloc("workspace", nbytes) if nbytes > 0 else None
        st = [t.strides_arg() for t in (q, k, v, o)]
        rc = lib.fla_poly_attn_chunked_fwd(q.ptr, k.ptr, v.ptr, o.ptr, denom, b, h, n, r, dv, *st, (ctypes.c_float * 3)(1.0, 1.0, 0.5), 1e-5, 0,
                                           state, work, nbytes, None)
        launches = lp.take_launches(lib)
        if nbytes < need and need > 0:
            assert rc == WORKSPACE and not launches
        elif nbytes >= 0:
            assert rc == 0
            checked(arena, launches, ("out",))
