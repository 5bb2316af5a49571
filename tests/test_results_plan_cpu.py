"""Where the chunk-wise calls store their results, on the CPU (tests/launch_plan.py): every result of a call is written, all of
it and nothing beside it, in each of the forms that the walks have -- 16-bit rows, rows of floats, rows of any alignment -- and a
buffer that is too small for the call is noticed."""

import ctypes

import pytest

import launch_plan as lp
from test_grads_f32_cpu import OPS, backward

F32 = 0x100  # FLA_GRADS_F32


@pytest.fixture(scope="module")
def lib():
    return lp.trace_lib()


def written(stats, arena, name):
    """the bytes of a tensor from its first to its last result store, and its size"""
    region = next(r for r in arena.regions if r.name == name)
    inside = [(lo, hi) for lo, hi in stats.results if region.lo <= lo < region.hi]
    return (min(lo for lo, _ in inside) - region.lo, max(hi for _, hi in inside) - region.lo) if inside else None, region.hi - region.lo


def checked(arena, launches, results):
    stats = lp.Stats()
    lp.check_all(arena, launches, stats)
    for name in results:
        got, size = written(stats, arena, name)
        assert got == (0, size), f"{name}: {got} of {size} bytes"
    return stats


def plain(lib, b, h, n, dqk, dv, causal, with_state, layout="contiguous", dtype=0):
    arena = lp.Arena()
    q, k, dq, dk = (lp.make_tensor(arena, nm, b, h, n, dqk, layout) for nm in ("q", "k", "dq", "dk"))
    v, g, o, dvv = (lp.make_tensor(arena, nm, b, h, n, dv, layout) for nm in ("v", "grad_out", "out", "dv"))
    wbytes = lib.fla_linear_attn_chunked_workspace_bytes(b, h, n, dqk, dv)
    sbytes = lib.fla_linear_attn_chunked_state_bytes(b, h, n, dqk, dv) if with_state else 0
    state, valid = arena.alloc("state", sbytes) if sbytes else None, ctypes.c_int32(0)
    st = [t.strides_arg() for t in (q, k, v, o)]
    assert lib.fla_linear_attn_chunked_fwd(q.ptr, k.ptr, v.ptr, o.ptr, b, h, n, dqk, dv, *st, dtype, state, ctypes.byref(valid),
                                           arena.alloc("forward workspace", max(wbytes, 16)), wbytes, None) == 0
    fwd = lp.take_launches(lib)
    st = [t.strides_arg() for t in (g, q, k, v, dq, dk, dvv)]
    call = lib.fla_linear_attn_chunked_bwd_causal if causal else lib.fla_linear_attn_chunked_bwd
    assert call(g.ptr, q.ptr, k.ptr, v.ptr, dq.ptr, dk.ptr, dvv.ptr, b, h, n, dqk, dv, *st, dtype, state if valid.value else None,
                arena.alloc("backward workspace", max(wbytes, 16)), wbytes, None) == 0
    return arena, fwd, lp.take_launches(lib)


@pytest.mark.parametrize("h,n", [(3, 300), (16, 2048), (40, 700), (300, 200)])
@pytest.mark.parametrize("dqk,dv", [(91, 91), (100, 100), (153, 64), (153, 57), (200, 30), (91, 64), (72, 57), (128, 128), (256, 64),
                                    (200, 72), (128, 64), (256, 256)])
@pytest.mark.parametrize("layout", ["contiguous", "bnhd"])
def test_results_of_the_plain_operator(lib, dqk, dv, h, n, layout):
    rows = set()
    for causal in (False, True):
        for with_state in (True, False):
            for dtype in (0, 1):
                arena, fwd, bwd = plain(lib, 1, h, n, dqk, dv, causal, with_state, layout, dtype)
                if layout == "contiguous" and all(l.kernel.startswith(("walk_", "pack_")) for l in fwd + bwd):
                    checked(arena, fwd, ("out",)), checked(arena, bwd, ("dq", "dk", "dv"))
                else:  # (rows between which other tensors' would lie; other kernels: each access against its tensor)
                    checked(arena, fwd, ()), checked(arena, bwd, ())
                rows |= {l.kernel for l in fwd + bwd if l.kernel.startswith("walk_") and l.args.get("a0.any_rows")}
    if (dqk, dv) == (91, 91) and n > 200:
        assert rows == {"walk_fwd_kernel", "walk_dkdv_kernel", "walk_bwd_rev_kernel"}
    if (dqk, dv) == (153, 64) and n == 2048:
        assert "walk_bwd_rev_wide_kernel" in rows
    if dqk % 8 == 0 and dv % 8 == 0:
        assert not rows


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dqk,dv", [(64, 64), (40, 40), (128, 128), (96, 104), (128, 64), (64, 128), (256, 64), (200, 64)])
def test_fp32_gradients(lib, op, dqk, dv):
    taken = 0
    for h, n in ((3, 300), (16, 1000), (64, 513), (300, 700), (12, 5000)):
        for with_state in (True, False):
            rc, launches, arena, _ = backward(lib, op, 1, h, n, dqk, dv, with_state)
            if rc == 0:
                checked(arena, launches, ("dq", "dk", "dv"))
                taken += 1
    assert taken or (op not in ("plain", "causal") and (dqk > 128 or (dqk > 64) != (dv > 64)))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("name", ["dq", "dk", "dv"])
def test_a_result_of_half_the_bytes_is_noticed(lib, d, name):
    """A 16-bit tensor in the place of a fp32 gradient: the second half of the stores lies outside it."""
    _, launches, arena, _ = backward(lib, "plain", 1, 16, 1000, d, d, True)
    region = next(r for r in arena.regions if r.name == name)
    region.hi = region.lo + (region.hi - region.lo) // 2
    with pytest.raises(AssertionError, match=name):
        lp.check_all(arena, launches, lp.Stats())


@pytest.mark.parametrize("dqk,dv", [(91, 91), (153, 64)])
@pytest.mark.parametrize("name", ["out", "dq", "dk"])
def test_a_result_at_odd_rows_that_lacks_its_last_element_is_noticed(lib, dqk, dv, name):
    for with_state in (True, False):
        arena, fwd, bwd = plain(lib, 1, 16, 2048, dqk, dv, True, with_state)
        region = next(r for r in arena.regions if r.name == name)
        region.hi -= 2
        with pytest.raises(AssertionError, match=r"runs past the end of " + name):
            lp.check_all(arena, fwd + bwd, lp.Stats())


@pytest.mark.parametrize("normalised", [False, True])
@pytest.mark.parametrize("flag", [0, F32])
@pytest.mark.parametrize("h,n,r,dv", [(3, 515, 16, 40), (64, 4096, 16, 64), (16, 4096, 8, 64), (300, 200, 8, 64), (2, 100, 16, 8)])
def test_polynomial_map(lib, h, n, r, dv, flag, normalised):
    arena = lp.Arena()
    q, k = (lp.make_tensor(arena, nm, 1, h, n, r) for nm in ("q", "k"))
    v, o, g = (lp.make_tensor(arena, nm, 1, h, n, dv) for nm in ("v", "out", "grad_out"))
    dq, dk, dvv = (lp.make_tensor(arena, nm, 1, h, n, w, size=4 if flag else 2) for nm, w in (("dq", r), ("dk", r), ("dv", dv)))
    denom = arena.alloc("denom", 4 * h * n) if normalised else None
    sbytes, wbytes = (getattr(lib, f"fla_poly_attn_chunked_{nm}_bytes")(1, h, n, r, dv) for nm in ("state", "workspace"))
    state = arena.alloc("state", sbytes)
    coef = (ctypes.c_float * 3)(1.0, 1.0, 0.5)
    st = [t.strides_arg() for t in (q, k, v, o)]
    assert lib.fla_poly_attn_chunked_fwd(q.ptr, k.ptr, v.ptr, o.ptr, denom, 1, h, n, r, dv, *st, coef, 1e-5, 0, state,
                                         arena.alloc("forward workspace", max(wbytes, 16)), wbytes, None) == 0
    checked(arena, lp.take_launches(lib), ("out",))
    st = [t.strides_arg() for t in (g, q, k, v)] + [o.strides_arg() if normalised else None] + [t.strides_arg() for t in (dq, dk, dvv)]
    assert lib.fla_poly_attn_chunked_bwd(g.ptr, q.ptr, k.ptr, v.ptr, o.ptr if normalised else None, denom, dq.ptr, dk.ptr, dvv.ptr, 1, h,
                                         n, r, dv, *st, coef, flag, state, arena.alloc("backward workspace", max(wbytes, 16)), wbytes,
                                         None) == 0
    launches = lp.take_launches(lib)
    checked(arena, launches, ("dq", "dk", "dv"))
    own_totals = [l.args["a0.u_totals"] for l in launches if l.kernel == "poly_walk_dq_kernel"] == [1]
    assert own_totals == (3 <= launches[-1].args["a0.n_seg"] <= 20)
    if own_totals:  # (without the walk for dq, nothing has written the totals)
        with pytest.raises(AssertionError, match="totals that nothing wrote"):
            lp.check_all(arena, [l for l in launches if l.kernel != "poly_walk_dq_kernel"], lp.Stats())
