"""The launches of ``fla_linear_attn_chunked_bwd_causal`` on the CPU (the trace build of the library): what the plan-level
checks of ``launch_plan`` ask of every launch, and none of the kernels that subtract from a later state."""

import pytest

import launch_plan as lp
from test_launch_plan_cpu import lib  # noqa: F401  (the fixture)


@pytest.mark.parametrize("dtype", [0, 1], ids=["bf16", "f16"])
@pytest.mark.parametrize("given", [False, True], ids=["no-state", "state"])
@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (8, 40, 512, 128, 128), (4, 32, 2048, 128, 128), (1, 32, 4096, 96, 96), (1, 4, 8192, 128, 128), (2, 16, 2048, 128, 64),
    (1, 6, 700, 64, 128), (4, 64, 512, 256, 64), (4, 16, 2048, 256, 64), (1, 8, 2048, 160, 32), (1, 20, 2048, 192, 128),
    (2, 3, 4096, 136, 128), (1, 9, 300, 136, 24),
])
def test_launches(lib, b, h, n, dqk, dv, given, dtype):  # noqa: F811
    arena = lp.Arena()
    q, k, dq, dk = (lp.make_tensor(arena, nm, b, h, n, dqk) for nm in ("q", "k", "dq", "dk"))
    v, g, dvv = (lp.make_tensor(arena, nm, b, h, n, dv) for nm in ("v", "grad_out", "dv"))
    wbytes = lib.fla_linear_attn_chunked_workspace_bytes(b, h, n, dqk, dv)
    sbytes = lib.fla_linear_attn_chunked_state_bytes(b, h, n, dqk, dv)
    work, state = arena.alloc("workspace", wbytes), arena.alloc("state", sbytes) if given else None
    rc = lib.fla_linear_attn_chunked_bwd_causal(
        g.ptr, q.ptr, k.ptr, v.ptr, dq.ptr, dk.ptr, dvv.ptr, b, h, n, dqk, dv, g.strides_arg(), q.strides_arg(),
        k.strides_arg(), v.strides_arg(), dq.strides_arg(), dk.strides_arg(), dvv.strides_arg(), dtype, state, work, wbytes, None)
    assert rc == 0, rc
    launches, stats = lp.take_launches(lib), lp.Stats()
    lp.check_all(arena, launches, stats)
    kernels = [l.kernel for l in launches]
    assert kernels.count("walk_fwd_kernel") == (2 if dqk > 128 else 1) and "walk_bwd_rev_kernel" not in kernels
    reverse = [l for l in launches if l.kernel in ("walk_dkdv_kernel", "walk_bwd_rev_wide_kernel")]
    assert len(reverse) == 1 and reverse[0].struct("a0")["dq"] == 0
