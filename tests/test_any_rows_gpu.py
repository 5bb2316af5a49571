"""Widths that are no multiples of 8, chunk-wise: the walks store results to rows of any alignment -- whole chunks of eight columns
and one to seven left over, a left-over chunk in each quarter of a block, narrow and wide sides, dQ by its own walk and by
subtraction -- against the fp32 oracle, and the columns beside a result's rows keep what they held (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import _lib
from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16), ids=("bf16", "fp16"))
@pytest.mark.parametrize("h,n,dqk,dv", [
    (2, 321, 65, 65), (3, 700, 100, 100), (1, 1030, 127, 127), (2, 500, 73, 118), (2, 513, 100, 60), (2, 513, 60, 100), (2, 449, 128, 99),
    (2, 450, 99, 128), (2, 577, 129, 64), (3, 640, 153, 64), (1, 900, 255, 32), (2, 600, 175, 8), (2, 600, 153, 61),
])
def test_against_the_oracle(h, n, dqk, dv, dtype, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    for causal in (False, True):
        for kept in (state, None):
            for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, kept, causal), want_g):
                assert_close(name, got, want)


@pytest.mark.parametrize("h,n,dqk,dv", [(2, 450, 100, 100), (2, 450, 153, 64), (2, 450, 100, 64), (2, 450, 96, 75)])
@pytest.mark.parametrize("causal", (False, True))
def test_columns_beside_the_results(h, n, dqk, dv, causal, gpu_device):
    """Results as column slices of wider tensors, one element into a row: the same values, and nothing beside them written."""
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, torch.bfloat16, seed=dqk))
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    want = (out, *linear_attention_chunked_bwd(do, q, k, v, state, causal))
    # (a side of whole chunks of eight columns is written where it lies: its rows stay aligned)
    lead = [1 if t.shape[-1] % 8 else 8 for t in want]
    wide = [torch.full((*t.shape[:-1], t.shape[-1] + 2 * e), 7.0, device=gpu_device, dtype=t.dtype) for t, e in zip(want, lead)]
    inner = [w[..., e:-e] for w, e in zip(wide, lead)]
    dims = (1, h, n, dqk, dv)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    work = torch.empty(_lib.query("fla_linear_attn_chunked_workspace_bytes", *dims), dtype=torch.uint8, device=gpu_device)
    st, kind = _lib.strides_arg, _lib.FLA_DTYPE_BF16
    fwd, bwd = lib.fla_linear_attn_chunked_fwd, lib.fla_linear_attn_chunked_bwd_causal if causal else lib.fla_linear_attn_chunked_bwd
    o, dq, dk, dvv = inner
    assert fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *dims, st(q), st(k), st(v), st(o), kind, None, None,
               work.data_ptr(), work.numel(), stream) == 0
    assert bwd(do.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), dq.data_ptr(), dk.data_ptr(), dvv.data_ptr(), *dims, st(do), st(q),
               st(k), st(v), st(dq), st(dk), st(dvv), kind, state.data_ptr(), work.data_ptr(), work.numel(), stream) == 0
    for w, got, ref, e in zip(wide, inner, want, lead):
        assert torch.equal(got, ref)
        assert bool((w[..., :e] == 7).all()) and bool((w[..., -e:] == 7).all())
