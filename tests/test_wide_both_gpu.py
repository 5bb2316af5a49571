"""q / k and v both wider than 128 columns through the chunk-wise operator (two column halves of each): one, two, a few and
many segments per (b, h), which form a walk's entry state differently, narrow second halves, ragged lengths, strided
rows; against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (10, 13, 257, 256, 256),  # one segment
    (4, 16, 520, 192, 256),   # two
    (1, 3, 700, 256, 136),    # eleven: added up by the walk
    (1, 16, 512, 136, 192),   # eight, of one chunk each
    (1, 2, 1217, 160, 160),   # twenty: scanned
    (1, 1, 260, 256, 256),    # the shortest sequences the walks take
])
@pytest.mark.parametrize("dtype,transposed", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, False)])
def test_both_sides_wide(b, h, n, dqk, dv, dtype, transposed, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(b, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    if transposed:  # (B, N, H, D) storage
        q, k, v, do = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v, do))
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    assert torch.equal(out, linear_attention_chunked_fwd(q, k, v))
    for st in (state, None):
        for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, st), want_g):
            assert_close(f"{name}, state {st is not None}", got, want)
