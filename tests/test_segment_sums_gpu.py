"""Plans at padded head dims up to 64 around the largest number of segments per (b, h) whose totals the walks add up
themselves (16): the state and both passes against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


# (B H, N): nine, sixteen and seventeen segments of one or two chunks, the last one ragged
@pytest.mark.parametrize("h,n", [(56, 1151), (32, 2047), (32, 4001), (30, 2175)])
@pytest.mark.parametrize("d,dtype", [(64, torch.bfloat16), (40, torch.float16), (32, torch.bfloat16)])
def test_segment_counts_around_the_rule(h, n, d, dtype, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, d, d, dtype, seed=n + d))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert state is not None
    assert_close("O", out, want_o)
    for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, state), want_g):
        assert_close(name, got, want)
