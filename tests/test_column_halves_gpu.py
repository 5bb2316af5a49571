"""Two workgroups per (b, h) on two column halves of O, on dV and dK, in place of two segments (csrc/fla_capi.hip,
walk_by_columns): 86 to 128 heads at padded head dim 128, both operators' backward, results in aligned rows, in rows of any
alignment and in fp32, and the states that forward hands over, against the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionAuto, LinearAttentionChunked
from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


# (heads, N, D_qk, D_v): the fewest chunks, an odd number of them, a ragged last one; a second half of 8, 32, 36 and 64 columns;
# both passes so above 2048 rows (B H 105, and 113 with a long sequence), backward alone (B H 100, N 2049; fp16), neither (B H 90; 72
# columns above 2048 rows)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("h,n,dqk,dv", [
    (128, 257, 128, 128), (97, 320, 72, 128), (100, 451, 96, 96), (128, 1000, 100, 100), (86, 600, 128, 72), (90, 1100, 128, 128),
    (100, 2049, 104, 96), (100, 2049, 72, 72), (105, 2300, 96, 128), (113, 4099, 128, 128),
])
def test_both_passes(h, n, dqk, dv, dtype, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    for op in (LinearAttentionAuto, LinearAttentionChunked):
        if dqk != dv and op is LinearAttentionAuto:
            out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
            grads = linear_attention_chunked_bwd(do, q, k, v, state, causal=True)
            for got, again in zip(grads, linear_attention_chunked_bwd(do, q, k, v, None, causal=True)):
                assert_close("without forward's states", again, got.float())
        else:
            leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
            out = op.apply(*leaves)
            grads = torch.autograd.grad(out, leaves, do)
        assert_close("O", out, want_o)
        for name, got, want in zip(("dQ", "dK", "dV"), grads, want_g):
            assert_close(name, got, want)


@pytest.mark.parametrize("h,n,d", [(128, 300, 96), (99, 1000, 128)])
def test_gradients_in_fp32(h, n, d, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(1, h, n, d, d, torch.bfloat16, seed=n + d))
    leaves = [t.float().requires_grad_(True) for t in (q, k, v)]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = LinearAttentionAuto.apply(*leaves)
    plain = [t.clone().requires_grad_(True) for t in (q, k, v)]
    for got, want in zip(torch.autograd.grad(out, leaves, do), torch.autograd.grad(LinearAttentionAuto.apply(*plain), plain, do)):
        assert got.dtype == torch.float32 and torch.equal(got, want.float())
