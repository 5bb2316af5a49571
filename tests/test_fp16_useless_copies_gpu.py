"""fp16 calls that are chunk-wise because the quadratic kernels refuse the length, at widths off the eights or on rows that the walks do not
take: backward makes no copies beside those of the library, natively and through the Python class (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import LinearAttentionAuto

from helpers import assert_close, gpu_fp32_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dqk,dv,shift", [(1500, 100, 100, 0), (700, 64, 100, 0), (1500, 91, 64, 0), (900, 64, 64, 1), (3100, 128, 128, 0)])
def test_backward_clones_nothing(n, dqk, dv, shift, gpu_device):
    gen = torch.Generator(device=gpu_device).manual_seed(n + dv)
    # (shift: rows of one element more, off the 16-byte grid)
    q, k, v, do = (torch.randn(1, 3, n, d + shift, generator=gen, device=gpu_device).mul(0.2).half()[..., shift:] for d in (dqk, dqk, dv, dv))
    want, grads = gpu_fp32_reference(q, k, v, do, True)
    for apply in (LinearAttentionAuto.apply, super(LinearAttentionAuto, LinearAttentionAuto).apply):
        args = [t.detach().requires_grad_(True) for t in (q, k, v)]
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            out = apply(*args)
            got = torch.autograd.grad(out, args, do)
        copies = [e.key for e in prof.key_averages() if e.key in ("aten::clone", "aten::copy_", "aten::contiguous")]
        assert not copies, copies
        for name, x, w in zip(("O", "dQ", "dK", "dV"), (out, *got), (want, *grads)):
            assert_close(name, x, w)
