"""The operators under forward-mode AD, which they refuse, and under ``torch.jit.trace``, which records them as the
Python function (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd import (
    FeatureMapLinearAttention,
    LinearAttention,
    LinearAttentionAuto,
    LinearAttentionChunked,
    LinearAttentionNormalised,
    LinearAttentionSmallVHD,
    PolynomialLinearAttention,
)

pytestmark = pytest.mark.gpu

OPERATORS = {
    "linear": (lambda q, k, v: LinearAttention.apply(q, k, v), 64, 64),
    "smallv": (lambda q, k, v: LinearAttentionSmallVHD.apply(q, k, v), 64, 32),
    "auto": (lambda q, k, v: LinearAttentionAuto.apply(q, k, v), 64, 64),
    "chunked": (lambda q, k, v: LinearAttentionChunked.apply(q, k, v), 64, 64),
    "normalised": (lambda q, k, v: LinearAttentionNormalised.apply(q, k, v, 1e-5), 64, 64),
    "feature": (lambda q, k, v: FeatureMapLinearAttention.apply(q, k, v, "elu1"), 64, 64),
    "poly": (lambda q, k, v: PolynomialLinearAttention.apply(q, k, v, 1.0, 1.0, 0.5), 16, 64),
}


def _inputs(dqk, dv, device, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return tuple(torch.rand(1, 2, 320, d, generator=gen).bfloat16().to(device) for d in (dqk, dqk, dv))


@pytest.mark.parametrize("which", range(3), ids=["q", "k", "v"])
@pytest.mark.parametrize("name", OPERATORS)
def test_forward_mode_is_refused(name, which, gpu_device):
    op, dqk, dv = OPERATORS[name]
    args = list(_inputs(dqk, dv, gpu_device))
    with torch.autograd.forward_ad.dual_level():
        args[which] = torch.autograd.forward_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises((NotImplementedError, RuntimeError)):
            op(*args)


@pytest.mark.parametrize("grad", [False, True], ids=["inference", "training"])
@pytest.mark.parametrize("name", OPERATORS)
def test_a_traced_call_computes(name, grad, gpu_device):
    op, dqk, dv = OPERATORS[name]
    first = tuple(t.requires_grad_(grad) for t in _inputs(dqk, dv, gpu_device))
    traced = torch.jit.trace(lambda q, k, v: op(q, k, v), first, check_trace=False)
    other = _inputs(dqk, dv, gpu_device, seed=1)
    assert torch.equal(traced(*other), op(*other))
