"""Widths that are no multiples of 8 through the chunk-wise operator (copies with aligned rows): the copy kernel's edges --
a row's last partial chunk, one row, one column, rows of other strides -- and plans of every kind behind it, against
the fp32 oracle (``-m gpu``)."""

import pytest
import torch

from flashy_linear_attention_amd.chunked import linear_attention_chunked_bwd, linear_attention_chunked_fwd

from helpers import assert_close, gpu_fp32_reference, reference_style_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,n,dqk,dv", [
    (1, 1, 1, 1, 1), (1, 2, 65, 7, 9), (2, 3, 300, 33, 31), (1, 2, 700, 100, 100), (1, 3, 1000, 91, 64), (2, 1, 520, 153, 64),
    (1, 2, 330, 64, 57), (1, 2, 390, 255, 255), (1, 1, 600, 129, 127), (1, 2, 640, 100, 250),
])
@pytest.mark.parametrize("dtype,transposed", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, True)])
def test_widths_off_the_eights(b, h, n, dqk, dv, dtype, transposed, gpu_device):
    q, k, v, do = (t.to(gpu_device) for t in reference_style_inputs(b, h, n, dqk, dv, dtype, seed=n + dqk))
    want_o, want_g = gpu_fp32_reference(q, k, v, do, True)
    if transposed:  # (B, N, H, D) storage
        q, k, v, do = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v, do))
    out, state = linear_attention_chunked_fwd(q, k, v, want_state=True)
    assert_close("O", out, want_o)
    assert torch.equal(out, linear_attention_chunked_fwd(q, k, v))
    for st in (state, None):  # (forward's copies, and copies of backward's own)
        for name, got, want in zip(("dQ", "dK", "dV"), linear_attention_chunked_bwd(do, q, k, v, st), want_g):
            assert_close(f"{name}, state {st is not None}", got, want)


def test_copies_are_kept_in_place_of_the_operands(gpu_device):
    """What a training step holds on to between forward and backward: the copies, and not q, k, v beside them."""
    from flashy_linear_attention_amd import LinearAttentionSmallVHD, _lib

    leaves = [t.to(gpu_device).requires_grad_(True) for t in reference_style_inputs(1, 8, 2048, 153, 64, torch.bfloat16, seed=3)[:3]]
    torch.cuda.synchronize()
    q, k, v = (t * 1.0 for t in leaves)  # (a product with a number keeps neither factor)
    base = torch.cuda.memory_allocated() - sum(t.numel() * 2 for t in (q, k, v))
    out = LinearAttentionSmallVHD.apply(q, k, v)
    size = q.numel() * 2
    del q, k
    state = _lib.query("fla_linear_attn_chunked_state_bytes", 1, 8, 2048, 153, 64)
    # (v, the output and the state buffer with the copies; allocations are rounded up to 2 MiB at most)
    held = torch.cuda.memory_allocated() - base
    assert held <= v.numel() * 2 + out.numel() * 2 + state + 3 * (2 << 20) < held + 2 * size
    out.backward(torch.ones_like(out))
    grads = [t.grad.clone() for t in leaves]
    for t in leaves:
        t.grad = None
    qc, kc, vc = leaves
    LinearAttentionSmallVHD.apply(qc, kc, vc).backward(torch.ones_like(out))
    assert all(torch.equal(a, t.grad) for a, t in zip(grads, leaves))


@pytest.mark.parametrize("which", range(3), ids=["q", "k", "v"])
def test_an_operand_written_to_in_place_is_refused(which, gpu_device):
    """... as autograd refuses it for an operand that a node keeps, copied or not."""
    from flashy_linear_attention_amd import LinearAttentionSmallVHD

    leaves = [t.to(gpu_device).requires_grad_(True) for t in reference_style_inputs(1, 2, 1024, 91, 64, torch.bfloat16, seed=5)[:3]]
    args = [t * 1.0 for t in leaves]
    out = LinearAttentionSmallVHD.apply(*args)
    args[which].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def test_saved_tensor_hooks_see_the_copies(gpu_device):
    from flashy_linear_attention_amd import LinearAttentionSmallVHD

    leaves = [t.to(gpu_device).requires_grad_(True) for t in reference_style_inputs(1, 2, 1024, 91, 64, torch.bfloat16, seed=6)[:3]]
    want = torch.autograd.grad(LinearAttentionSmallVHD.apply(*leaves).sum(), leaves)
    with torch.autograd.graph.save_on_cpu():
        out = LinearAttentionSmallVHD.apply(*leaves)
    for a, b in zip(torch.autograd.grad(out.sum(), leaves), want):
        assert torch.equal(a, b)
