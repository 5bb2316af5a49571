"""The calls that the operators of this package are timed on.

A case is one operator call of a training step (forward, then the gradients through autograd) or of
inference (forward alone) with the sizes, types and layout given in its fields:

``op``        the autograd Function: ``linear`` (LinearAttention), ``smallv`` (LinearAttentionSmallVHD), ``auto``
              (LinearAttentionAuto), ``chunked`` (LinearAttentionChunked), ``normalised`` / ``normalised_chunked``
              (LinearAttentionNormalised), ``feature`` / ``feature_normalised`` (FeatureMapLinearAttention with elu + 1),
              ``poly`` (PolynomialLinearAttention, 1 + u + u^2 / 2, normalised)
``dtype``     bf16 or fp16
``layout``    bhnd: contiguous (B, H, N, D); bnhd: (B, N, H, D) storage seen through a transpose, which is what the view
              of a projection's output gives
``backward``  whether the gradients are formed too
``amp``       fp32 tensors under ``torch.autocast`` (the operators cast to bf16)
"""

from __future__ import annotations

import math

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

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_EPS = 1e-5


def _case(op, batch, heads, seq, d_qk, d_v, dtype="bf16", layout="bhnd", backward=True, amp=False):
    return {"op": op, "batch": batch, "heads": heads, "seq": seq, "d_qk": d_qk, "d_v": d_v, "dtype": dtype,
            "layout": layout, "backward": backward, "amp": amp}


def listed():
    return [
        # a step of a toy or test-sized model: launches and the host path
        {"name": "small_train", **_case("linear", 1, 2, 256, 64, 64)},
        # prompt processing with moderate sequences, in half precision
        {"name": "fp16_prefill", **_case("linear", 4, 16, 2048, 64, 64, dtype="fp16", backward=False)},
        # the benchmark's training shape
        {"name": "train_d128", **_case("linear", 4, 32, 4096, 128, 128)},
        # the benchmark's second-order Taylor features: 256 feature columns over 64 value columns
        {"name": "taylor_256_64", **_case("smallv", 4, 16, 4096, 256, 64)},
        # one long document
        {"name": "long_context", **_case("linear", 1, 16, 32768, 64, 64)},
        # fp32 activations under autocast, a sequence that is no multiple of any tile, heads of 80 columns
        {"name": "ragged_amp", **_case("auto", 2, 12, 1500, 80, 80, layout="bnhd", amp=True)},
        # Taylor features without the duplicates, 1 + 16 + 136 = 153 columns: rows that are not 16-byte aligned
        {"name": "taylor_153_64", **_case("smallv", 2, 16, 2048, 153, 64)},
        # heads of 256 columns, chunk-wise
        {"name": "wide_heads", **_case("chunked", 2, 8, 4096, 256, 256, layout="bnhd")},
        # the normalised operator with its defaults, many short sequences
        {"name": "normalised_batch", **_case("normalised", 16, 12, 512, 64, 64, layout="bnhd")},
        # normalised prompt processing of one long ragged sequence
        {"name": "normalised_long", **_case("normalised_chunked", 1, 16, 20000, 128, 128, backward=False)},
        # the whole recipe, feature map and normaliser, of a training step
        {"name": "recipe_train", **_case("feature_normalised", 4, 16, 4096, 64, 64, layout="bnhd")},
        # the Taylor map of exp from the 16 columns behind it
        {"name": "poly_train", **_case("poly", 4, 16, 4096, 16, 64)},
    ]


def _flops(case):
    """Least floating-point operations of one pass: the quadratic sums (lower triangle only) or the running state
    (every row updates it and is multiplied by it), whichever is less."""
    rows = case["batch"] * case["heads"] * case["seq"]
    dqk, dv = case["d_qk"], case["d_v"]
    quad = rows * case["seq"] * ((dqk + dv) + (3 * dqk + 2 * dv if case["backward"] else 0))
    width = 1 + dqk + dqk * (dqk + 1) // 2 if case["op"] == "poly" else dqk
    return min(quad, rows * width * dv * (14 if case["backward"] else 4))


def work(case):
    """Forward reads q, k, v and writes the output; backward, a call of its own that starts when the output's gradient
    is there, reads q, k, v and that gradient and writes three gradients."""
    rows = case["batch"] * case["heads"] * case["seq"]
    columns = 2 * (case["d_qk"] + case["d_v"])
    if case["backward"]:
        columns += 4 * case["d_qk"] + 3 * case["d_v"]
    # under autocast q, k, v come and their gradients leave in fp32; backward re-reads what the forward call cast them to
    size = 2.0 * rows * columns
    if case["amp"]:
        size += 2.0 * rows * (2 * case["d_qk"] + case["d_v"]) * (2 if case["backward"] else 1)
    return {"bytes": size, "flops": float(_flops(case))}


def tolerance(case):
    """Scores, running states and results are rounded to the storage type, each once (the repository's tests hold every
    result to 1e-2 in bf16)."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}


def _cost(case):
    """A rough time in seconds, for the bound on drawn cases: the larger of the bytes' and the quadratic sums' time
    (an eighth of the rate with rows that are not 16-byte aligned)."""
    rows = case["batch"] * case["heads"] * case["seq"]
    quad = rows * case["seq"] * (case["d_qk"] + case["d_v"]) * (3.5 if case["backward"] else 1.0)
    rate = 1e15 if case["d_qk"] % 8 == 0 and case["d_v"] % 8 == 0 else 1.25e14
    return max(work(case)["bytes"] / 4e12, quad / rate)


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    most_bytes = max(work(c)["bytes"] for c in listed())
    most_cost = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["linear", "linear", "smallv", "auto", "chunked", "normalised", "normalised_chunked", "feature",
                         "feature_normalised", "poly"])
        batch = _log_int(rng, 1, 16)
        heads = rng.choice([1, 2, 4, 6, 8, 12, 16, 20, 24, 32])
        seq = _log_int(rng, 100, 32768)
        if op in ("linear", "smallv"):
            seq = max(64, seq // 64 * 64)  # these two keep the reference's rule
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        if op == "poly":
            d_qk, d_v = rng.choice([8, 16, 16, 24, 32]), rng.choice([32, 48, 64, 64, 128])
        elif op == "smallv":
            d_qk, d_v = rng.choice([(64, 32), (128, 64), (128, 32), (153, 64), (91, 64), (256, 64), (256, 128), (192, 128)])
        elif op in ("linear", "auto", "chunked"):
            d_qk = d_v = rng.choice([32, 40, 64, 64, 80, 96, 100, 128, 128, 160, 256])
        else:
            d_qk = d_v = rng.choice([32, 48, 64, 64, 96, 128, 128])
        if dtype == "fp16" and seq > 4096:
            dtype = "bf16"  # fp16 ends at 65504 and the un-normalised sums grow with the sequence
        case = _case(op, batch, heads, seq, d_qk, d_v, dtype, rng.choice(["bhnd", "bnhd"]), rng.random() < 0.7,
                     dtype == "bf16" and rng.random() < 0.15)
        if work(case)["bytes"] <= most_bytes and _cost(case) <= most_cost:
            return case


def _taylor(x, width):
    """`width` second-order Taylor feature columns: x (x) x / sqrt 2 for a square, else 1, x and the upper triangle."""
    r = math.isqrt(width)
    outer = x[..., :, None] * x[..., None, :] / math.sqrt(2.0)
    if r * r == width:
        return outer.flatten(-2)
    i, j = torch.triu_indices(x.shape[-1], x.shape[-1], device=x.device)
    upper = outer[..., i, j] * torch.where(i == j, 1.0, math.sqrt(2.0))
    return torch.cat([torch.ones_like(x[..., :1]), x, upper], dim=-1)


def _query_or_key(case, shape, gen):
    width = case["d_qk"]
    if case["op"] in ("feature", "feature_normalised"):
        return torch.randn(*shape, width, generator=gen, device="cuda")  # the operator applies elu + 1
    if case["op"] == "poly":
        return 0.5 * torch.randn(*shape, width, generator=gen, device="cuda")
    if case["op"] == "smallv":
        r = math.isqrt(width)
        if r * r != width:
            r = next((r for r in range(2, 17) if 1 + r + r * (r + 1) // 2 == width), 0)
        if r:
            return _taylor(0.5 * torch.randn(*shape, r, generator=gen, device="cuda"), width)
    return torch.nn.functional.elu(torch.randn(*shape, width, generator=gen, device="cuda")) + 1.0


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    transposed = case["layout"] == "bnhd"
    b, h, n = case["batch"], case["heads"], case["seq"]
    shape = (b, n, h) if transposed else (b, h, n)
    q, k = _query_or_key(case, shape, gen), _query_or_key(case, shape, gen)
    v = torch.randn(*shape, case["d_v"], generator=gen, device="cuda")
    grad = torch.randn(*shape, case["d_v"], generator=gen, device="cuda")
    if case["dtype"] == "fp16" and case["seq"] > 2048:
        q = q * case["d_qk"] ** -0.5
    dtype = _DTYPES[case["dtype"]]
    tensors = []
    for t, kept in ((q, case["amp"]), (k, case["amp"]), (v, case["amp"]), (grad, False)):
        t = t.contiguous() if kept else t.to(dtype).contiguous()
        tensors.append(t.transpose(1, 2) if transposed else t)
    q, k, v = (t.detach().requires_grad_(case["backward"]) for t in tensors[:3])
    return {"case": case, "q": q, "k": k, "v": v, "grad": tensors[3]}


def _apply(op, q, k, v):
    if op == "linear":
        return LinearAttention.apply(q, k, v)
    if op == "smallv":
        return LinearAttentionSmallVHD.apply(q, k, v)
    if op == "auto":
        return LinearAttentionAuto.apply(q, k, v)
    if op == "chunked":
        return LinearAttentionChunked.apply(q, k, v)
    if op == "normalised":
        return LinearAttentionNormalised.apply(q, k, v, _EPS)
    if op == "normalised_chunked":
        return LinearAttentionNormalised.apply(q, k, v, _EPS, True)
    if op == "feature":
        return FeatureMapLinearAttention.apply(q, k, v, "elu1")
    if op == "feature_normalised":
        return FeatureMapLinearAttention.apply(q, k, v, "elu1", True, _EPS)
    return PolynomialLinearAttention.apply(q, k, v, 1.0, 1.0, 0.5, True, _EPS)


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["amp"]:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = _apply(case["op"], q, k, v)
    else:
        out = _apply(case["op"], q, k, v)
    if not case["backward"]:
        return out
    return (out, *torch.autograd.grad(out, (q, k, v), state["grad"]))
