"""Which evaluation the library names (host arithmetic, no GPU): the chunk-wise one where it was measured to be the faster one.
Widths up to 128 that are multiples of 8, forward alone and pairs of 128 columns, and the normalised forward; widths that are no
multiples of 8 and the polynomial map, later for forward alone than for a pair; and the polynomial map's state."""

import pytest

from flashy_linear_attention_amd import _lib


@pytest.mark.parametrize("dqk,dv,pair_from,forward_from", [
    (20, 20, 256, 513), (31, 7, 256, 513), (36, 36, 128, 256), (100, 100, 1, 128), (91, 64, 1, 128), (153, 64, 1, 1),
])
@pytest.mark.parametrize("bh", [1, 64])
def test_widths_that_are_no_multiples_of_8(bh, dqk, dv, pair_from, forward_from):
    for name, first in (("fla_linear_attn_prefers_chunked", pair_from), ("fla_linear_attn_forward_prefers_chunked", forward_from)):
        if first > 1:
            assert _lib.query(name, 1, bh, first - 1, dqk, dv) == 0
        assert _lib.query(name, 1, bh, first, dqk, dv) == 1
        assert _lib.query(name, 1, bh, 4096, dqk, dv) == 1


# (129 heads of 128 columns and 257 of 64 are a single segment each, 128 and 256 are two: W = B H N^2 D from 1.2e10 on)
@pytest.mark.parametrize("bh,dqk,dv,first", [
    (1, 64, 64, 768), (1, 32, 32, 1024), (1, 128, 128, 1024), (1, 64, 32, 1024), (1, 128, 64, 1024), (1, 128, 32, 1024),
    (129, 128, 128, 257), (257, 64, 64, 257), (128, 128, 128, 856), (256, 64, 64, 768),
])
def test_forward_alone(bh, dqk, dv, first):
    for n, want in ((first - 1, 0), (first, 1)):
        assert _lib.query("fla_linear_attn_forward_prefers_chunked", 1, bh, n, dqk, dv) == want


@pytest.mark.parametrize("bh,first", [(130, 439), (128, 699), (1, 2048)])
def test_pairs_of_128_columns(bh, first):
    """From W = B H N^2 128 = 3.2e9 on with a single segment per head, else from 8e9 or 2048 rows."""
    for n, want in ((first - 1, 0), (first, 1)):
        assert _lib.query("fla_linear_attn_prefers_chunked", 1, bh, n, 128, 128) == want


@pytest.mark.parametrize("bh,d,first", [(1, 64, 1024), (1, 32, 1024), (1, 128, 2048), (129, 128, 257), (257, 64, 257), (128, 128, 856)])
def test_normalised_forward(bh, d, first):
    for n, want in ((first - 1, 0), (first, 1)):
        assert _lib.query("fla_normalised_forward_prefers_chunked", 1, bh, n, d, d, 0) == want
        assert _lib.query("fla_normalised_forward_prefers_chunked", 1, bh, n, d, d, 1) == 0  # fp16


def test_polynomial_state_is_for_several_segments_alone():
    """Room for 224 features over 64 columns, and their column of ones, per segment (a state takes 160 of them); nothing where a (b, h) is one segment
    (256 workgroups at a time, 128 rows a chunk), however many heads there are."""
    nbytes = lambda *shape: _lib.query("fla_poly_attn_chunked_state_bytes", *shape)  # noqa: E731
    assert nbytes(16, 256, 128, 16, 64) == nbytes(4, 100, 4096, 16, 64) == nbytes(1, 1, 100, 8, 32) == 16
    assert nbytes(4, 16, 4096, 16, 64) == 64 * 4 * 224 * 65 * 4


@pytest.mark.parametrize("bh,n,dv,pair,forward", [
    (1, 128, 64, 1, 0), (64, 1024, 64, 1, 0), (1024, 512, 64, 1, 0), (4, 2048, 64, 1, 1), (8, 2048, 64, 1, 0), (64, 4096, 64, 1, 1),
    (256, 512, 32, 1, 0), (512, 512, 32, 0, 0), (512, 128, 32, 1, 0), (512, 2048, 32, 1, 0), (1024, 4096, 32, 1, 1),
    (64, 1024, 72, 0, 0),
])
def test_polynomial(bh, n, dv, pair, forward):
    for dtype, backward, want in ((0, 1, pair), (0, 0, forward), (1, 1, 0), (1, 0, 0)):
        assert _lib.query("fla_poly_attn_prefers_chunked", 1, bh, n, 16, dv, dtype, backward) == want


def test_forward_workspace_of_copied_operands():
    """Forward asks for the copies it makes: of O, and of q, k, v where no state buffer takes them (rows of 160 and 64 elements)."""
    shape = (2, 16, 2048, 153, 64)
    full = _lib.query("fla_linear_attn_chunked_workspace_bytes", *shape)
    with_state, without = (_lib.query("fla_linear_attn_chunked_fwd_workspace_bytes", *shape, s) for s in (1, 0))
    copy = 2 * 16 * 2048 * 160 * 2
    assert without - with_state == 2 * copy and full - with_state == 4 * copy
    assert _lib.query("fla_linear_attn_chunked_fwd_workspace_bytes", 2, 16, 2048, 160, 64, 1) == _lib.query(
        "fla_linear_attn_chunked_workspace_bytes", 2, 16, 2048, 160, 64) == with_state


@pytest.mark.parametrize("name", ["fla_linear_attn_prefers_chunked", "fla_linear_attn_forward_prefers_chunked"])
def test_a_wide_v_has_one_rule(name):
    """A v of more than 128 columns: the same line whatever the widths (W = B H N^2 256 from 3e10 on)."""
    for width in (250, 255, 256):
        assert _lib.query(name, 1, 16, 2048, width, width) == 0 and _lib.query(name, 1, 16, 4096, width, width) == 1


@pytest.mark.parametrize("bh,dqk,dv,first", [
    (2, 128, 128, 3072), (16, 128, 128, 1977), (130, 80, 72, 768), (2, 128, 64, 1536), (64, 128, 32, 989), (2, 64, 40, 3072), (64, 64, 64, 1308),
    (2, 32, 32, 4096), (600, 32, 32, 768),
])
def test_half_precision_pairs(bh, dqk, dv, first):
    name = "fla_linear_attn_f16_pair_prefers_chunked"
    for n, want in ((first - 1, 0), (first, 1), (16384, 1)):
        assert _lib.query(name, 1, bh, n, dqk, dv) == want
    for widths in ((64, 32), (136, 128), (100, 100), (256, 64)):
        assert _lib.query(name, 1, bh, 16384, *widths) == 0


# (what takes 128 to 256 rows in one segment: padded widths that differ, q and k above 128 columns)
@pytest.mark.parametrize("dqk,dv,bh,n,pair,forward", [
    (128, 64, 256, 128, 0, 0), (128, 64, 257, 128, 1, 0), (128, 32, 5000, 127, 0, 0), (64, 128, 202, 256, 0, 0), (72, 40, 203, 256, 1, 0),
    (128, 32, 1430, 256, 1, 0), (128, 32, 1431, 256, 1, 1), (256, 64, 256, 127, 0, 0), (256, 64, 239, 128, 1, 0), (192, 40, 238, 128, 0, 0),
    (192, 64, 60, 256, 1, 0), (160, 128, 5000, 256, 0, 0), (256, 72, 1600, 257, 1, 0),
])
def test_up_to_256_rows(dqk, dv, bh, n, pair, forward):
    for name, want in (("fla_linear_attn_prefers_chunked", pair), ("fla_linear_attn_forward_prefers_chunked", forward)):
        assert _lib.query(name, 1, bh, n, dqk, dv) == want
    for backward, want in ((1, pair), (0, forward)):
        assert _lib.query("fla_linear_attn_operator_prefers_chunked", 1, bh, n, dqk, dv, backward) == want


# (pairs over two halves of v: one chunk, the lines beyond it, the normalised call over a full second half; above 16 columns of q and k)
@pytest.mark.parametrize("bh,n,r,dv,plain,normalised", [
    (512, 64, 16, 128, 1, 1), (513, 64, 16, 128, 0, 0), (1024, 128, 8, 120, 1, 1), (49, 128, 16, 72, 0, 0),
    (1, 129, 16, 128, 0, 1), (128, 255, 16, 128, 0, 1), (129, 255, 16, 128, 0, 0), (129, 256, 8, 128, 0, 1),
    (300, 767, 16, 120, 0, 0), (300, 768, 16, 120, 1, 1), (33, 767, 16, 72, 0, 0), (33, 768, 8, 104, 1, 1), (48, 3071, 16, 96, 0, 0),
    (48, 3072, 16, 96, 1, 1), (9, 8192, 32, 72, 0, 0), (9, 9216, 24, 96, 1, 1), (9, 8192, 32, 104, 1, 1), (8, 4096, 24, 72, 1, 1),
])
def test_polynomial_pairs_over_two_halves(bh, n, r, dv, plain, normalised):
    for flag, want in ((0, plain), (1, normalised)):
        assert _lib.query("fla_poly_attn_operator_prefers_chunked", 1, bh, n, r, dv, 0, 1, flag) == want
    assert _lib.query("fla_poly_attn_prefers_chunked", 1, bh, n, r, dv, 0, 1) == plain
    assert _lib.query("fla_poly_attn_operator_prefers_chunked", 1, bh, n, r, dv, 1, 1, 1) == 0  # fp16


@pytest.mark.parametrize("bh,dv,want", [(2, 32, 1), (3, 32, 0), (4, 40, 1), (5, 40, 0)])
def test_polynomial_forward_above_sixteen_columns(bh, dv, want):
    assert _lib.query("fla_poly_attn_operator_prefers_chunked", 1, bh, 8192, 24, dv, 0, 0, 1) == want


@pytest.mark.parametrize("bh,n,dqk,dv,forward,backward", [
    (4, 511, 20, 20, 0, 0), (4, 512, 20, 20, 0, 1), (300, 255, 36, 60, 0, 0), (1, 256, 36, 36, 0, 1), (256, 127, 100, 100, 1, 0),
    (257, 64, 100, 100, 1, 1), (1, 128, 153, 64, 1, 1), (4, 64, 153, 64, 1, 0), (1, 64, 250, 250, 1, 1), (128, 64, 91, 64, 1, 0),
    (129, 64, 91, 64, 0, 0), (129, 128, 91, 64, 1, 1), (4, 4096, 64, 64, 0, 0),
])
def test_copies_through_the_operators(bh, n, dqk, dv, forward, backward):
    for back, want in ((0, forward), (1, backward)):
        assert _lib.query("fla_linear_attn_operator_prefers_copies", 1, bh, n, dqk, dv, back) == want
