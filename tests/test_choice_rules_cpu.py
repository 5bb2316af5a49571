"""Which evaluation the library names for widths that are no multiples of 8 (host arithmetic, no GPU): the chunk-wise one from
the sequence length on from which it was measured to be the faster one, later for forward alone than for a pair."""

import pytest

from flashy_linear_attention_amd import _lib


@pytest.mark.parametrize("dqk,dv,pair_from,forward_from", [
    (20, 20, 256, 513), (31, 7, 256, 513), (36, 36, 128, 256), (100, 100, 1, 128), (91, 64, 1, 128), (153, 64, 1, 1), (250, 250, 1, 1),
])
@pytest.mark.parametrize("bh", [1, 64])
def test_widths_that_are_no_multiples_of_8(bh, dqk, dv, pair_from, forward_from):
    for name, first in (("fla_linear_attn_prefers_chunked", pair_from), ("fla_linear_attn_forward_prefers_chunked", forward_from)):
        if first > 1:
            assert _lib.query(name, 1, bh, first - 1, dqk, dv) == 0
        assert _lib.query(name, 1, bh, first, dqk, dv) == 1
        assert _lib.query(name, 1, bh, 4096, dqk, dv) == 1
