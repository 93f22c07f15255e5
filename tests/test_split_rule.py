"""The rule that divides self-attention calls between k_attention_hm and k_attention_split (a host
function) against calls timed both ways on 256 CUs, behind their operands' kernels in captured graphs:
it leaves alone what is faster undivided, and divides what is clearly faster divided."""
import h3attn as H
import pytest
from helpers import split_plan

# (tokens, rows, heads): us undivided, us as an earlier rule divided it
FASTER_UNDIVIDED = {
    (9375, 9375, 1): (163, 198), (12340, 12340, 1): (214, 259), (17246, 2948, 4): (305, 387),
    (5548, 5318, 2): (102, 121), (3565, 1083, 9): (68, 81), (3512, 3512, 3): (69, 79),
    (2593, 2593, 4): (65, 78), (1430, 1430, 10): (32, 37)}
# (tokens, rows, heads): us undivided, us divided
FASTER_DIVIDED = {
    (1024, 1024, 8): (26.3, 16.5), (502, 478, 4): (16.0, 11.0), (390, 390, 4): (14.7, 11.1),
    (252, 252, 3): (11.2, 8.0), (8193, 8193, 16): (566, 530), (2048, 2048, 4): (56.5, 22.6), (16385, 16385, 32): (3302, 3241)}


@pytest.mark.parametrize("call", FASTER_UNDIVIDED)
def test_calls_that_are_faster_undivided_are_not_divided(call):
    assert split_plan(*call, H.capacity(call[0])) is None


@pytest.mark.parametrize("call", FASTER_DIVIDED)
def test_calls_that_are_faster_divided_are_divided(call):
    assert split_plan(*call, H.capacity(call[0])) is not None


def test_every_division_covers_the_call():
    """main_blocks are whole blocks of the call, tiles per unit are one or two, and the search ends at
    the largest call the entries take."""
    for tokens, rows, heads in [(1, 1, 65535), (1048576, 1048576, 256), (1048576, 1, 65535),
                                (4097, 4097, 56), (34007, 34007, 2), (447, 447, 3), (512, 449, 4)]:
        for capacity in (H.capacity(tokens), -(-tokens // 16) * 16 + 16):
            plan = split_plan(tokens, rows, heads, capacity)
            if plan:
                assert plan[0] <= rows // 256 * heads and set(plan[1:]) <= {1, 2}
