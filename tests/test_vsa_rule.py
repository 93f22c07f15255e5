"""The rule that launches a VSA runtime's prefix cubes apart (a host function) against runtime calls timed
both ways on 256 CUs."""
import pytest
from helpers import vsa_prefix

# (key cubes, prefix cubes, top-k, heads): us in one order for all cubes, us with the prefix's apart
TIMED = {
    (112, 28, 83, 18): (562, 703), (54, 27, 26, 4): (168, 210), (118, 64, 53, 2): (247, 303),
    (195, 33, 160, 8): (705, 821), (100, 28, 50, 6): (238, 272), (41, 1, 28, 18): (161, 181),
    (253, 125, 26, 3): (504, 566), (421, 70, 347, 17): (8301, 9122), (434, 38, 392, 8): (4217, 4539),
    (504, 4, 10, 40): (13000, 2108), (811, 1, 405, 17): (15397, 11074), (393, 3, 8, 29): (7938, 1089),
    (325, 109, 151, 35): (6655, 6255), (352, 1, 246, 7): (1478, 1383), (464, 16, 314, 1): (758, 724),
    (127, 1, 63, 1): (249, 235), (230, 80, 45, 3): (444, 425)}


@pytest.mark.parametrize("call", TIMED)
def test_prefix_cubes_go_apart_where_that_is_faster(call):
    blocks, cubes, topk, heads = call
    one, apart = TIMED[call]
    assert (vsa_prefix(heads, cubes, blocks, topk)[0] > 0) == (apart < one)


def test_ranges_fit_one_generation_and_the_plan():
    for heads in (1, 7, 32, 256):
        for blocks in (1, 9, 64, 387, 2112, 16384):
            for cubes in {0, 1, blocks // 3, blocks}:
                got, splits = vsa_prefix(heads, cubes, blocks, 4)
                assert got in (0, cubes) and 1 <= splits <= 16
                if splits > 1:
                    assert splits * heads * got <= 1024 and blocks // splits >= 8
