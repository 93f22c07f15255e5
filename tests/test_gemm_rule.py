"""The rule that picks the projection's tiling (a host function) against shapes timed on every tiling on
256 CUs, behind the output quantizer in captured graphs."""
import pytest
from helpers import gemm_tiling

# (tokens, channels, K): us on 256 x 256, on 128 x 128 with two ring stages, on four
TIMED = {
    # many tiles over large operands: 128 x 128 read A and W more often
    (34453, 5760, 1984): (520, 611, 662), (60216, 3456, 2304): (576, 655, 680),
    (28355, 5760, 2048): (402, 459, 489), (19587, 9984, 1536): (406, 454, 497),
    (62324, 1920, 2112): (368, 406, 424), (17609, 7296, 1536): (285, 291, 333),
    # many tiles over operands that stay behind the L2s
    (23844, 2304, 1280): (131, 112, 129), (9972, 5376, 1024): (121, 98, 120),
    # too few tiles for 256 x 256
    (129, 12288, 4096): (57, 29, 22), (513, 12288, 4096): (64, 41, 44),
    (1025, 12288, 4096): (76, 73, 77), (2049, 21504, 1024): (113, 87, 108),
    # one round and more
    (641, 21504, 7168): (110, 120, 124), (5000, 12288, 4096): (246, 279, 298)}


@pytest.mark.parametrize("shape", TIMED)
def test_the_tiling_is_within_five_percent_of_the_best(shape):
    at = dict(zip(("256x256", "128x128 ring 2", "128x128 ring 4"), TIMED[shape]))
    assert at[gemm_tiling(*shape)] <= 1.05 * min(at.values())


def test_small_calls_take_the_small_tilings():
    assert gemm_tiling(1, 12288, 4096) == gemm_tiling(32, 384, 64) == "few"
    assert gemm_tiling(33, 6144, 4096) == "64x128"
    assert gemm_tiling(33, 12288, 4096) == "128x128 ring 4"
    assert gemm_tiling(16777216, 65280, 65536) == "256x256"
