"""Which tile the p-norm forward that trains takes for few rows and outputs (csrc/norm_forward.hip): the one that was measured
fastest, by size and exponent alone.  Needs the library, not a GPU."""
import ctypes

import pytest

import __graft_entry__ as entry

CUS = 256


def tile(B, CO, CI, p, G=1):
    got = entry.load_package()._lib.lib().ldist_which_forward_tile(B, CO, CI, G, ctypes.c_float(p), CUS)
    return divmod(got, 1000) if got > 0 else got


# Rows, outputs, inputs; the tile that 16 x 16 would replace.  Three and five rounds of it took, as a share of that tile's time,
# 1.10 to 1.20 at p = 2, 1.12 to 1.18 at 3 and 4, 1.01 to 1.16 at 8, and 0.92 to 0.99 at any other exponent.
SEVERAL_ROUNDS = [(64, 3072, 5120, (32, 32)), (48, 4096, 4096, (32, 32)), (96, 2048, 2048, (32, 32)), (192, 1024, 1024, (32, 32)),
                  (32, 5120, 3072, (32, 32)), (128, 1536, 2048, (32, 32)), (80, 4096, 4096, (16, 32)), (65, 4096, 4096, (16, 32))]


@pytest.mark.parametrize("case", SEVERAL_ROUNDS)
def test_several_rounds_of_the_smallest_tile(case):
    B, CO, CI, other = case
    for p in (2.0, 3.0, 4.0, 8.0):
        assert tile(B, CO, CI, p) == other
    for p in (1.5, 5.0, 7.0, 16.0, 37.3, 300.0, 1000.0):
        assert tile(B, CO, CI, p) == (16, 16)


def test_short_or_unaligned_reductions_in_several_rounds():
    """64 x 511 -> 3072 at p = 37.3: 16 x 16 3 % slower."""
    assert tile(64, 3072, 511, 37.3) == (32, 32) and tile(64, 3072, 256, 37.3) == (32, 32)


# the first seven are those of tests/test_gpu_eight_groups.py, which are there for this tile: they have to take it
@pytest.mark.parametrize("case", [(33, 300, 300, 1), (17, 63, 257, 1), (64, 500, 516, 1), (1, 17, 2053, 1), (100, 64, 1030, 2),
                                  (40, 35, 31, 1), (128, 512, 256, 1), (128, 512, 16384, 1), (64, 1024, 3072, 1), (16, 1024, 784, 1),
                                  (16, 4096, 4096, 1), (9, 4096, 1024, 1)])
def test_one_round_of_the_smallest_tile(case):
    """0.6 to 0.66 of the time of 16 x 32 at every exponent."""
    B, CO, CI, G = case
    for p in (2.0, 3.0, 4.0, 8.0, 1.5, 37.3, 500.0):
        assert tile(B, CO, CI, p, G) == (16, 16)


def test_other_kernels_and_refused_arguments():
    assert tile(512, 5120, 5120, 8.0) == 0 and tile(64, 10, 5120, 8.0) == 0
    assert tile(64, 5120, 5120, 8.0) == (32, 40) and tile(24, 3072, 5120, 8.0) == (16, 32)
    assert tile(0, 64, 64, 8.0) == -1 and tile(4, 64, 64, 1.0) == -1 and tile(4, 64, 65, 8.0, 2) == -1
