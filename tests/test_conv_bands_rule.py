"""Into how many bands of output rows the one-pass p-norm conv backward cuts an image (csrc/norm_conv_backward.hip): by what the
busiest CU has to work through with as many workgroups as LDS admits.  Needs the library, not a GPU."""
import ctypes

import pytest

import __graft_entry__ as entry
from test_gpu_conv_bands import CASES

CUS = 256


def bands(B, C, H, W, CO, G=1, stride=1, padding=1, dilation=1, p=8.0):
    return entry.load_package()._lib.lib().ldist_which_conv_bands(B, C, H, W, CO, G, stride, padding, dilation, ctypes.c_float(p), CUS)


# one workgroup to a CU, or two and an odd third: bands took 1.07 to 1.45 times the time of whole images
@pytest.mark.parametrize("case", [(20, 64, 32, 32, 128), (64, 32, 32, 32, 128, 2), (115, 8, 10, 22, 242, 2), (37, 40, 37, 26, 150, 2),
                                  (56, 24, 38, 22, 113), (31, 60, 33, 33, 224, 4), (194, 6, 39, 23, 176, 2)])
def test_whole_images(case):
    assert bands(*case) == 1


# one workgroup to a CU: bands beyond one round of them run in turn, each with its halo (0.78 to 0.89 of the time with fewer)
@pytest.mark.parametrize("case,want", [((64, 3, 32, 32, 128), 4), ((128, 3, 32, 32, 128), 2), ((32, 3, 32, 32, 128), 8), ((59, 3, 24, 16, 128), 3),
                                       ((16, 22, 38, 40, 89), 4), ((31, 16, 19, 33, 133), 2)])
def test_a_round_of_bands(case, want):
    assert bands(*case) == want


@pytest.mark.parametrize("case,want", [((128, 3, 32, 32, 32), 4), ((16, 32, 32, 32, 32), 6), ((48, 32, 32, 32, 32), 2), ((20, 64, 32, 32, 64), 2),
                                       ((77, 32, 32, 32, 32), 1), ((128, 128, 32, 32, 128, 4), 1)])
def test_several_workgroups_to_a_cu(case, want):
    assert bands(*case) == want


@pytest.mark.parametrize("case", CASES)
def test_the_geometries_of_the_gpu_tests_are_cut(case):
    lib = entry.load_package()._lib.lib()
    assert lib.ldist_set_tile_override(0) == 0
    try:
        assert bands(*case) > 1
    finally:
        lib.ldist_set_tile_override(-1)


def test_other_kernels_and_refused_arguments():
    assert bands(1, 3, 32, 32, 32) == 0 and bands(0, 3, 32, 32, 32) == -1 and bands(64, 3, 32, 32, 32, p=1.0) == -1
    assert bands(64, 3, 32, 32, 32, 2) == -1 and bands(64, 3, 1, 1, 32, padding=0) == -1
