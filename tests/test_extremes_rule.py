"""Which layers take the lists of outermost values (csrc/extremes_forward.hip): those that were measured faster with them, by their
size alone.  Needs the library, not a GPU."""
import ctypes

import pytest

import __graft_entry__ as entry

WHAT = {"positions": 0, "values": 1, "bounds": 2}


def has_lists(B, CO, K, what):
    need = ctypes.c_int64(-1)
    assert entry.load_package()._lib.lib().ldist_inf_dist_workspace(B, CO, K, 1, 1, WHAT[what], ctypes.byref(need)) == 0
    return need.value > 0


@pytest.mark.parametrize("case", [(256, 256, 25088, "positions"), (1024, 64, 25088, "values"), (128, 512, 40000, "values"),
                                  (400, 128, 40000, "positions"), (2048, 17, 40000, "positions"), (400, 64, 25088, "bounds"),
                                  (128, 256, 25088, "bounds"), (64, 1024, 40000, "positions"), (600, 64, 25088, "bounds")])
def test_few_outputs_of_a_long_reduction(case):
    """1.3 to 2.2 times the time of the full walk, with lists, on inputs between 0 and 1."""
    assert not has_lists(*case)


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("shape", [(272, 5120, 5120), (512, 5120, 3072), (1024, 5120, 5120), (1280, 416, 36864), (300, 5000, 20000)])
def test_large_layers(shape, what):
    """A quarter to two thirds of the time."""
    assert has_lists(*shape, what)


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("shape", [(8, 5120, 5120), (1024, 10, 5120), (512, 5120, 511), (1024, 1024, 40961), (64, 256, 1024)])
def test_layers_without(shape, what):
    assert not has_lists(*shape, what)
