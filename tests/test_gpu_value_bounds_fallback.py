"""Values and bounds of a wide layer where the one pass through lists of outermost values (csrc/extremes_forward.hip) cannot be
taken, or is taken in parts: the same results, bit for bit, as without lists, and in no more memory than two passes need."""
import ctypes

import pytest
import torch

import __graft_entry__ as entry

MOST = 256 << 20


def workspace(B, CO, K):
    need = ctypes.c_int64(-1)
    assert entry.load_package()._lib.lib().ldist_inf_dist_value_bound_workspace(B, CO, K, 1, 1, ctypes.byref(need)) == 0
    return need.value


@pytest.mark.parametrize("shape", [(1024, 5120, 5120), (4096, 5120, 5120), (100000, 5120, 5120), (400000, 4096, 4096),
                                   (2000000, 1024, 1024), (16, 100000, 5120), (300, 80000, 20000), (257, 130000, 16000)])
def test_scratch_is_bounded_whatever_the_batch(shape):
    assert 0 <= workspace(*shape) <= MOST
    if shape[0] >= 1024 and shape[2] > 1024:
        assert workspace(*shape) > 0


def test_arguments_are_checked_without_a_device():
    lib = entry.load_package()._lib.lib()
    need, one = ctypes.c_int64(-1), ctypes.c_void_p(16)   # never dereferenced: the checks fail first
    assert lib.ldist_inf_dist_value_bound_workspace(1024, 5120, 5120, 1, 1, None) == -1
    for sizes, code in (((0, 64, 64, 1, 1), -1), ((4, 64, 65, 2, 1), -1), ((1 << 20, 1 << 12, 8, 1, 1), -2)):
        assert lib.ldist_inf_dist_value_bound_workspace(*sizes, ctypes.byref(need)) == code and need.value == 0
    for sizes in ((1024, 5120, 5121, 1, 1), (1024, 10, 5120, 1, 1), (1024, 5120, 5120, 2, 1), (1024, 5120, 5120, 1, 4), (16, 64, 64, 1, 1)):
        assert lib.ldist_inf_dist_value_bound_workspace(*sizes, ctypes.byref(need)) == 0 and need.value == 0

    def forward(sizes, x=one, ws=one):
        return lib.ldist_inf_dist_value_bound_forward_ws(x, one, one, one, *sizes, None, None, one, one, one, ws, 1 << 30, None)
    assert forward((1024, 5120, 5120, 1, 1), x=None) == -1 and forward((1024, 5120, 5120, 1, 1), ws=None) == -1
    assert forward((0, 5120, 5120, 1, 1)) == -1 and forward((1 << 20, 1 << 12, 8, 1, 1)) == -2


def layer_and_inputs(B, CO, CI, seed=5):
    from gpu_common import DEV, pkg
    g = torch.Generator(device=DEV).manual_seed(seed)
    layer = pkg.NormDist(CI, CO, p=float("inf"), bias=True, mean_normalize=True).to(DEV).eval()
    with torch.no_grad():
        layer.weight.copy_((torch.randn(CO, CI, device=DEV, generator=g) / CI ** 0.5).view_as(layer.weight))
        layer.bias.normal_(0, 0.1, generator=g)
        layer.normalize.running_mean.normal_(0, 0.1, generator=g)
    return layer, torch.randn(B, CI, device=DEV, generator=g)


def in_full(layer, *triple):
    from gpu_common import pkg
    pkg._lib.lib().ldist_set_extremes(0)
    try:
        return layer(*triple)
    finally:
        pkg._lib.lib().ldist_set_extremes(-1)


ONE_PASS, TWO = {"values": "one_pass", "bounds": "one_pass"}, {"values": "columns", "bounds": "columns"}


@pytest.mark.gpu
@torch.no_grad()
def test_a_batch_in_parts():
    """Parts of unequal size; the last rows, two values like the weights, are for the full walks of either."""
    from gpu_common import say
    B, CO, CI = 12301, 2600, 3072
    say("values and bounds in parts", B, CO, CI)
    assert B * CO * 12 > MOST and 0 < workspace(B, CO, CI) <= MOST
    layer, x = layer_and_inputs(B, CO, CI)
    x[9000:] = (x[9000:] > 0) * 0.01
    layer.weight[:, :300] = layer.weight[:, :300].sign() * 0.1
    triple = (x, x - 0.1, x + 0.1)
    got = layer(*triple)
    assert layer.last_route == ONE_PASS
    assert [int((a != b).sum()) for a, b in zip(got, in_full(layer, *triple))] == [0, 0, 0]


@pytest.mark.gpu
@torch.no_grad()
@pytest.mark.parametrize("which", range(4))
def test_tensors_that_128_bit_loads_do_not_reach(which):
    """One of input, ends of the boxes and weight four bytes off a 16-byte boundary."""
    from gpu_common import DEV, say
    B, CO, CI = 300, 4104, 5120
    say("values and bounds, misaligned", which)
    layer, x = layer_and_inputs(B, CO, CI)
    tensors = [x, x - 0.1, x + 0.1, layer.weight.data]
    room = torch.empty(tensors[which].numel() + 1, device=DEV)[1:]
    tensors[which] = room.view_as(tensors[which]).copy_(tensors[which])
    layer.weight.data = tensors[3]
    got = layer(*tensors[:3])
    assert layer.last_route == (TWO if which in (0, 3) else ONE_PASS)   # the boxes are read in single words
    for a, b in zip(got, in_full(layer, *tensors[:3])):
        assert torch.equal(a, b)


@pytest.mark.gpu
@torch.no_grad()
def test_no_memory_for_the_scratch():
    """An allocator that has room for three results, and neither for the lists beside them nor for a fourth."""
    from gpu_common import DEV, say
    B, CO, CI = 1024, 5120, 5120
    result = B * CO * 4
    say("values and bounds without memory")
    layer, x = layer_and_inputs(B, CO, CI)
    triple = (x, x - 0.1, x + 0.1)
    want = [t.cpu() for t in layer(*triple)]
    assert layer.last_route == ONE_PASS and workspace(B, CO, CI) > 2 * result
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 3 * result + (16 << 20)) / total)
    try:
        held = []                      # what the allocator has free inside its segments, and what was put aside for the results
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 1000:
                held.append(torch.empty(result, dtype=torch.uint8, device=DEV))
        del held[-3:]
        got = layer(*triple)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert layer.last_route == TWO
    for a, b in zip(got, want):
        assert torch.equal(a.cpu(), b)
