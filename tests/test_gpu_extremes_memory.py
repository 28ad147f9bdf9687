"""Scratch memory of the lists of outermost values (csrc/extremes_forward.hip): bounded, by taking large batches in parts, and not
needed where there is none."""
import ctypes

import pytest
import torch

import __graft_entry__ as entry

WHAT = {"positions": 0, "values": 1, "bounds": 2}
MOST = 256 << 20


def workspace(B, CO, K, what):
    need = ctypes.c_int64(-1)
    assert entry.load_package()._lib.lib().ldist_inf_dist_workspace(B, CO, K, 1, 1, WHAT[what], ctypes.byref(need)) == 0
    return need.value


@pytest.mark.parametrize("what", WHAT)
@pytest.mark.parametrize("shape", [(1024, 5120, 5120), (4096, 5120, 5120), (100000, 5120, 5120), (400000, 4096, 4096),
                                   (2000000, 1024, 1024), (16, 100000, 5120), (300, 80000, 20000), (257, 130000, 16000)])
def test_bounded_whatever_the_batch(shape, what):
    need = workspace(*shape, what)
    assert 0 <= need <= MOST
    if shape[0] >= 1024 and shape[2] > 1024:
        assert need > 0          # large batches are still taken this way


def run(forms, x, up, w):
    """The forms' results for whatever the library does now."""
    from gpu_common import DEV, cpp
    shape, out = (x.size(0), w.size(0), 1), {}
    for form in forms:
        a, b = torch.full(shape, float("nan"), device=DEV), torch.full(shape, float("nan"), device=DEV)
        if form == "positions":
            b = torch.full(shape, -7, device=DEV, dtype=torch.int32)
            cpp.inf_dist_forward(x, w, a, b, 1)
        elif form == "values":
            assert cpp.inf_dist_forward_values(x, w, a, 1)
            b = a
        else:
            cpp.inf_dist_bound_forward(x, up, w, a, b, 1)
        out[form] = (a, b)
    return out


def differing(got, want):
    return {form: sum(int((a != b).sum()) for a, b in zip(got[form], want[form])) for form in want}


@pytest.mark.gpu
@pytest.mark.parametrize("extension", [True, False])
def test_a_batch_in_parts_against_the_full_walk(extension):
    """Two or three parts of unequal size, of which the last rows are for the full walk: two values, like the weights."""
    from gpu_common import DEV, cpp, pkg, say
    B, CO, K = 16399, 2600, 3072
    say("extremes in parts", B, CO, K, extension)
    assert all(B * CO * 8 > MOST and 0 < workspace(B, CO, K, what) <= MOST for what in WHAT)
    g = torch.Generator(device=DEV).manual_seed(5)
    x, w = torch.randn(B, K, 1, device=DEV, generator=g), torch.randn(CO, K, device=DEV, generator=g) / K ** 0.5
    x[12000:] = (x[12000:] > 0) * 0.01
    w[:, :300] = w[:, :300].sign() * 0.1
    up = x + 0.1
    cpp.use_torch_extension(extension)
    try:
        got = run(WHAT, x, up, w)
        pkg._lib.lib().ldist_set_extremes(0)
        want = run(WHAT, x, up, w)
    finally:
        pkg._lib.lib().ldist_set_extremes(-1)
        cpp.use_torch_extension(True)
    assert differing(got, want) == dict.fromkeys(WHAT, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("extension", [True, False])
def test_no_memory_for_the_scratch(extension):
    """An allocator that has room for the results but not for the lists: the full walk, not an error."""
    from gpu_common import DEV, cpp, say
    B, CO, K = 1024, 5120, 5120
    say("extremes without memory", extension)
    g = torch.Generator(device=DEV).manual_seed(5)
    x, w = torch.randn(B, K, 1, device=DEV, generator=g), torch.randn(CO, K, device=DEV, generator=g) / K ** 0.5
    up = x + 0.1
    assert min(workspace(B, CO, K, what) for what in WHAT) > 30 << 20
    want = run(WHAT, x, up, w)
    a, b = torch.empty(B, CO, 1, device=DEV), torch.empty(B, CO, 1, device=DEV)
    pos = torch.empty(B, CO, 1, device=DEV, dtype=torch.int32)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    cpp.use_torch_extension(extension)
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (8 << 20)) / total)
    try:
        held = []                      # what the allocator has free inside its segments
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 1000:
                held.append(torch.empty(30 << 20, dtype=torch.uint8, device=DEV))
        cpp.inf_dist_forward(x, w, a, pos, 1)
        first = (a.cpu(), pos.cpu())
        assert cpp.inf_dist_forward_values(x, w, a, 1)
        second = a.cpu()
        cpp.inf_dist_bound_forward(x, up, w, a, b, 1)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        cpp.use_torch_extension(True)
    want = {form: [t.cpu() for t in tensors] for form, tensors in want.items()}
    assert [torch.equal(i, j) for i, j in zip(first, want["positions"])] == [True, True]
    assert torch.equal(second, want["values"][0])
    assert torch.equal(a.cpu(), want["bounds"][0]) and torch.equal(b.cpu(), want["bounds"][1])
