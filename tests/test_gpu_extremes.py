"""The L_inf forward passes that evaluate only what lists of outermost values leave possible (csrc/extremes_forward.hip):
forced onto small layers at the edges of chunks, strips, lane groups and list blocks, and chosen by the library on layers
where its sample sends the work to the lists, to the full walk, or first to the one and then to the other.  Everything bit for bit,
against the oracle and, at full size, against the full walk."""
import pytest
import torch

import oracle
from helpers import gen, make_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset():
    from gpu_common import pkg
    yield
    pkg._lib.lib().ldist_set_extremes(-1)


def set_extremes(choice):
    from gpu_common import pkg
    assert pkg._lib.lib().ldist_set_extremes(choice) == 0


def values(x, w):
    from gpu_common import DEV, cpp
    out = torch.full((x.size(0), w.size(0), 1), float("nan"), device=DEV)
    return out.cpu() if not cpp.inf_dist_forward_values(x.to(DEV), w.to(DEV), out, 1) else out.cpu()


# B, CO, CI: rows and outputs around strips of 8 (boxes: 4), blocks of 16, waves and lane groups of 64 to 512; k around
# vectors, waves, chunk widths (1024, 1536, 2048, 2560) and two or three chunks
SHAPES = [(1, 17, 4), (7, 33, 63), (8, 64, 65), (9, 130, 1000), (17, 257, 1025), (65, 40, 1537), (129, 72, 2049), (70, 100, 2560),
          (33, 81, 2561), (12, 530, 2564), (515, 23, 300), (20, 48, 5121), (260, 18, 5200)]


@pytest.mark.parametrize("kind", ["plain", "ties", "offset", "heavy"])
@pytest.mark.parametrize("shape", SHAPES)
def test_forced_lists(shape, kind):
    from gpu_common import gpu_bound_forward, gpu_inf_forward, say
    B, CO, CI = shape
    say("extremes", shape, kind)
    x, w = make_inputs(B, CO, CI, 1, 1, seed=sum(shape), quantize=4 if kind == "ties" else None)
    if kind == "offset":                      # far from zero, and rows of very different spread
        x = (x * torch.logspace(-3, 2, B).view(B, 1, 1) + 7).contiguous()
        w = (w + 5).contiguous()
    if kind == "heavy":                       # a few values far beyond the histogram's octaves
        x = torch.where(torch.rand(x.shape, generator=gen(1)) < 0.003, x * 1e4, x).contiguous()
        w = torch.where(torch.rand(w.shape, generator=gen(2)) < 0.003, w * 1e6, w).contiguous()
    set_extremes(1)
    ev, ep = oracle.inf_dist_forward(x, w, 1)
    out, pos = gpu_inf_forward(x, w, 1)
    assert torch.equal(out, ev) and torch.equal(pos, ep)
    if CI % 4 == 0:
        assert torch.equal(values(x, w), ev)
    half = 0.1 * torch.rand(x.shape, generator=gen(3)) if kind != "ties" else torch.full_like(x, 0.25)
    lo, up = (x - half).contiguous(), (x + half).clamp(max=float(x.max())).contiguous()
    up = torch.maximum(lo, up).contiguous()
    for got, want in zip(gpu_bound_forward(lo, up, w, 1), oracle.inf_dist_bound_forward(lo, up, w, 1)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("shape", [(9, 130, 1000), (33, 81, 2561), (65, 40, 5120)])
def test_forced_lists_with_nan_infinities_and_reversed_boxes(shape):
    from gpu_common import gpu_bound_forward, gpu_inf_forward, say
    B, CO, CI = shape
    say("extremes, irregular", shape)
    x, w = make_inputs(B, CO, CI, 1, 1, seed=3)
    lo, up = (x - 0.1).contiguous(), (x + 0.1).contiguous()
    flip = torch.rand(x.shape, generator=gen(4)) < 0.05
    lo, up = torch.where(flip, up, lo), torch.where(flip, lo, up)
    lo[B // 2:], up[B // 2:] = x[B // 2:] - 0.1, x[B // 2:] + 0.1      # regular rows beside them
    lo[0, 0, 0], up[B - 1, CI - 1, 0], w[CO - 1, CI - 1], w[0, 5], lo[1] = (float("nan"), float("inf"), float("-inf"),
                                                                         float("nan"), float("nan"))
    lo, up = lo.contiguous(), up.contiguous()
    set_extremes(1)
    for got, want in zip(gpu_bound_forward(lo, up, w, 1), oracle.inf_dist_bound_forward(lo, up, w, 1)):
        assert torch.equal(torch.nan_to_num(got, nan=-1.0), torch.nan_to_num(want, nan=-1.0))
    out, pos = gpu_inf_forward(lo, w, 1)
    ev, ep = oracle.inf_dist_forward(lo, w, 1)
    assert torch.equal(out, ev) and torch.equal(pos, ep)
    zero = torch.zeros(B, CI, 1)               # every difference is zero: position 0, and no list passes
    out, pos = gpu_inf_forward(zero, torch.zeros(CO, CI), 1)
    assert not out.any() and not pos.any()


# Layers that the library sends this way by itself.  "two values": the bound is attained everywhere, the sample says so;
# "unsampled": the sampled rows are ordinary and the others are not.
@pytest.mark.parametrize("data", ["uniform", "two values", "unsampled", "nan"])
@pytest.mark.parametrize("shape", [(500, 5120, 3072), (300, 4104, 5120)])
def test_chosen_by_the_library(shape, data):
    from gpu_common import DEV, cpp, say
    B, CO, CI = shape
    say("extremes, chosen", shape, data)
    g = torch.Generator(device=DEV).manual_seed(5)
    x = (torch.rand(B, CI, 1, device=DEV, generator=g) - 0.47) / 0.2
    w = torch.randn(CO, CI, device=DEV, generator=g) / CI ** 0.5
    if data == "two values":
        x, w = torch.sign(x), torch.sign(w)
    if data == "unsampled":
        keep = torch.arange(64, device=DEV) * B // 64
        y = torch.sign(x)
        y[keep] = x[keep]
        kept = torch.arange(64, device=DEV) * CO // 64
        v = torch.sign(w)
        v[kept] = w[kept]
        x, w = y, v
    if data == "nan":
        x[3, 7] = float("nan")
    lo, up = x - 0.1, x + 0.1

    def passes():
        out, pos = torch.empty(B, CO, 1, device=DEV), torch.empty(B, CO, 1, device=DEV, dtype=torch.int32)
        only, a, b = torch.empty_like(out), torch.empty_like(out), torch.empty_like(out)
        cpp.inf_dist_forward(x, w, out, pos, 1)
        cpp.inf_dist_forward_values(x, w, only, 1)
        cpp.inf_dist_bound_forward(lo, up, w, a, b, 1)
        return out, pos, only, a, b

    set_extremes(-1)
    need = [workspace(B, CO, CI, what) for what in range(3)]
    assert all(n > 0 for n in need)
    got = passes()
    set_extremes(0)
    for a, b in zip(got, passes()):
        assert torch.equal(torch.nan_to_num(a, nan=-1.0) if a.is_floating_point() else a,
                           torch.nan_to_num(b, nan=-1.0) if b.is_floating_point() else b)


def workspace(B, CO, CI, what, G=1, HW=1):
    import ctypes

    from gpu_common import pkg
    need = ctypes.c_int64(-1)
    assert pkg._lib.lib().ldist_inf_dist_workspace(B, CO, CI, G, HW, what, ctypes.byref(need)) == 0
    return need.value


def test_replays_of_a_captured_graph():
    from gpu_common import DEV, cpp
    B, CO, CI = 300, 4104, 5120
    g = torch.Generator(device=DEV).manual_seed(6)
    x, w = torch.rand(B, CI, 1, device=DEV, generator=g), torch.randn(CO, CI, device=DEV, generator=g)
    out, pos = torch.empty(B, CO, 1, device=DEV), torch.empty(B, CO, 1, device=DEV, dtype=torch.int32)
    cpp.inf_dist_forward(x, w, out, pos, 1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        cpp.inf_dist_forward(x, w, out, pos, 1)
    for seed in range(3):
        g.manual_seed(seed)
        x.copy_(torch.sign(torch.randn(x.shape, device=DEV, generator=g)) if seed == 1 else torch.rand(x.shape, device=DEV, generator=g))
        if seed == 1:
            w.sign_()
        graph.replay()
        torch.cuda.synchronize()
        want, at = torch.empty_like(out), torch.empty_like(pos)
        set_extremes(0)
        cpp.inf_dist_forward(x, w, want, at, 1)
        set_extremes(-1)
        assert torch.equal(out, want) and torch.equal(pos, at)
