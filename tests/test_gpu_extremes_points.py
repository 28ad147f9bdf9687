"""Values and bounds from one set of lists of outermost values (csrc/extremes_forward.hip, boxes and the points inside them):
forced onto small layers at the edges of chunks, strips, lane groups and list blocks, and chosen by the library.  Bit for bit."""
import pytest
import torch

import oracle
from helpers import gen, make_inputs

pytestmark = pytest.mark.gpu

# rows and outputs around strips of 8 (second scan: 4 and 8), blocks of 16, waves and lane groups; k around vectors, waves and chunks
SHAPES = [(1, 17, 4), (7, 33, 64), (9, 130, 1000), (17, 257, 1028), (65, 40, 1540), (70, 100, 2560), (33, 81, 2564), (12, 530, 2564),
          (515, 23, 300), (20, 48, 5124), (260, 18, 5200)]


@pytest.fixture(autouse=True)
def _reset():
    from gpu_common import pkg
    yield
    pkg._lib.lib().ldist_set_extremes(-1)


def shifted(v, mean, bias):
    return (v - mean.view(1, -1, 1)) + bias.view(1, -1, 1)


# "longer w": a few weights far out, so that both operands have lists and the first scan's results go through the second
@pytest.mark.parametrize("kind", ["plain", "longer w", "ties", "outside", "irregular"])
@pytest.mark.parametrize("shape", SHAPES)
def test_forced_lists(shape, kind):
    from gpu_common import gpu_value_bound_forward, pkg, say
    B, CO, CI = shape
    say("extremes, points", shape, kind)
    x, w = make_inputs(B, CO, CI, 1, 1, seed=sum(shape), quantize=4 if kind == "ties" else None)
    if kind == "longer w":
        w = (w * 20).contiguous()
    half = 0.1 * torch.rand(x.shape, generator=gen(3)) if kind != "ties" else torch.full_like(x, 0.25)
    lo, up = (x - half).contiguous(), torch.maximum(x - half, (x + half).clamp(max=float(x.max()))).contiguous()
    if kind == "outside":      # points need not lie in their boxes
        x = torch.where(torch.rand(x.shape, generator=gen(5)) < 0.1, x * 3 - 1, x).contiguous()
    if kind == "irregular":
        lo[0, 0, 0], up[B - 1, CI - 1, 0], x[B // 2, CI // 2, 0] = float("nan"), float("inf"), float("nan")
        lo[B // 3], up[B // 3] = up[B // 3].clone(), lo[B // 3].clone()
        w[CO - 1, CI - 1] = float("-inf")
    mean, bias = torch.randn(CO, generator=gen(6)), torch.randn(CO, generator=gen(7))
    values, _ = oracle.inf_dist_forward(x, w, 1)
    want = (values, *oracle.inf_dist_bound_forward(lo, up, w, 1))
    assert pkg._lib.lib().ldist_set_extremes(1) == 0
    for m, b in ((None, None), (mean, bias)):
        for got, expected in zip(gpu_value_bound_forward(x, lo, up, w, 1, m, b), want):
            if m is not None:
                expected = shifted(expected, m, b)
            assert torch.equal(torch.nan_to_num(got, nan=-1.0), torch.nan_to_num(expected, nan=-1.0))


# the sample sends the first to the lists and the second to the full walk, which the third gets to after its lists
@pytest.mark.parametrize("data", ["uniform", "two values", "unsampled"])
def test_layers_chosen_by_the_library(data):
    from gpu_common import DEV, pkg, say
    B, CO, CI = 300, 4104, 5120
    say("extremes, points, chosen", data)
    g = torch.Generator(device=DEV).manual_seed(5)
    x = (torch.rand(B, CI, device=DEV, generator=g) - 0.47) / 0.2
    layer = pkg.NormDist(CI, CO, p=float("inf"), bias=True, mean_normalize=True).to(DEV).eval()
    with torch.no_grad():
        w = torch.randn(CO, CI, device=DEV, generator=g) / CI ** 0.5
        if data != "uniform":
            y, v = torch.sign(x), torch.sign(w)
            if data == "unsampled":
                keep, kept = torch.arange(64, device=DEV) * B // 64, torch.arange(64, device=DEV) * CO // 64
                y[keep], v[kept] = x[keep], w[kept]
            x, w = y, v
        layer.weight.copy_(w.view_as(layer.weight))
        layer.bias.normal_(0, 0.1, generator=g)
        layer.normalize.running_mean.normal_(0, 0.1, generator=g)
        got = layer(x, x - 0.1, x + 0.1)
        assert layer.last_route == {"values": "one_pass", "bounds": "one_pass"}
        assert pkg._lib.lib().ldist_set_extremes(0) == 0
        for a, b in zip(got, layer(x, x - 0.1, x + 0.1)):
            assert torch.equal(a, b)
        assert layer.last_route == {"values": "columns", "bounds": "columns"}
