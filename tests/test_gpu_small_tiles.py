"""The forward kernels for layers that do not fill the device (csrc/small_forward.hip: small tiles with the reduction split
over k-groups; csrc/few_rows_forward.hip: a handful of rows), every tile forced, at the sizes where they can go wrong:
tails of rows, outputs and k, k not a multiple of four, k shorter than a vector group, groups, ties between k-groups,
NaN and infinities.  L_inf values, indices and bounds against the oracle bit for bit, p-norm within rel 1e-5 / abs 1e-6."""
import pytest
import torch

import oracle
from helpers import gen, make_inputs

pytestmark = pytest.mark.gpu
KERNELS = [10, 11, 12, 13, 14, 15, 16, 30]   # ldist_set_tile_override: the seven small tiles, the few-rows kernel
# B, CO, CI, G
SHAPES = [(1, 17, 4, 1), (3, 33, 7, 1), (8, 100, 63, 1), (9, 41, 129, 1), (17, 80, 257, 1), (33, 81, 1001, 1),
          (65, 64, 64, 1), (40, 90, 512, 2), (6, 120, 390, 3)]


@pytest.fixture(autouse=True)
def _reset_tile():
    from gpu_common import set_tile
    yield
    set_tile(-1)


@pytest.mark.parametrize("tile", KERNELS)
@pytest.mark.parametrize("shape", SHAPES)
def test_small_forward_kernels(shape, tile):
    from gpu_common import gpu_bound_forward, gpu_inf_forward, gpu_norm_forward, say, set_tile
    B, CO, CI, G = shape
    say("small forward", shape, "tile", tile)
    set_tile(tile)
    for quant in (None, 4):   # quantised: many equal maxima, within one k-group and across them
        x, w = make_inputs(B, CO, CI, G, 1, seed=sum(shape), quantize=quant)
        out, pos = gpu_inf_forward(x, w, G)
        ev, ep = oracle.inf_dist_forward(x, w, G)
        assert torch.equal(out, ev) and torch.equal(pos, ep)
    lo, up = (x - 0.1).contiguous(), (x + 0.1).contiguous()
    for irregular in (False, True):
        if irregular:
            flip = torch.rand(x.shape, generator=gen(4)) < 0.05
            lo, up = torch.where(flip, up, lo).contiguous(), torch.where(flip, lo, up).contiguous()
            lo[0, 0, 0], up[-1, -1, -1], w[-1, -1] = float("nan"), float("inf"), float("-inf")
        ol, ou = gpu_bound_forward(lo, up, w, G)
        el, eu = oracle.inf_dist_bound_forward(lo, up, w, G)
        for a, b in ((ol, el), (ou, eu)):
            assert torch.equal(torch.nan_to_num(a, nan=-1.0), torch.nan_to_num(b, nan=-1.0))
    # NaN differences never win; infinities do
    out, pos = gpu_inf_forward(lo, w, G)
    ev, ep = oracle.inf_dist_forward(lo, w, G)
    assert torch.equal(out, ev) and torch.equal(pos, ep)
    x, w = make_inputs(B, CO, CI, G, 1, seed=sum(shape) + 1)
    for p, scale in ((8.0, 1.0), (3.0, 1.0), (8.0, 1e-7), (4.0, 1e9), (37.3, 1.0), (1.5, 1.0), (500.0, 1e-3)):
        xs, ws = (x * scale).contiguous(), (w * scale).contiguous()
        got, want = gpu_norm_forward(xs, ws, G, p), oracle.norm_dist_forward(xs, ws, G, p)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-6 * min(1.0, scale))


@pytest.mark.parametrize("shape", [(70, 100, 2051, 1), (5, 40, 2200, 1)])
@pytest.mark.parametrize("tile", [12, 13, 30])
def test_long_reductions_at_large_exponents_pass_over_small_terms(shape, tile):
    from gpu_common import gpu_norm_forward, say, set_tile
    B, CO, CI, G = shape
    say("small forward, large p", shape, "tile", tile)
    set_tile(tile)
    x, w = make_inputs(B, CO, CI, G, 1, seed=5)
    x[0], w[0] = 0.25, 0.25                       # an output of exactly 0 stays on the reference's seeds
    for p in (128.0, 1000.0):
        got, want = gpu_norm_forward(x, w, G, p), oracle.norm_dist_forward(x, w, G, p)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-6)


# The forward pass without gradients at the kernel that the library chooses by itself: a few rows, small tiles, the large
# tiles, a handful of outputs, k that is odd or shorter than a vector, a window's positions.
@pytest.mark.parametrize("p", [2.0, 3.0, 8.0, 37.3, 300.0])
@pytest.mark.parametrize("shape", [(1, 1000, 1030, 1, 1), (5, 40, 3, 1, 1), (33, 130, 258, 2, 1), (100, 513, 2051, 1, 1),
                                   (1030, 700, 64, 1, 1), (40, 10, 400, 1, 1), (6, 48, 54, 2, 35)])
def test_values_without_gradients(shape, p):
    from gpu_common import DEV, cpp, say
    B, CO, CI, G, HW = shape
    say("values", shape, "p", p)
    x, w = make_inputs(B, CO, CI, G, HW, seed=sum(shape))
    got = torch.full((B, CO, HW), float("nan"), device=DEV)
    cpp.norm_dist_forward_values(x.to(DEV), w.to(DEV), got, G, p)
    torch.testing.assert_close(got.cpu(), oracle.norm_dist_forward(x, w, G, p), rtol=1e-5, atol=1e-6)
