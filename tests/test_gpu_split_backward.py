"""p-norm gradients whose reduction is shared out over workgroups: the one-pass kernel (csrc/norm_backward_fused.hip) and the
grad_input of the general kernel (csrc/norm_backward_kernel.hpp) at the edges of their tiles and shares, against the oracle: one row to one
past a tile, outputs that end inside a stage and inside a share, four inputs to one vector past a tile, groups."""
import pytest
import torch

import oracle
from helpers import assert_sum_close, gen, make_inputs

pytestmark = pytest.mark.gpu
# B, CO, CI, G
ONE_PASS = [(1, 128, 4, 1), (8, 132, 60, 1), (33, 260, 68, 1), (64, 1028, 64, 1), (65, 196, 132, 1), (7, 280, 128, 2),
            (129, 644, 4, 1), (2, 4100, 12, 1)]
SEPARATE = [(1, 300, 5, 1), (33, 1000, 63, 1), (40, 390, 130, 2), (65, 1100, 31, 1), (100, 513, 67, 1)]


@pytest.mark.parametrize("p", [3.0, 4.0, 8.0, 37.3, 62.0, 300.0])
@pytest.mark.parametrize("shape", ONE_PASS + SEPARATE)
def test_shared_reductions(shape, p):
    from gpu_common import DEV, cpp, say
    B, CO, CI, G = shape
    say("split backward", shape, "p", p)
    x, w = make_inputs(B, CO, CI, G, 1, seed=sum(shape))
    go = torch.randn(B, CO, 1, generator=gen(7))
    out = oracle.norm_dist_forward(x, w, G, p)
    ex, mx = oracle.norm_dist_backward_input(go, x, w, out, G, p, with_abs_terms=True)
    ew, mw = oracle.norm_dist_backward_weight(go, x, w, out, G, p, with_abs_terms=True)
    args = [t.to(DEV) for t in (go, x, w, out)]
    for both in (True, False):
        gx = torch.full((B, CI, 1), float("nan"), device=DEV)   # overwritten, whatever it held
        gw = torch.full((CO, CI // G), 0.125, device=DEV)       # added to
        if both:
            cpp.norm_dist_backward(*args, gx, gw, G, p)
        else:
            cpp.norm_dist_backward_input(*args, gx, G, p)
            cpp.norm_dist_backward_weight(*args, gw, G, p)
        torch.cuda.synchronize()
        assert_sum_close(gx.cpu(), ex, mx, p, 1e-5, 1e-6)
        assert_sum_close(gw.cpu() - 0.125, ew, mw, p, 1e-5, 1e-6)


# 16 x 32 tiles, 32 x 40 tiles (their busiest CU has least to do there), ragged ends of both
@pytest.mark.parametrize("p", [2.0, 8.0, 37.3, 200.0])
@pytest.mark.parametrize("shape", [(17, 33, 260, 1), (100, 1001, 513, 1), (30, 66, 1000, 2), (64, 5117, 300, 1), (61, 5120, 2052, 1)])
def test_forward_tiles_of_eight_groups(shape, p):
    from gpu_common import gpu_norm_forward, say
    B, CO, CI, G = shape
    say("eight groups", shape, "p", p)
    x, w = make_inputs(B, CO, CI, G, 1, seed=sum(shape))
    got = gpu_norm_forward(x, w, G, p)
    torch.testing.assert_close(got, oracle.norm_dist_forward(x, w, G, p), rtol=1e-5, atol=1e-6)


# Groups that a workgroup takes whole, in chunks and in blocks: with workgroups for several per CU, 96 and 200 outputs go in
# blocks, 40 and 64 in chunks; with one or two per CU they stay whole as far as LDS reaches (270 and 300 do not fit whole).
@pytest.mark.parametrize("p", [8.0, 37.3])
@pytest.mark.parametrize("case", [(600, 2, 3, 4, 40), (800, 1, 3, 3, 64), (600, 2, 3, 4, 96), (520, 1, 4, 4, 200), (300, 1, 4, 5, 33),
                                  (280, 3, 4, 4, 67), (9, 8, 5, 7, 130), (5, 2, 6, 6, 270), (3, 10, 5, 5, 300)])
def test_conv_backward_in_pieces(case, p):
    from test_gpu_parity import test_norm_conv_backward_both_gradients_in_one_pass_from_the_image as from_the_image
    B, C, H, W, outputs = case
    from_the_image((B, C, H, W, outputs, 1, 1, 1, 1), p)


# Large groups left to the library: the two separate kernels where the layer has few images or column tiles, blocks in one pass
# where it fills the device.
@pytest.mark.parametrize("p", [3.0, 20.5])
@pytest.mark.parametrize("case", [(17, 4, 31, 33, 171), (260, 7, 8, 8, 170), (520, 9, 6, 7, 150)])
def test_conv_backward_of_large_groups(case, p):
    import torch.nn.functional as F
    from gpu_common import DEV, cpp, say
    B, C, H, W, outputs = case
    say("large group", case, "p", p)
    g = gen(sum(case))
    img, w = torch.rand(B, C, H, W, generator=g), torch.randn(outputs, C * 9, generator=g) / (C * 9) ** 0.5
    cols = F.unfold(img, 3, 1, 1, 1).contiguous()
    go = torch.randn(B, outputs, H * W, generator=g)
    out = oracle.norm_dist_forward(cols, w, 1, p)
    ex, mx = oracle.norm_dist_backward_input(go, cols, w, out, 1, p, with_abs_terms=True)
    ew, mw = oracle.norm_dist_backward_weight(go, cols, w, out, 1, p, with_abs_terms=True)
    fold = lambda t: F.fold(t.double(), (H, W), 3, 1, 1, 1)
    gi, gw = torch.full((B, C, H, W), float("nan"), device=DEV), torch.zeros((outputs, C * 9), device=DEV)
    cpp.norm_dist_conv_backward(*(t.to(DEV) for t in (go, img, w, out)), gi, gw, 1, p, 3, 1, 1, 1)
    gx, gc = torch.full(cols.shape, float("nan"), device=DEV), torch.zeros_like(gw)
    cpp.norm_dist_backward(*(t.to(DEV) for t in (go, cols, w, out)), gx, gc, 1, p)
    torch.cuda.synchronize()
    assert_sum_close(gi.cpu(), fold(ex), fold(mx), p, 1e-5, 1e-6)
    assert_sum_close(gx.cpu(), ex, mx, p, 1e-5, 1e-6)
    for got in (gw, gc):
        assert_sum_close(got.cpu(), ew, mw, p, 1e-5, 1e-6)


# More outputs per group than one block of 64 holds: just over it, equal blocks, a short last one.
@pytest.mark.parametrize("p", [8.0, 5.5, 37.3])
@pytest.mark.parametrize("outputs", [65, 96, 257])
def test_conv_backward_in_blocks_of_outputs(outputs, p):
    from gpu_common import DEV, cpp, say, set_tile
    from test_gpu_parity import test_norm_conv_backward_both_gradients_in_one_pass_from_the_image as from_the_image
    try:
        from_the_image((2, 10, 11, 9, outputs, 1, 2 if outputs == 96 else 1, 1, 1), p)
        B, CI, HW = 3, 70, 50
        say("blocks, columns", outputs, "p", p)
        x, w = make_inputs(B, CI=CI, CO=outputs, G=1, HW=HW, seed=outputs)
        go = torch.randn(B, outputs, HW, generator=gen(3))
        out = oracle.norm_dist_forward(x, w, 1, p)
        ex, mx = oracle.norm_dist_backward_input(go, x, w, out, 1, p, with_abs_terms=True)
        ew, mw = oracle.norm_dist_backward_weight(go, x, w, out, 1, p, with_abs_terms=True)
        set_tile(0)
        gx, gw = torch.full((B, CI, HW), float("nan"), device=DEV), torch.zeros((outputs, CI), device=DEV)
        cpp.norm_dist_backward(*(t.to(DEV) for t in (go, x, w, out)), gx, gw, 1, p)
        torch.cuda.synchronize()
        assert_sum_close(gx.cpu(), ex, mx, p, 1e-5, 1e-6)
        assert_sum_close(gw.cpu(), ew, mw, p, 1e-5, 1e-6)
    finally:
        set_tile(-1)


# Exponents below 2: a term whose x equals its w is 0 whatever form the kernel takes.  Quantised inputs and weights meet in
# many elements; a zero row of weights meets the zeros of the padding and the rows past a ragged last tile.
@pytest.mark.parametrize("p", [1.25, 1.5, 1.9])
@pytest.mark.parametrize("outputs", [9, 33, 70, 150])
def test_conv_backward_below_two(outputs, p):
    import torch.nn.functional as F
    from gpu_common import DEV, cpp, say, set_tile
    B, C, H, W = 3, 10, 9, 11
    say("conv backward below 2", outputs, "p", p)
    img, w = torch.round(torch.rand(B, C, H, W, generator=gen(outputs)) * 8) / 8, torch.randn(outputs, C * 9, generator=gen(8))
    w = torch.round(w * 4) / 8
    w[outputs // 2] = 0.0
    cols = F.unfold(img, 3, 1, 1, 1).contiguous()
    go = torch.randn(B, outputs, cols.size(2), generator=gen(9))
    out = oracle.norm_dist_forward(cols, w, 1, p)
    ex, mx = oracle.norm_dist_backward_input(go, cols, w, out, 1, p, with_abs_terms=True)
    ew, mw = oracle.norm_dist_backward_weight(go, cols, w, out, 1, p, with_abs_terms=True)
    fold = lambda t: F.fold(t.double(), (H, W), 3, 1, 1, 1)
    g, x, xc, wd, o = (t.to(DEV) for t in (go, img, cols, w, out))
    try:
        set_tile(0)
        gi, gw = torch.full_like(x, float("nan")), torch.zeros_like(wd)
        cpp.norm_dist_conv_backward(g, x, wd, o, gi, gw, 1, p, 3, 1, 1, 1)
        gx, gc = torch.full_like(xc, float("nan")), torch.zeros_like(wd)
        cpp.norm_dist_backward(g, xc, wd, o, gx, gc, 1, p)
        torch.cuda.synchronize()
    finally:
        set_tile(-1)
    assert_sum_close(gi.cpu(), fold(ex), fold(mx), p, 1e-5, 1e-6)
    assert_sum_close(gx.cpu(), ex, mx, p, 1e-5, 1e-6)
    for got in (gw, gc):
        assert_sum_close(got.cpu(), ew, mw, p, 1e-5, 1e-6)


# ldist_set_tile_override(2): the separate kernels, whose grad_input is added up in the order that its own entry point keeps.
@pytest.mark.parametrize("shape", [(40, 1040, 130, 1, 1), (64, 2048, 96, 2, 1), (3, 520, 24, 1, 20)])
def test_forced_separate_kernels_keep_the_order_of_grad_input(shape):
    from gpu_common import DEV, cpp, gpu_norm_forward, say, set_tile
    B, CO, CI, G, HW = shape
    say("fixed order", shape)
    x, w = make_inputs(B, CO, CI, G, HW, seed=sum(shape))
    go = torch.randn(B, CO, HW, generator=gen(7)).to(DEV)
    out = gpu_norm_forward(x, w, G, 37.3).to(DEV)
    x, w = x.to(DEV), w.to(DEV)
    own, both, gw = torch.empty_like(x), torch.empty_like(x), torch.zeros_like(w)
    try:
        set_tile(2)
        cpp.norm_dist_backward_input(go, x, w, out, own, G, 37.3)
        cpp.norm_dist_backward(go, x, w, out, both, gw, G, 37.3)
        torch.cuda.synchronize()
    finally:
        set_tile(-1)
    assert torch.equal(own, both)


# The same split in the unfolded layout: few tiles, many outputs.
@pytest.mark.parametrize("p", [3.0, 37.3])
@pytest.mark.parametrize("shape", [(3, 520, 24, 1, 20), (2, 1030, 70, 2, 33), (1, 300, 9, 1, 2)])
def test_shared_grad_input_of_columns(shape, p):
    from gpu_common import DEV, cpp, say
    B, CO, CI, G, HW = shape
    say("split grad_input, columns", shape, "p", p)
    x, w = make_inputs(B, CO, CI, G, HW, seed=sum(shape))
    go = torch.randn(B, CO, HW, generator=gen(7))
    out = oracle.norm_dist_forward(x, w, G, p)
    ex, mx = oracle.norm_dist_backward_input(go, x, w, out, G, p, with_abs_terms=True)
    ew, mw = oracle.norm_dist_backward_weight(go, x, w, out, G, p, with_abs_terms=True)
    gx, gw = torch.full((B, CI, HW), float("nan"), device=DEV), torch.zeros((CO, CI // G), device=DEV)
    cpp.norm_dist_backward(*(t.to(DEV) for t in (go, x, w, out)), gx, gw, G, p)
    torch.cuda.synchronize()
    assert_sum_close(gx.cpu(), ex, mx, p, 1e-5, 1e-6)
    assert_sum_close(gw.cpu(), ew, mw, p, 1e-5, 1e-6)
