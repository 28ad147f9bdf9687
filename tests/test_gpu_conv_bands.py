"""The one-pass p-norm conv backward from few images, which it cuts into bands of output rows (csrc/norm_conv_backward.hip):
bands whose halo is less than a tile, exactly one and several, strides, paddings and dilations that leave image rows between or
beyond the windows.  Against the oracle, as the other geometries of this kernel."""
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # B, C, H, W, CO, G, stride, padding, dilation
    (1, 3, 32, 32, 32, 1, 1, 1, 1),      # halo of two rows of 32: one tile; three channels: the two halves of a workgroup
    (2, 8, 33, 17, 9, 1, 1, 1, 1),       # 561 positions, bands that divide nothing, two column tiles
    (1, 4, 41, 70, 6, 2, 1, 1, 1),       # a halo of 140 positions: three tiles, the last a partial one
    (2, 7, 50, 23, 5, 1, 1, 3, 3),       # dilation 3: six rows of halo, and padding that the first bands lie in
    (3, 5, 37, 29, 12, 1, 2, 1, 1),      # stride 2, odd sizes: one row of halo
    (2, 4, 40, 31, 7, 1, 2, 0, 1),       # stride 2 without padding: the last image row has no window
    (1, 4, 61, 40, 4, 1, 3, 0, 1),       # stride 3: no halo
    (1, 2, 45, 35, 3, 1, 4, 0, 1),       # stride 4: image rows between the windows belong to none
    (1, 14, 20, 64, 70, 1, 1, 1, 1),     # outputs in two blocks, an output row to a tile
]


@pytest.fixture(autouse=True)
def _reset():
    from gpu_common import set_tile
    yield
    set_tile(-1)


@pytest.mark.parametrize("p", [8.0, 2.0, 5.5, 100.0])
@pytest.mark.parametrize("case", CASES)
def test_bands(case, p):
    from test_gpu_parity import test_norm_conv_backward_both_gradients_in_one_pass_from_the_image as from_the_image
    from_the_image(case, p)
