"""The p-norm forward that trains on tiles of 16 x 16 with eight k-groups and two rows and columns per lane (csrc/norm_forward.hip:
few rows and outputs of long reductions): tails of rows, outputs, k and vectors, groups, and every kind of exponent."""
import pytest
import torch

import oracle
from helpers import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(33, 300, 300, 1), (17, 63, 257, 1), (64, 500, 516, 1), (1, 17, 2053, 1), (100, 64, 1030, 2),
                                   (40, 35, 31, 1), (128, 512, 256, 1)])   # B, CO, CI, G
def test_small_square_tiles(shape):
    from gpu_common import gpu_norm_forward, say
    B, CO, CI, G = shape
    say("eight groups", shape)
    x, w = make_inputs(B, CO, CI, G, 1, seed=sum(shape))
    x[0, 0], w[0, 0] = 3.0, -2.0
    for p, scale in ((8.0, 1.0), (2.0, 1.0), (3.0, 1e-7), (4.0, 1e9), (37.3, 1.0), (1.5, 1.0), (500.0, 1e-3)):
        xs, ws = (x * scale).contiguous(), (w * scale).contiguous()
        got, want = gpu_norm_forward(xs, ws, G, p), oracle.norm_dist_forward(xs, ws, G, p)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-6 * min(1.0, scale))
