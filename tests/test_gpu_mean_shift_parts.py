"""Channel mean shift where several workgroups share a channel."""
import pytest
import torch

from helpers import gen

pytestmark = pytest.mark.gpu


# below and at the first shared length (12288 vectors of four values, or of one where L is odd), ragged last parts,
# the most parts a channel can have, the most channels that are shared and one more
@pytest.mark.parametrize("shape", [(1, 3, 49148), (1, 3, 49152), (2, 3, 26004), (2, 5, 6143), (2, 5, 6145), (7, 3, 4999),
                                   (128, 32, 1024), (77, 32, 784), (1, 1, 1 << 20), (1, 1, (1 << 18) + 1), (49, 64, 1024),
                                   (49, 65, 1024), (13, 128, 961), (13, 129, 961)])
def test_shared_channels(shape):
    from gpu_common import DEV, cpp, say
    say("mean_shift parts", shape)
    B, C, L = shape
    x = torch.randn(B, C, L, generator=gen(31)) + torch.linspace(-3, 3, C).view(1, C, 1)
    running = torch.linspace(-1, 1, C)
    mean = x.double().mean(dim=(0, 2))
    xd, rm, mean_out = x.to(DEV), running.to(DEV), torch.empty(C, device=DEV)
    y = torch.full_like(xd, float("nan"))
    cpp.mean_shift(xd, y, mean_out, rm, 0.1)
    # A value goes through one addition per 1024 vectors in its lane, 2 in the vector, 6 in the wave and 16 over the waves; each
    # rounds by 2^-24 of a partial sum, which is at most the sum of magnitudes.
    n = B * L // 1024 + 25
    off = n * 2.0 ** -24 * x.double().abs().mean(dim=(0, 2)) + 2.0 ** -23 * mean.abs()
    assert ((mean_out.cpu().double() - mean).abs() <= off).all()
    shifted = x.double() - mean.view(1, C, 1)
    assert ((y.cpu().double() - shifted).abs() <= off.view(1, C, 1) + 2.0 ** -23 * shifted.abs()).all()
    assert torch.equal(y, xd - mean_out.view(1, C, 1))
    moved = 0.9 * running.double() + 0.1 * mean
    assert ((rm.cpu().double() - moved).abs() <= 0.1 * off + 2.0 ** -22 * (running.double().abs() + mean.abs())).all()
    again = torch.empty_like(xd)
    cpp.mean_shift(xd, again)
    assert torch.equal(again, y)
