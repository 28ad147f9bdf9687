"""The image kernels with the channels of a tile shared by several groups of lanes (launches that would leave CUs idle):
values, indices and bounds against the oracle on torch's unfolded columns, bit for bit."""
import pytest
import torch
import torch.nn.functional as F

import oracle
from helpers import gen

pytestmark = pytest.mark.gpu

CASES = [  # B, C, H, W, CO, G, stride, padding
    (3, 32, 14, 14, 64, 1, 1, 1),     # eight stages over up to eight groups
    (2, 36, 14, 14, 64, 1, 1, 1),     # nine stages: groups with a stage less, or with none
    (2, 64, 28, 28, 64, 1, 2, 1),
    (2, 22, 16, 16, 24, 1, 1, 1),     # a last stage of two channels
    (1, 128, 16, 16, 96, 4, 1, 1),
    (2, 40, 9, 11, 10, 1, 1, 2),      # ragged segments, an output count that is no multiple of four
]


@pytest.mark.parametrize("groups", [0, 1, 2, 3, 5, 8])
@pytest.mark.parametrize("staging", [0, 2])
@pytest.mark.parametrize("case", CASES)
def test_groups_of_channels_bit_exact(case, staging, groups):
    from gpu_common import DEV, cpp, pkg, say
    B, C, H, W, CO, G, s_, p_ = case
    say("conv groups", case, "staging", staging, "groups", groups)
    lib = pkg._lib.lib()
    assert lib.ldist_set_conv_groups_override(groups) == 0 and lib.ldist_set_conv_staging_override(staging) == 0
    try:
        if not cpp.inf_dist_conv_forward_supported(C, H, W, CO, G, 3, s_, p_, 1):
            pytest.skip("left to the column path by the library")
        img = (torch.randn(B, C, H, W, generator=gen(71)) * 4).round() / 4      # ties: the lowest index is what is checked
        w = (torch.randn(CO, C // G * 9, generator=gen(72)) * 3).round() / 4
        img[0, -1, 2, 2], img[0, 0, 3, 1] = float("nan"), float("inf")
        eo, ep = oracle.inf_dist_forward(F.unfold(img, 3, 1, p_, s_).contiguous(), w, G, literal=True)
        out = torch.full(eo.shape, float("nan"), device=DEV)
        only = torch.full(eo.shape, float("nan"), device=DEV)
        pos = torch.full(eo.shape, -7, device=DEV, dtype=torch.int32)
        cpp.inf_dist_conv_forward(img.to(DEV), w.to(DEV), out, pos, G, 3, s_, p_, 1)
        cpp.inf_dist_conv_forward_values(img.to(DEV), w.to(DEV), only, G, 3, s_, p_, 1)
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), eo) and torch.equal(only.cpu(), eo)
        assert torch.equal(pos.cpu(), ep)
        if staging or not cpp.inf_dist_bound_conv_forward_supported(C, H, W, CO, G, 3, s_, p_, 1):
            return
        centre, radius = torch.randn(B, C, H, W, generator=gen(73)), torch.rand(B, C, H, W, generator=gen(74)) * 0.3
        lo, up = centre - radius, centre + radius
        for irregular in (False, True):
            if irregular:
                lo[0, C // 2, 1, 1], up[0, -1, 4, 4], lo[-1, 0, 2, 2] = float("nan"), float("inf"), 9.0
            el, eu = oracle.inf_dist_bound_forward(F.unfold(lo, 3, 1, p_, s_).contiguous(), F.unfold(up, 3, 1, p_, s_).contiguous(), w, G)
            ol, ou = torch.full(el.shape, float("nan"), device=DEV), torch.full(el.shape, float("nan"), device=DEV)
            cpp.inf_dist_bound_conv_forward(lo.to(DEV), up.to(DEV), w.to(DEV), ol, ou, G, 3, s_, p_, 1)
            torch.cuda.synchronize()
            assert torch.equal(torch.nan_to_num(ol.cpu(), nan=-7.0), torch.nan_to_num(el, nan=-7.0))
            assert torch.equal(torch.nan_to_num(ou.cpu(), nan=-7.0), torch.nan_to_num(eu, nan=-7.0))
    finally:
        lib.ldist_set_conv_groups_override(0)
        lib.ldist_set_conv_staging_override(0)
