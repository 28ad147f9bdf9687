"""Scratch memory of instantiations that stand beside others of the same kernel, as the compiler reports it for the library's own
flags (no GPU needed): what a rarer form needs must not cost the usual one its registers."""
import re
import shutil

import pytest

from test_register_use import scratch_of

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")


def test_conv_backward_of_whole_images_beside_bands(tmp_path):
    """Four waves per SIMD, multiply-only exponents: 60 bytes without bands of images, 72 in the one form that has them."""
    sizes = scratch_of("norm_conv_backward.hip", tmp_path)
    whole = [size for name, size in sizes.items() if re.search(r"norm_conv_backward_kernelILb1ELi[1-9]ELb0ELi4E", name)]
    bands = [size for name, size in sizes.items() if re.search(r"norm_conv_backward_kernelILb1ELi(?:16|17|18|19|23)ELb0ELi4E", name)]
    assert len(whole) == 8 and max(whole) <= 60
    assert len(bands) == 10 and max(bands) <= 72


def test_lists_of_outermost_values(tmp_path):
    """extremes_select_kernel<NV, ENDS, SPREAD> of up to 32 values per lane: no scratch memory in any form."""
    sizes = {name: size for name, size in scratch_of("extremes_forward.hip", tmp_path).items()
             if re.search(r"extremes_select_kernelILi(?:16|24|32)E", name)}
    assert len(sizes) == 12 and max(sizes.values()) == 0


def test_scans_and_samples_of_lists(tmp_path):
    """What the first scans of boxes, and the longest rows of the sample and list kernels, spill outside of their loops; no more, and
    nothing in any other form."""
    allowed = {"scan_kernelILi3ELb0E": 40, "scan_kernelILi2ELb0E": 16, "sample_kernelILi40ELi3E": 68, "sample_kernelILi40ELi1E": 8,
               "select_kernelILi40ELi2E": 76, "select_kernelILi40ELi3E": 76}
    sizes = {name: size for name, size in scratch_of("extremes_forward.hip", tmp_path).items() if "extremes_" in name}
    assert sum(any(form in name for name in sizes) for form in allowed) == len(allowed)
    for name, size in sizes.items():
        assert size <= max((most for form, most in allowed.items() if form in name), default=0), name
