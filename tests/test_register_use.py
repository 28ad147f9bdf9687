"""Scratch memory of kernels whose speed depends on keeping their values in registers, as the compiler reports it for the
library's own flags (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from test_shortk_parked_loads import CSRC, library_flags

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")


def reported(source, tmp_path, what):
    """Mangled kernel name -> a number that the compiler reports."""
    cmd = ["hipcc"] + library_flags() + ["-Rpass-analysis=kernel-resource-usage", "-c", "--cuda-device-only",
                                         os.path.join(CSRC, source), "-o", str(tmp_path / "out.o")]
    text = subprocess.run(cmd, check=True, capture_output=True, text=True).stderr
    names = re.findall(r"Function Name: (\S+)", text)
    sizes = re.findall(re.escape(what) + r": (\d+)", text)
    assert names and len(names) == len(sizes)
    return dict(zip(names, map(int, sizes)))


def scratch_of(source, tmp_path):
    """Mangled kernel name -> bytes of scratch per lane."""
    return reported(source, tmp_path, "ScratchSize [bytes/lane]")


def test_one_pass_conv_backward_at_four_waves(tmp_path):
    """norm_conv_backward_kernel<IMG, IE, BLOCKS, 4, ...>: groups staged whole, of up to 39 outputs."""
    four = {name: size for name, size in scratch_of("norm_conv_backward.hip", tmp_path).items()
            if re.search(r"norm_conv_backward_kernelILb[01]ELi\dELb[01]ELi4E", name)}
    columns = [size for name, size in four.items() if "kernelILb0E" in name]
    image = [size for name, size in four.items() if "kernelILb1E" in name]
    assert len(columns) == 5 and max(columns) == 0
    assert len(image) == 10 and max(image) <= 72


def test_image_forward_without_pos_at_three_waves(tmp_path):
    """inf_conv_forward_kernel<1, RESIDENT, no POS, not GROUPED>: three waves per SIMD share its 512 registers."""
    waves = [n for name, n in reported("inf_conv_forward.hip", tmp_path, "Occupancy [waves/SIMD]").items()
             if "inf_conv_forward_kernelILi1ELb1ELb0ELb0E" in name]
    assert waves == [3]
