"""Scratch memory of kernels whose speed depends on keeping their values in registers, as the compiler reports it for the
library's own flags (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from test_shortk_parked_loads import CSRC, library_flags

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")


def scratch_of(source, tmp_path):
    """Mangled kernel name -> bytes of scratch per lane."""
    cmd = ["hipcc"] + library_flags() + ["-Rpass-analysis=kernel-resource-usage", "-c", "--cuda-device-only",
                                         os.path.join(CSRC, source), "-o", str(tmp_path / "out.o")]
    text = subprocess.run(cmd, check=True, capture_output=True, text=True).stderr
    names = re.findall(r"Function Name: (\S+)", text)
    sizes = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", text)
    assert names and len(names) == len(sizes)
    return dict(zip(names, map(int, sizes)))


def test_one_pass_conv_backward_at_four_waves(tmp_path):
    """norm_conv_backward_kernel<IMG, IE, BLOCKS, 4, ...>: groups staged whole, of up to 39 outputs."""
    four = {name: size for name, size in scratch_of("norm_conv_backward.hip", tmp_path).items()
            if re.search(r"norm_conv_backward_kernelILb[01]ELi\dELb[01]ELi4E", name)}
    columns = [size for name, size in four.items() if "kernelILb0E" in name]
    image = [size for name, size in four.items() if "kernelILb1E" in name]
    assert len(columns) == 5 and max(columns) == 0
    assert len(image) == 10 and max(image) <= 72
