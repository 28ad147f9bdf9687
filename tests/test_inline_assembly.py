"""Inline assembly of the kernels (csrc/*.hip, *.hpp): the compiler adds wait states between instructions it knows, not inside
an assembly string.  On gfx9 targets a load to LDS (buffer_load ... lds) reads its LDS address from M0 and needs one wait
state behind a scalar write of M0."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "l_inf-dist-net_amd", "csrc")
STATEMENT = re.compile(r"\basm\s+volatile\s*\((.*?)\)\s*;", re.S)


def unguarded_m0_writes(source):
    """Assembly statements that write M0 without a wait state behind the write, or without telling the compiler."""
    bad = []
    for body in STATEMENT.findall(source):
        text = "\n".join(re.findall(r'"((?:[^"\\]|\\.)*)"', body))
        code = [line.strip() for line in re.split(r"\\n|\n|;", text.replace("\\t", " ")) if line.strip()]
        for at, line in enumerate(code):
            if re.match(r"s_\w+\s+m0\b", line):
                waits = at + 1 < len(code) and code[at + 1].startswith("s_nop")
                if not waits or '"m0"' not in body:
                    bad.append(body)
    return bad


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))), ids=os.path.basename)
def test_a_write_of_m0_is_followed_by_a_wait_state(path):
    assert unguarded_m0_writes(open(path).read()) == []


def test_the_check_finds_what_it_looks_for():
    good = r'asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(a) : "memory", "m0");'
    assert unguarded_m0_writes(good) == []
    assert len(unguarded_m0_writes(good.replace(r"s_nop 0\n\t", ""))) == 1
    assert len(unguarded_m0_writes(good.replace(', "m0"', ""))) == 1
