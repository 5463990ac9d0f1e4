"""Inline assembly that writes m0 (the LDS address of a load straight to LDS)
says so, or the compiler may keep a value of its own there."""
import glob
import os
import re

from conftest import ROOT


def test_m0_is_clobbered_where_it_is_written():
    written = 0
    for path in glob.glob(os.path.join(ROOT, "stratum_amd", "csrc", "*.h*")):
        with open(path) as f:
            text = f.read()
        for stmt in re.findall(r'asm volatile\((.*?)\);', text, re.S):
            if re.search(r"s_\w+ m0,", stmt):
                written += 1
                assert '"m0"' in stmt.rsplit(":", 1)[1], f"{os.path.basename(path)}: {stmt}"
    assert written
