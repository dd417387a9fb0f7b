"""The LDS windows of the boundary tiles, for odd and even row pitches, checked
on the CPU by tests/edge_window_check.cpp built against the kernel's header:
every chunk is aligned and inside the array, and every neighbour a boundary
stencil reads is where the kernel looks for it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "nr-amssncku_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_edge_windows_hold_every_stencil_read(tmp_path):
    exe = str(tmp_path / "edge_window_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, os.path.join(HERE, "edge_window_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
