"""Every array index the boundary stencils read in global memory, the upwind
stencil's clamped samples among them, lies inside the array:
tests/edge_reads_check.cpp, built against the kernel's header."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "nr-amssncku_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_every_boundary_read_is_inside_the_array(tmp_path):
    exe = str(tmp_path / "edge_reads_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, os.path.join(HERE, "edge_reads_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
