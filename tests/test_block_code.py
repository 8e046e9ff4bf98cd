"""The 80-bit code of a block, on the host: tests/block_code.cpp walks every arrangement of magnitudes of shells up to 13 in both
parities (that each has a code, and what it decodes to), every class boundary and 400 000 ranks through the decoder."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "llvq_amd", "csrc")


def test_every_point_has_a_code_that_gives_it_back(tmp_path, boundary_indices):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = tmp_path / "block_code"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), os.path.join(HERE, "block_code.cpp"), os.path.join(CSRC, "codebook.cpp")], check=True)
    run = subprocess.run([str(exe), *map(str, boundary_indices)], capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stdout + run.stderr
