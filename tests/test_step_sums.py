"""The batch-1 product's sums over a tile's steps stay in their place in LDS, and its work is shared out over all wavefronts:
tests/step_sums.cpp walks every row length, round and team."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "llvq_amd", "csrc")


def test_sums_are_read_where_they_were_left(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = tmp_path / "step_sums"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), os.path.join(HERE, "step_sums.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
