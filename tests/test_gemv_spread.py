"""The batch-1 product of rows past sixteen steps: tests/gemv_spread.cpp walks every number of steps."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "llvq_amd", "csrc")


def test_every_step_is_computed_and_every_tile_finished_once(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = tmp_path / "gemv_spread"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), os.path.join(HERE, "gemv_spread.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
