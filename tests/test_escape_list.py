"""A tile's list of escapes on the host: tests/escape_list.cpp checks its number of places against the share of escapes that draws
show, for every row length, and the order in which a tile's codes are walked where the places were too few."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "llvq_amd", "csrc")


def test_places_and_walk(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = tmp_path / "escape_list"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), os.path.join(HERE, "escape_list.cpp"), os.path.join(CSRC, "codebook.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stdout + run.stderr
