"""The two-step kernel's split of a grid into segments (hippolbm_amd/csrc/
pair_grid.hpp): the search over distinct segment lengths finds what the search
over every segment count finds, and stays short on long thin grids.  Compiled for
the host with g++."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_distinct_segment_lengths_find_the_same_split(tmp_path):
    exe = tmp_path / "pair_grid_check"
    src = os.path.join(HERE, "csrc", "pair_grid_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", str(exe), src], check=True)
    # the check itself takes under a second; a thousand full searches of 2^29 planes would take an hour
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("failures 0 ")
