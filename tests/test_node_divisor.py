"""Node indices to rows and planes by multiply-high (NodeDivisors,
hippolbm_amd/csrc/d3q19.hpp), checked against the division.  Compiled for the
host with g++."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_multiply_high_is_the_division(tmp_path):
    exe = tmp_path / "node_divisor_check"
    src = os.path.join(HERE, "csrc", "node_divisor_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", str(exe), src], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("failures 0 ")
