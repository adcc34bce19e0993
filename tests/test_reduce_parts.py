"""The scratch of the simulation_state reduction holds every record that the
reduction writes, whatever the grid (hippolbm_amd/csrc/reduce_parts.hpp), and the
domain and batch paths both allocate that scratch and nothing of their own
making.  Compiled for the host with g++."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "hippolbm_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_records_fit_the_scratch(tmp_path):
    exe = tmp_path / "reduce_parts_check"
    src = os.path.join(HERE, "csrc", "reduce_parts_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", str(exe), src], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "failures 0" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("source,scratch", [("api.hip", "red_part"), ("batch.hip", "d_part")])
def test_every_caller_allocates_the_whole_scratch(source, scratch):
    text = open(os.path.join(CSRC, source)).read()
    sizes = re.findall(r"hipMalloc\(\(void\*\*\)&\w+->" + scratch + r", ([^)]*\)?)\)", text)
    assert sizes == ["RED_SCRATCH_BYTES"]
