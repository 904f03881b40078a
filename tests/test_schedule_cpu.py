"""How runs are cut into launches and tiles dealt to workgroups
(csrc/schedule.h), every case of a range in a host program: each item dealt
once, one per workgroup in a launch of one round, launches that add up, stay
inside a staging block and come in an even number."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_schedule(tmp_path):
    exe = str(tmp_path / "schedule_check")
    csrc = os.path.join(HERE, "..", "meep-torch_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", csrc, os.path.join(HERE, "schedule_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
