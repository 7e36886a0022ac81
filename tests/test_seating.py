"""The decision whether a resident launch takes place (csrc/seating.h) on the
CPU: all of its workgroups decide alike (tests/native/seating.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "diploma_research_amd", "csrc")
CXX = os.environ.get("CXX", "g++")


@pytest.mark.skipif(shutil.which(CXX) is None, reason=f"{CXX} not found")
def test_all_workgroups_decide_alike(tmp_path):
    exe = str(tmp_path / "seating")
    subprocess.run([CXX, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, os.path.join(HERE, "native", "seating.cpp"),
                    "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "done, 0 failures" in r.stdout, r.stdout[-4000:]
