"""The search of a cumulative table by a group of lanes (csrc/group_probe.hpp,
compiled with the system g++): with no entry past the target it ends at the last
entry, for every group size and length.  The mixed STS-CP draw searches the leaf
masses of its first mode with it; a component without mass has no such entry."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rdist_tensor_amd", "csrc")


def test_ends_inside_the_table(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = str(tmp_path / "probe")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "group_probe_host.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    assert out.startswith("ok "), out
