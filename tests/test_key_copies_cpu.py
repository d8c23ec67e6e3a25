"""The key-order copies of a lookup where an allocation fails (CPU: the host
logic of csrc/key_copies.hpp, compiled with the system g++ against buffers whose
allocations fail on request).  A buffer that was allocated and never written must
not be taken for filled by the next call: kernels index by its contents."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rdist_tensor_amd", "csrc")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = str(tmp_path_factory.mktemp("copies") / "copies")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "key_copies_host.cpp"), "-o", exe],
                   check=True)
    return lambda *calls: subprocess.run([exe, *calls], capture_output=True, text=True, check=True).stdout.split("\n")[:-1]


@pytest.mark.parametrize("calls,states", [
    (("0", "0"), ["1 r1 v1", "1 r1 v1"]),
    (("2", "0"), ["0 -0 -0", "1 r1 v1"]),                 # the values' allocation fails, then the call is repeated
    (("1", "2", "0"), ["0 -0 -0", "0 -0 -0", "1 r1 v1"]),
    # values of another type with the rows there already: the rows stay
    (("0", "v1", "v0"), ["1 r1 v1", "0 r1 -0", "1 r1 v1"]),
])
def test_failed_allocations(replay, calls, states):
    assert replay(*calls) == states
