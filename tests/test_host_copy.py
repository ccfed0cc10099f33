"""Host logic of the copies to the host (pdp3_amd/csrc/host_copy.hpp), on a fake
HIP runtime of two devices (tests/native/fakehip): the copies through pinned
slots work whatever the calling thread's current device is, every failure of
what they need ends in a plain copy, and no exception leaves them."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_copy") / "host_copy_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-rdynamic", "-I", os.path.join(NATIVE, "fakehip"),
                    "-I", os.path.join(ROOT, "pdp3_amd", "csrc"), os.path.join(NATIVE, "host_copy_test.cpp"), "-o", exe,
                    "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("case", ["same_device", "other_device_current", "record_fails", "no_pinned_memory",
                                  "no_threads", "no_host_memory"])
def test_copy(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (case, r.returncode, r.stderr)
