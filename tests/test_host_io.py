"""Host buffers to the device and back (csrc/host_io.hip), compiled for the CPU against a stand-in for the HIP runtime
(tests/host_io): a queue that a thread works off and that a check can hold.  No GPU involved."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_io") / "host_io_check")
    src = os.path.join(HERE, "..", "oxibonsai_amd", "csrc", "host_io.hip")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-I", os.path.join(HERE, "host_io"), "-x", "c++", src,
                           os.path.join(HERE, "host_io", "host_io_check.cpp"), "-lpthread", "-o", exe])
    return exe


@pytest.mark.parametrize("check", ["round_trip", "error_exit", "first_call", "pool_of_results", "few_cpus"])
def test_host_io(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
