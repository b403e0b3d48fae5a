"""The staged host copies (csrc/ctx.hip) on a host-only stand-in for the HIP
runtime, where copies stay in flight until something waits for them and can be
made to fail (no GPU)."""
import os
import shutil
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
MOCK = os.path.join(TESTS, "mock_hip")
CTX = os.path.join(os.path.dirname(TESTS), "powerspectra.jl_amd", "csrc", "ctx.hip")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path_factory.mktemp("mock") / "host_copy")
    subprocess.run([gxx, "-std=c++17", "-O1", "-pthread", "-I", MOCK, "-x", "c++", CTX,
                    os.path.join(MOCK, "host_copy.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("case", ["round_trips", "nothing_in_flight_after_an_error",
                                  "nothing_in_flight_when_a_buffer_is_given_back",
                                  "pool_without_memory"])
def test_host_copies(program, case):
    assert subprocess.run([program, case], timeout=120).returncode == 0
