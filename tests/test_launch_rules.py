"""Combinations that the kernels' launchers refuse before they reach a
device. Only refused ones are called here: a launch that is let through
would run on pointers that are no device's."""
import ctypes
import os
import subprocess

import pytest

import rrhip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXTEND, SHADOW, ROUND = 0, 1, 2
REFUSED = 1  # hipErrorInvalidValue


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    lib = tmp_path_factory.mktemp("native") / "launch_check.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{ROOT}/render.rs_amd/csrc", f"-I{ROOT}/include",
                    f"{ROOT}/tests/native/launch_check.cpp", "-o", str(lib), rrhip.LIB_PATH,
                    f"-Wl,-rpath,{os.path.dirname(rrhip.LIB_PATH)}"], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("transparent,profiled,queue,work", [
    (1, 0, 1, ROUND), (0, 1, 1, ROUND), (1, 1, 1, ROUND),  # closest hits and shadow records in one launch: opaque only
    (0, 0, 0, ROUND), (0, 0, 0, EXTEND), (1, 0, 0, EXTEND), (0, 1, 0, EXTEND),  # closest hits of no queue
])
def test_trace_launches_that_have_no_kernel_are_refused(check, transparent, profiled, queue, work):
    assert check.check_trace(transparent, profiled, queue, work) == REFUSED
