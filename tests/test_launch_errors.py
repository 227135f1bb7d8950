"""A refused launch of a call's first kernel ends the call with its error (CPU:
the built library with stand-ins for the HIP launch calls,
tests/cpp/launch_errors.cpp)."""

import os
import shutil
import subprocess

import pytest

import plainmp_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_first_kernel_of_two(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe, lib = str(tmp_path / "launch_errors"), os.path.dirname(plainmp_amd.LIBRARY_PATH)
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-rdynamic",
                    os.path.join(ROOT, "tests", "cpp", "launch_errors.cpp"), plainmp_amd.LIBRARY_PATH,
                    "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{lib}", "-Wl,-rpath,/opt/rocm/lib", "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True, timeout=100).stdout.split("\n")
    rows = [line.split() for line in out if line]
    assert [r[0] for r in rows] == ["edges", "vjp"] * 2
    assert all(int(r[1]) == 9 for r in rows), out  # hipErrorInvalidConfiguration
    assert int(rows[-1][3]) == 0  # and nothing is launched behind it
