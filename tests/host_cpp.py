"""Builds a host program of tests/cpp against the library and its internal headers."""
import os
import subprocess

import pytest

from conftest import ROOT

LIBDIR = os.path.join(ROOT, "ndarray-conv_amd", "lib")
BUILD = os.path.join(ROOT, "ndarray-conv_amd", "_build")


def program(name):
    if not os.path.exists(os.path.join(LIBDIR, "libndconv.so")):
        pytest.skip("libndconv.so not built")
    os.makedirs(BUILD, exist_ok=True)
    exe = os.path.join(BUILD, name)
    cmd = ["/opt/rocm/bin/amdclang++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include",
           f"-I{ROOT}/ndarray-conv_amd/csrc", "-I/opt/rocm/include", os.path.join(ROOT, "tests", "cpp", name + ".cpp"),
           "-o", exe, f"-L{LIBDIR}", "-lndconv", "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{LIBDIR}"]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    return exe
