"""Builds a test program with the engine's host code and the one-lane device
in host memory (fake_device.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "hvm-64_amd", "csrc")
HIP = "/opt/rocm/include"


def build(program, out):
    """The executable of tests/<program>.cpp in directory `out`."""
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists(os.path.join(HIP, "hip", "hip_runtime.h")):
        pytest.skip("g++ or the HIP headers not available")
    flags = ["-O1", "-w", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", HIP, "-I", CSRC, "-I",
             os.path.join(ROOT, "include"), "-I", HERE]
    src = [os.path.join(CSRC, f"hvm64_{x}.cpp") for x in ("api", "host", "defcomp")]
    src += [os.path.join(HERE, f + ".cpp") for f in ("fake_device", program)]
    exe = os.path.join(str(out), program)
    subprocess.run([gxx] + flags + src + ["-o", exe], check=True)
    return exe
