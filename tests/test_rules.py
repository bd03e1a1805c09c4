"""Single rules of the device (hvm-64_amd/csrc/hvm64_rules.h) built for the
host and run on one lane with a small heap (tests/rules_check.cpp).  CPU
only; the same functions run in the kernels."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hvm-64_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("rules") / "rules_check")
    subprocess.run([gxx, "-O2", "-w", "-std=c++17", "-I", CSRC, os.path.join(HERE, "rules_check.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("case", ["wide definition", "first error", "out of nodes first", "outside the heap",
                                  "arena remainders"])
def test_rule(rules, case):
    r = subprocess.run([rules, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
