"""The allocator of a serving slot (serve_take, hvm-64_amd/csrc/hvm64_rules.h)
built for the host and driven by threads (tests/serve_stress.cpp): blocks
never overlap, a block is refused only when no sub-arena has room for it, and
no node is lost.  CPU only; the same function runs in the kernels."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hvm-64_amd", "csrc")


@pytest.fixture(scope="module")
def stress(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("serve") / "serve_stress")
    subprocess.run([gxx, "-O2", "-w", "-std=c++17", "-pthread", "-I", CSRC, os.path.join(HERE, "serve_stress.cpp"),
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("threads,rounds,most", [(1, 400, 6), (1, 400, 1024), (1, 200, 1100), (2, 400, 300),
                                                 (8, 300, 6), (8, 300, 300), (8, 200, 2000), (16, 100, 64)])
def test_blocks_never_overlap_and_none_is_lost(stress, threads, rounds, most):
    r = subprocess.run([stress, str(threads), str(rounds), str(most), "20"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert int(r.stdout.split()[1]) >= rounds * 8
