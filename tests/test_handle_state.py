"""A handle after launches the host lost: its root cell and its redex ring
(tests/handle_check.cpp).  CPU only: the engine's host code on a one-lane
device in host memory."""
import subprocess

import fake_device


def test_root_cell_after_a_lost_launch(tmp_path):
    r = subprocess.run([fake_device.build("handle_check", tmp_path)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
