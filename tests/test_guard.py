"""The order of team and cluster launches between streams (csrc/ring_guard.hpp) over a made-up runtime: which launches wait
for which, and that a single-stream program records no event.  Compiled with the host compiler and run here."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launch_order_between_streams(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "guard_harness")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", f"-I{ROOT}/rnn_train_ring_attractor_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "guard_harness.cpp"), "-o", exe], check=True, timeout=120)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and "guard ok" in out.stdout, out.stdout
