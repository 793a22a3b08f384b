"""The arithmetic that decides which texel boxes get an LDS window in the
texture backward (mlx-swift-diffrast_amd/csrc/window_box.h, the header the
kernels include), in a host build over every side a box can have
(tests/texture_windows.cpp; a signed overflow ends it).  CPU only."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "mlx-swift-diffrast_amd", "csrc")


def test_window_arithmetic(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs g++")
    exe = tmp_path / "texture_windows"
    subprocess.run([cxx, "-O1", "-std=c++17", "-Wall", "-ftrapv", "-I", CSRC, "-o", str(exe),
                    os.path.join(HERE, "texture_windows.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    boxes, windows = map(int, re.search(r"(\d+) boxes, (\d+) windows", r.stdout).groups())
    assert boxes > 1_000_000 and windows > 1000
