"""Launches of thin segments over very long grids stay within the runtime's 2^32
work-items, with every launch shape that a caller may set: run against a HIP
runtime in host memory that refuses more (fake_hip.cpp)."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BODY = """
import sys
sys.path.insert(0, %r)
import numpy as np
import le2d_amd
ny = (1 << 32) // 64 + 100000  # one row a segment on 64 lanes is past the limit
with le2d_amd.Task(3, ny, 0.2, (1.0, 1.0), (2.0, 1.0, 1.0), dtype=np.float32) as t:
    t.set_tiles(y_seg=1, y_block=64)
    t.time_sweeps(1)
    t.set_step_pairs(1)
    t.set_step_pair_window(64)
    t.time_pairs(1)
    t.time_steps(1)
print("done")
"""


def test_one_row_segments(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    so = str(tmp_path / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "fake_hip.cpp")], check=True)
    out = subprocess.run([sys.executable, "-c", BODY % ROOT], env=dict(os.environ, LD_PRELOAD=so),
                         capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "done" in out.stdout, out.stderr[-2000:]
