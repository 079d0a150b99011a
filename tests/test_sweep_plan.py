"""The pipelined sweeps' schedule (ofx_sweep.h) on the CPU: every dependency is
where its slot points, received before its level, from an earlier range."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


def test_sweep_plan(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = tmp_path / "sweep_plan_check"
    subprocess.run(["g++", "-O2", "-std=c++17", str(HERE / "sweep_plan_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert out.startswith("ok "), out
