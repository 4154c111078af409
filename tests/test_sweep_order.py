"""The triangular sweeps' count of solved superblocks (updes_amd/csrc/sweep_order.h),
driven on the CPU by tests/sweep_order_check.cpp with chunks that publish,
store and count in random orders: it never stands for a superblock whose
solution is not all in memory, and it reaches the last one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_solved_superblocks_are_counted_in_order(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "sweep_order_check")
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", os.path.join(ROOT, "tests", "sweep_order_check.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.stdout + res.stderr
