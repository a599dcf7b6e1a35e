"""The FP64 production form of the cada3 face states beside steep jumps and
infinite neighbours, against the general form of the same device header,
compiled for the CPU: each side's error is bounded by its own cell's size."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "face64_cpu")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_fp64_cada3_keeps_the_small_cell_beside_a_jump(tmp_path):
    exe = str(tmp_path / "cada3_jump_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", ".", "cada3_jump_check.cpp", "-o",
                    exe], cwd=HERE, check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count("worst / bound") == 3
