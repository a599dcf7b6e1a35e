"""Supersonic faces of the FP64 production HLL flux, compiled for the CPU from
the device header: an infinite state on the side the flow goes to is not read."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "face64_cpu")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_supersonic_hll_face_takes_one_side(tmp_path):
    exe = str(tmp_path / "hll_sides_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", ".", "hll_sides_check.cpp", "-o",
                    exe], cwd=HERE, check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "32000 faces" in r.stdout
