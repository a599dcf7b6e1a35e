"""The FP32 cada3 face states without branches against the limiter's
definition, bit for bit, compiled for the CPU from the device header: both
sides of the switch, its edge, flat stretches and values that are not
finite."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "face64_cpu")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_fp32_cada3_face_equals_the_definition(tmp_path):
    exe = str(tmp_path / "face32_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", ".", "face32_check.cpp", "-o", exe],
                   cwd=HERE, check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "1600000 faces equal" in r.stdout
