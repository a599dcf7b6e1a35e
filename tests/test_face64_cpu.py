"""The FP64 production forms of the face states (cada3, WENO5) and of the roots
and reciprocals against the general forms of the same device header, compiled
for the CPU: both sides of the limiter's switch, its blend, flat stretches,
sizes beyond the range of the weights' products, and values that are not
finite."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "face64_cpu")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_fp64_face_forms_match_the_general_forms(tmp_path):
    exe = str(tmp_path / "face64_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-mfma", "-ffp-contract=off", "-I", ".", "face64_check.cpp", "-o", exe],
                   cwd=HERE, check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count("worst / bound") == 5
