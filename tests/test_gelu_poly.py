"""The GELU pass's polynomial (csrc/gelu_poly.h) against erfc in 64 bits, on the CPU:
the errors that its comment states."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gelu_poly(tmp_path):
    exe = str(tmp_path / "gelu_poly_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unknown-pragmas",
                    "-I", os.path.join(ROOT, "anima-on-android_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "gelu_poly_check.cpp"), "-o", exe],
                   check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True)
    weighted, to2, to6, to14 = (float(x) for x in run.stdout.split())
    assert weighted <= 4.2e-9
    assert to2 <= 1e-7 and to6 <= 4e-6 and to14 <= 6e-5
