"""The balanced flash grids' cut of the key tiles (csrc/flash_deal.h), checked on
the CPU over every tail of query tiles and key range: tests/native/flash_deal_check.cpp
compiles the header the kernels and their launcher share."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pieces_cover_every_key_tile_once(tmp_path):
    exe = str(tmp_path / "flash_deal_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "anima-on-android_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "flash_deal_check.cpp"), "-o", exe],
                   check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout + run.stderr
