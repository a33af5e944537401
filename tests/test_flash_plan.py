"""The launch shape of a flash attention (csrc/flash_plan.h), asked for on the CPU
through tests/native/flash_plan_shape.cpp: the shapes that were measured fastest
where the cost models of two of them come close, and the shape that each case of
the GPU tests of one shape is there for."""
import os
import shutil
import subprocess

import pytest

import test_gpu_balanced
import test_gpu_keys
import test_gpu_nan_parts
from anima_hip import rt

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MODES = {rt.F32: "f32", rt.BF16: "bf16", rt.F32X3: "f32x3"}
RAW_SAVES = 6.0  # attention.hip's kRowPassUs: cached keys, raw query rows

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "flash_plan_shape")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    "-Wall", "-Werror", "-I", os.path.join(ROOT, "anima-on-android_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "flash_plan_shape.cpp"), "-o", exe],
                   check=True)

    def ask(mode, BH, S_q, S_kv, causal=False, keys=None, saves=0.0):
        keys = mode != rt.F32 if keys is None else keys
        line = f"{MODES[mode]} {BH} {S_q} {S_kv} {int(causal)} {int(keys)} {saves}\n"
        run = subprocess.run([exe], input=line, capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stdout + run.stderr
        return run.stdout.strip()
    return ask


# Whole calls of anima_hip_attention_dev in every shape (us): the fastest one, with
# the next beside it.
@pytest.mark.parametrize("mode,BH,S_q,S_kv,fastest", [
    (rt.F32X3, 5, 64, 512, "split"),      # 24.1, keys 29.5
    (rt.F32X3, 16, 64, 512, "split"),     # 27.6, keys 31.2
    (rt.F32X3, 5, 256, 385, "split"),     # 26.8, keys 28.5
    (rt.F32X3, 32, 64, 512, "split"),     # 32.7, keys 36.7
    (rt.F32X3, 16, 256, 512, "keys"),     # split 1.2 more
    (rt.F32X3, 16, 256, 256, "keys"),
    (rt.F32X3, 16, 1024, 1024, "keys"),
    (rt.F32, 32, 257, 257, "split"),      # 52.2, small 60.5
    (rt.F32, 32, 320, 320, "split"),      # 52.6, balanced 60.9
    (rt.F32, 16, 768, 320, "balanced"),
    (rt.F32, 16, 600, 600, "balanced"),
    (rt.F32, 5, 64, 65, "split"),         # 21.9, small 27.5
    (rt.BF16, 5, 256, 1000, "keys"),
    (rt.BF16, 16, 768, 192, "small")])
def test_measured_shapes(shape, mode, BH, S_q, S_kv, fastest):
    assert shape(mode, BH, S_q, S_kv) == fastest


@pytest.mark.parametrize("mode,BH,S", [(rt.F32, 7, 2500), (rt.F32, 20, 1000), (rt.BF16, 9, 2000),
                                       (rt.F32X3, 7, 2500)])
def test_causal_split(shape, mode, BH, S):
    """Causal splits of which a third ends at once and the rest fills one round
    (f32: host calls 1376 against 1530 us whole, 1343 against 1414)."""
    assert shape(mode, BH, S, S, causal=True, keys=False) == "split"


@pytest.mark.parametrize("mode,B,H,S_q,S_kv", test_gpu_keys.CASES)
def test_keys_cases(shape, mode, B, H, S_q, S_kv):
    assert shape(mode, B * H, S_q, S_kv) == "keys"


@pytest.mark.parametrize("mode", test_gpu_keys.MODES)
@pytest.mark.parametrize("case", test_gpu_keys.RAW_CASES)
def test_raw_keys_cases(shape, mode, case):
    B, S_q, S_kv = case
    assert shape(mode, 16 * B, S_q, S_kv, saves=RAW_SAVES) == "keys"


def test_nan_cases(shape):
    for mode, S, _ in test_gpu_nan_parts.KEYS:
        assert shape(mode, 16, S, S) == "keys"
    for mode in (rt.F32X3, rt.BF16):
        assert shape(mode, 16, 100, 65, saves=RAW_SAVES) == "keys"
    for mode, BH, S_q, S_kv, _ in test_gpu_nan_parts.BALANCED:
        assert shape(mode, BH, S_q, S_kv, keys=False) == "balanced"
    for mode in MODES:
        assert shape(mode, 2, 961, 961, keys=False) == "split"


def test_balanced_cases(shape):
    for B, H, S_q, S_kv, modes in test_gpu_balanced.CASES:
        for mode in modes:
            assert shape(mode, B * H, S_q, S_kv) == "balanced"
