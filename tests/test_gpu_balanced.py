"""Balanced flash grids: the query tiles that do not come out even over the CUs
run with their key tiles dealt out evenly, through anima_hip_attention_dev.

Against the oracle at the stated tolerances (max-abs 1e-4 in f32 and f32x3,
normwise 2e-2 in bf16), on heads of the whole tiles and of the dealt ones; and
with scratch of the size the call needs without balancing, which runs too and
differs by summation order only.
"""
import ctypes as ct

import numpy as np
import pytest

import oracle
from anima_hip import _lib, rt

pytestmark = pytest.mark.gpu

D = 128


@pytest.fixture(scope="module", autouse=True)
def _init():
    rt.init()


def _round_up(n):
    return -(-n // 256) * 256


def _required(B, S_q, S_kv, H, mode):
    """Scratch of the prepared operands; grids of 256 and more query tiles and
    these small ones need no split partials on top."""
    w = 2 if mode == rt.BF16 else 4
    n = _round_up(B * S_q * H * D * w) + _round_up(B * S_kv * H * D * w)
    if mode != rt.F32:
        n += _round_up(B * H * D * (-(-S_kv // 64) * 64) * w)
    return n


# Query tiles of 256 rows: 272 = 256 + 16 (ragged last query tile, whole key
# tiles), 290 = 256 + 34 with a ragged last key tile, 200 < 256 and 255 < 256
# query tiles without a whole round (f32 only: the bf16-MFMA modes run those
# whole), 513 = 2 rounds + 1.
CASES = [(1, 17, 4000, 2560, (rt.F32, rt.BF16, rt.F32X3)),
         (2, 29, 1100, 2497, (rt.F32, rt.BF16, rt.F32X3)),
         (1, 20, 2500, 3000, (rt.F32,)),
         (1, 129, 300, 1666, (rt.F32,)),
         (1, 171, 520, 3136, (rt.F32, rt.BF16, rt.F32X3))]


@pytest.mark.parametrize("B,H,S_q,S_kv,mode", [c[:4] + (m,) for c in CASES for m in c[4]])
def test_balanced_grid(B, H, S_q, S_kv, mode):
    from devmem import DevBuf
    lib = _lib.load()
    rng = np.random.default_rng(B + 3 * H + S_q + S_kv + mode)
    q = rng.standard_normal((B, S_q, H, D), dtype=np.float32)
    k, v = (rng.standard_normal((B, S_kv, H, D), dtype=np.float32) for _ in range(2))
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    bufs = [DevBuf.of(x) for x in (q, k, v, qw, kw)]
    out = DevBuf(q.nbytes)
    n = lib.anima_hip_attention_scratch_bytes(B, S_q, B, S_kv, H, D, mode)
    required = _required(B, S_q, S_kv, H, mode)
    assert n > required, "the shape does not run balanced"
    scratch = DevBuf(n)
    res = []
    for nbytes in (n, required, required - 1):
        print(f"balanced B={B} H={H} S_q={S_q} S_kv={S_kv} mode={mode} scratch={nbytes}",
              flush=True)
        out.put(np.full(q.shape, np.nan, np.float32), 0)
        ok = lib.anima_hip_attention_dev(*(b.addr for b in bufs), None, out.addr, scratch.addr,
                                         nbytes, B, S_q, B, S_kv, H, D, ct.c_float(1e-6), mode,
                                         None)
        if nbytes < required:
            assert not ok
        else:
            _lib.check(ok, "attention_dev")
            res.append(out.get(q.shape))
    bound = 2e-2 * float(np.abs(res[1]).max()) if mode == rt.BF16 else 1e-4
    assert float(np.abs(res[0] - res[1]).max()) <= bound
    # The first heads are in whole tiles (where there are any), the last dealt.
    for b, h in ((0, 0), (B - 1, H - 2), (B - 1, H - 1)):
        one = [x[b:b + 1, :, h:h + 1] for x in (q, k, v)]
        ref = oracle.attention_dataflow(*one, qw, kw, None,
                                        sdpa=lambda a, c, d: oracle.flash_sdpa(a, c, d, threads=4))
        err = float(np.abs(res[0][b, :, h] - ref[0, :, 0]).max())
        print(f"  b={b} h={h}: max-abs {err:.3e}", flush=True)
        assert err <= (2e-2 * float(np.abs(ref).max()) if mode == rt.BF16 else 1e-4)
