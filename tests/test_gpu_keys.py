"""Small attention grids whose waves share the keys of 64 query rows, through
anima_hip_attention_dev (prepared query rows) and the cached cross-attention
(raw query rows), against the oracle at the stated tolerances: one ragged query
tile and a full grid of 256; one key past a tile, key ranges that leave key
groups idle in the last round, several rounds.  test_flash_plan.py holds CASES and
RAW_CASES to the shape they are here for; OTHER runs small grids beside it.
"""
import ctypes as ct

import numpy as np
import pytest

import oracle
from anima_hip import _lib, rt

pytestmark = pytest.mark.gpu

D = 128
MODES = [rt.F32X3, rt.BF16]


@pytest.fixture(scope="module", autouse=True)
def _init():
    rt.init()


def _check(out, ref, mode):
    err = float(np.abs(out - ref).max())
    print(f"  max-abs {err:.3e}", flush=True)
    assert err <= (2e-2 * float(np.abs(ref).max()) if mode == rt.BF16 else 1e-4)


CASES = [(rt.F32X3, 1, 3, 65, 65), (rt.F32X3, 1, 16, 200, 129), (rt.F32X3, 2, 5, 64, 300),
         (rt.F32X3, 1, 16, 1024, 96), (rt.F32X3, 1, 16, 1000, 1000), (rt.BF16, 1, 2, 1, 1000),
         (rt.BF16, 1, 16, 200, 193), (rt.BF16, 1, 16, 1024, 250), (rt.BF16, 1, 16, 200, 600),
         (rt.BF16, 2, 5, 64, 900)]
OTHER = [(rt.F32X3, 1, 2, 1, 1000), (rt.BF16, 1, 3, 65, 65), (rt.BF16, 1, 16, 200, 129),
         (rt.BF16, 2, 5, 64, 300), (rt.BF16, 1, 16, 1024, 96)]


@pytest.mark.parametrize("mode,B,H,S_q,S_kv", CASES + OTHER)
def test_keys_shape(mode, B, H, S_q, S_kv):
    from devmem import DevBuf
    lib = _lib.load()
    rng = np.random.default_rng(B + H + S_q + S_kv + mode)
    q = rng.standard_normal((B, S_q, H, D), dtype=np.float32)
    k, v = (rng.standard_normal((B, S_kv, H, D), dtype=np.float32) for _ in range(2))
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    q[0, 0, 0, 5] = np.nan  # every score of that row: zeros, as the reference leaves it
    v[0, 7, 1, 9] = np.nan  # that column of its head
    bufs = [DevBuf.of(x) for x in (q, k, v, qw, kw)]
    out = DevBuf.of(np.full((B * S_q + 1, H, D), np.float32(-7.25)))
    n = lib.anima_hip_attention_scratch_bytes(B, S_q, B, S_kv, H, D, mode)
    scratch = DevBuf(n)
    print(f"keys B={B} H={H} S_q={S_q} S_kv={S_kv} mode={mode}", flush=True)
    _lib.check(lib.anima_hip_attention_dev(*(b.addr for b in bufs), None, out.addr, scratch.addr,
                                           n, B, S_q, B, S_kv, H, D, ct.c_float(1e-6), mode, None),
               "attention_dev")
    got = out.get((B * S_q + 1, H, D))
    assert (got[-1] == -7.25).all()
    got = got[:-1].reshape(B, S_q, H, D)
    ref = oracle.attention_dataflow(q, k, v, qw, kw, None)
    nan = np.isnan(ref)
    assert nan.any() and (ref[0, 0, 0] == 0).all()
    np.testing.assert_array_equal(np.isnan(got), nan)
    assert (got[0, 0, 0] == 0).all()
    _check(np.where(nan, 0, got), np.where(nan, 0, ref), mode)


RAW_CASES = [(1, 100, 77), (2, 256, 512), (1, 1000, 65)]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("B,S_q,S_kv", RAW_CASES)
def test_keys_shape_raw_queries(B, S_q, S_kv, mode):
    rng = np.random.default_rng(B + S_q + S_kv + 7 * mode)
    H, C = 16, 256
    ctx = rng.standard_normal((1, S_kv, C), dtype=np.float32)
    bits = [oracle.f32_to_bf16_bits(rng.standard_normal((H * D, C), dtype=np.float32) * 0.06)
            for _ in range(2)]
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((B, S_q, H, D), dtype=np.float32)
    print(f"keys raw B={B} S_q={S_q} S_kv={S_kv} mode={mode}", flush=True)
    kv = rt.ContextKV(ctx, *bits, kw, heads=H, head_dim=D, mode=mode)
    try:
        got = kv.attend(q, qw)
    finally:
        kv.close()
    k, v = (np.broadcast_to(oracle.gemm_bf16(ctx[0], b).reshape(1, S_kv, H, D),
                            (B, S_kv, H, D)) for b in bits)
    _check(got, oracle.attention_dataflow(q, k, v, qw, kw, None), mode)
