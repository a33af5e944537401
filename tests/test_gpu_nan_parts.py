"""NaN keys in launch shapes that share the keys of a query tile out.

A part of a row's keys whose every live score is NaN must not drop out of the
merge like a part that saw masked keys only: the reference's running sum becomes
NaN (flash_attention.h:145-201), and only a row without any score above -inf keeps
its zeros.  The NaN keys sit where one part holds nothing else: the last key, alone
in its key tile, or all tiles of one key group.  NaN exactly where the oracle has
it, zeros where it has them, and elsewhere within the mode's tolerance (max-abs 1e-4
for f32 and f32x3, normwise 2e-2 for bf16).  Balanced grids also see an infinite
key (alone in its part: -inf or +inf scores, as a row's sign has it; not in f32x3,
whose low term of it is NaN) and a row whose scores are all low.
"""
import ctypes as ct

import numpy as np
import pytest

import oracle
from anima_hip import _lib, rt

pytestmark = pytest.mark.gpu

D = 128
NAMES = {rt.F32: "f32", rt.BF16: "bf16", rt.F32X3: "f32x3"}


@pytest.fixture(scope="module", autouse=True)
def _init():
    rt.init()


def check(got, ref, mode):
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[ref == 0], 0.0)
    if nan.all():
        return
    err = float(np.abs(got[~nan] - ref[~nan]).max())
    print(f"  max-abs {err:.3e}, {nan.sum()} NaN", flush=True)
    assert err <= (2e-2 * float(np.abs(ref[~nan]).max()) if mode == rt.BF16 else 1e-4)


# The keys shape, prepared rows: the last key is alone in its tile (32 keys in
# f32x3, 64 in bf16) and that tile in its group; or one group's tiles.
KEYS = [(rt.F32X3, 65, [64]), (rt.F32X3, 97, [96]), (rt.BF16, 193, [192]),
        (rt.F32X3, 193, [*range(32, 64), *range(160, 192)]), (rt.BF16, 256, [*range(64, 128)])]


@pytest.mark.parametrize("mode,S,nan_keys", KEYS)
def test_keys_shape(mode, S, nan_keys):
    from devmem import DevBuf
    lib = _lib.load()
    H = 16
    rng = np.random.default_rng(S + mode)
    q, k, v = (rng.standard_normal((1, S, H, D), dtype=np.float32) for _ in range(3))
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    for h in (0, 7):
        k[0, nan_keys, h, 3 * h] = np.nan
    q[0, 5, 7, 1] = np.nan  # every score of that row
    bufs = [DevBuf.of(x) for x in (q, k, v, qw, kw)]
    out = DevBuf(q.nbytes)
    n = lib.anima_hip_attention_scratch_bytes(1, S, 1, S, H, D, mode)
    scratch = DevBuf(n)
    print(f"keys {NAMES[mode]} S={S}", flush=True)
    _lib.check(lib.anima_hip_attention_dev(*(b.addr for b in bufs), None, out.addr, scratch.addr,
                                           n, 1, S, 1, S, H, D, ct.c_float(1e-6), mode, None),
               "attention_dev")
    ref = oracle.attention_dataflow(q, k, v, qw, kw, None)
    assert np.isnan(ref[0, :5, (0, 7)]).all() and (ref[0, 5, 7] == 0).all()
    check(out.get(q.shape), ref, mode)


@pytest.mark.parametrize("mode", [rt.F32X3, rt.BF16])
def test_keys_shape_raw_queries(mode):
    rng = np.random.default_rng(65 + mode)
    B, H, C, S_q, S_kv = 1, 16, 64, 100, 65
    ctx = rng.standard_normal((1, S_kv, C), dtype=np.float32)
    ctx[0, 64, 9] = np.nan
    bits = [oracle.f32_to_bf16_bits(rng.standard_normal((H * D, C), dtype=np.float32) * 0.1)
            for _ in range(2)]
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((B, S_q, H, D), dtype=np.float32)
    q[0, 40, 2, 7] = np.nan
    print(f"keys raw {NAMES[mode]} S_kv={S_kv}", flush=True)
    kv = rt.ContextKV(ctx, *bits, kw, heads=H, head_dim=D, mode=mode)
    try:
        got = kv.attend(q, qw)
    finally:
        kv.close()
    ref = np.full(q.shape, np.nan, np.float32)
    ref[0, 40, 2] = 0
    check(got, ref, mode)


# Balanced grids of one ragged query tile a head, the last key alone in its key
# tile; the first head named has that tile as a part of its own, and the second.
# An odd head count keeps the host call in one group of heads.
BALANCED = [(rt.F32, 27, 200, 1601, (1, 4, 7)), (rt.F32X3, 27, 200, 1601, (1, 4, 7)),
            (rt.BF16, 27, 200, 3329, (4, 10, 16))]


@pytest.mark.parametrize("mode,BH,S_q,S_kv,heads", BALANCED)
def test_balanced_grid(mode, BH, S_q, S_kv, heads):
    rng = np.random.default_rng(S_kv + mode)
    q = rng.standard_normal((BH, S_q, D), dtype=np.float32)
    k, v = (rng.standard_normal((BH, S_kv, D), dtype=np.float32) for _ in range(2))
    for h in heads[:2]:
        k[h, -1, 17] = np.nan
    k[2, 70, 5] = np.nan  # among finite keys of its part
    q[heads[0], 9, 0] = np.nan  # every score of that row
    v[0, 100, 11] = np.nan
    if mode != rt.F32X3:
        k[heads[2], -1, 3] = np.inf
    k[3] = np.abs(k[3])
    q[3, 50] = -4.0
    print(f"balanced {NAMES[mode]} BH={BH} S_q={S_q} S_kv={S_kv}", flush=True)
    got = rt.sdpa(q, k, v, scale=0.088, mode=mode)
    check(got, oracle.flash_sdpa(q, k, v, 0.088, threads=8), mode)


@pytest.mark.parametrize("mode", [rt.F32, rt.F32X3, rt.BF16])
def test_split_grid(mode):
    """Two heads of 961 keys: a split of one ragged key tile."""
    rng = np.random.default_rng(961 + mode)
    q, k, v = (rng.standard_normal((2, 961, D), dtype=np.float32) for _ in range(3))
    k[1, 960, 2] = np.nan
    q[1, 7, 0] = np.nan
    print(f"split {NAMES[mode]}", flush=True)
    check(rt.sdpa(q, k, v, scale=0.088, mode=mode), oracle.flash_sdpa(q, k, v, 0.088, threads=8),
          mode)
