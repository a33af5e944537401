"""The f32-mode projection on f32 activations in tiles of 160 to 256 columns
(anima_hip_linear_dev): the float64 product of the activations' bf16 hi and lo
terms, and, where the kernel on term rows takes the shape too, the same bits
as the split pass and that kernel (activation rows that are not 16-byte aligned).

Bound: the 2K products of bf16 values are exact in f32 and added in f32, which
errs by about sqrt(2K) half units of 2^-24 of the result's scale when roundings
are independent; 2-norms over the whole result are held to sqrt(2K) * 2^-23.
"""
import numpy as np
import pytest

import oracle
from anima_hip import _lib, rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    rt.init()


def run(a, w, M, N, K, lda):
    from devmem import DevBuf
    lib = _lib.load()
    rows = np.full((M, lda), np.nan, np.float32)
    rows[:, :K] = a
    ldc = N + 4
    sb = lib.anima_hip_linear_scratch_bytes(M, K, rt.F32)
    da, dw, dc = DevBuf.of(rows), DevBuf.of(w), DevBuf.of(np.full((M, ldc), -7.0, np.float32))
    scr = DevBuf(sb)
    _lib.check(lib.anima_hip_linear_dev(da.addr, lda, dw.addr, K, dc.addr, ldc, M, N, K, rt.F32,
                                        scr.addr, sb, None), "linear_dev")
    c = dc.get((M, ldc))
    assert (c[:, N:] == -7.0).all()
    return c[:, :N]


# Columns of a tile: 160 (1536 x 6144 whole; 4352 x 2048, 2700 x 2040 a ragged
# last tile), 192 (2700 x 8192, 3333 x 6140), 224 (4552 x 8192, 3016 x 8100), 256
# (1100 x 8192); one to six chunks of K; ragged last rows.  The kernel on term
# rows takes K in multiples of 64.
@pytest.mark.parametrize("M,N,K,same_bits", [
    (1536, 6144, 32, False), (1100, 8192, 192, True), (4352, 2048, 192, True),
    (2700, 2040, 128, False), (2700, 8192, 64, True), (3333, 6140, 96, False),
    (4552, 8192, 64, True), (3016, 8100, 128, True)])
def test_tile_widths(M, N, K, same_bits):
    rng = np.random.default_rng(M + 3 * N + 5 * K)
    a = rng.standard_normal((M, K), dtype=np.float32)
    w = oracle.f32_to_bf16_bits(rng.standard_normal((N, K), dtype=np.float32))
    out = run(a, w, M, N, K, K)
    wf = oracle.bf16_bits_to_f32(w).astype(np.float64)
    hi = oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(a))
    lo = oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(a - hi))
    ref = (hi.astype(np.float64) + lo) @ wf.T
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"  2-norm {err:.3e}", flush=True)
    assert err <= np.sqrt(2 * K) * 2.0 ** -23
    if same_bits:
        assert np.array_equal(out.view(np.uint32), run(a, w, M, N, K, K + 2).view(np.uint32))
