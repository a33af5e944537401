"""anima_hip_gemm_dev with f32 weights: the DMA-staged tile kernel (16-byte aligned
rows, K a multiple of 32) and the bounds-checked kernel for everything else,
against float64 products.

Bound: K products rounded and added in f32 in one or two chains err by about
sqrt(K) half units of 2^-24 of the result's scale when roundings are
independent; 2-norms over the whole result are held to sqrt(K) * 2^-23.
"""

import numpy as np
import pytest

from anima_hip import _lib, rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    rt.init()


# (M, N, K, lda - K, ldw - K, ldc - N, offset of A in floats): one row and one
# column, tile edges and one past them, one to three chunks of K, wide rows, and
# forms the tile kernel does not take (unaligned A, odd row strides, K = 33).
CASES = [(1, 1, 32, 0, 0, 0, 0), (64, 64, 64, 0, 0, 0, 0), (65, 63, 96, 4, 8, 3, 0),
         (63, 129, 2048, 0, 0, 0, 0), (300, 200, 32, 4, 4, 64, 0), (257, 640, 1024, 0, 12, 1, 4),
         (65, 63, 96, 0, 0, 0, 1), (65, 63, 96, 2, 0, 0, 0), (65, 63, 96, 0, 1, 0, 0),
         (65, 63, 33, 0, 0, 0, 0)]


@pytest.mark.parametrize("M,N,K,pa,pw,pc,off", CASES)
def test_gemm_f32_weights(M, N, K, pa, pw, pc, off):
    from devmem import DevBuf
    lib = _lib.load()
    rng = np.random.default_rng(M + 3 * N + 5 * K + 7 * pa + off)
    a = rng.standard_normal((M, K + pa), dtype=np.float32)
    w = rng.standard_normal((N, K + pw), dtype=np.float32)
    flat = np.concatenate([np.full(off, np.nan, np.float32), a.reshape(-1)])
    da, dw = DevBuf.of(flat), DevBuf.of(w)
    dc = DevBuf.of(np.full((M + 1, N + pc), np.float32(-7.25)))
    print(f"gemm f32 M={M} N={N} K={K} pads={pa},{pw},{pc} offset={off}", flush=True)
    _lib.check(lib.anima_hip_gemm_dev(da.addr + 4 * off, K + pa, dw.addr, 0, K + pw, dc.addr,
                                      N + pc, M, N, K, None), "gemm_dev")
    out = dc.get((M + 1, N + pc))
    ref = a[:, :K].astype(np.float64) @ w[:, :K].astype(np.float64).T
    err = np.linalg.norm(out[:M, :N] - ref) / np.linalg.norm(ref)
    print(f"  2-norm error {err:.2e}", flush=True)
    assert err <= np.sqrt(K) * 2.0 ** -23
    assert (out[M:] == -7.25).all() and (out[:, N:] == -7.25).all()
