"""The attention sub-layer at sizes where the f32-activation kernel runs the output
projection and its epilogue updates the residual (2 heads keep the CPU's part
small), against the oracle's composition at the stated 1e-4 of the update's scale:
batch boundaries inside a wave's 32 rows, a ragged last tile, one entry.
"""
import ctypes as ct

import numpy as np
import pytest

import oracle
from anima_hip import _lib, rt
from anima_hip.rope import generate_rope_freqs

pytestmark = pytest.mark.gpu

DM, H, D = 2048, 2, 128


@pytest.mark.parametrize("mode", [rt.F32, rt.F32X3])
@pytest.mark.parametrize("B,gh,gw", [(2, 27, 50), (3, 17, 53), (1, 50, 55)])
def test_residual_epilogue(B, gh, gw, mode):
    from devmem import DevBuf
    rt.init()
    lib = _lib.load()
    S = gh * gw
    rng = np.random.default_rng(S + mode)
    x = rng.standard_normal((B, S, DM), dtype=np.float32)
    mod = (rng.standard_normal((B, 3, DM)) * 0.5).astype(np.float32)
    w = [oracle.f32_to_bf16_bits(rng.standard_normal(s, dtype=np.float32) * np.float32(0.02))
         for s in [(H * D, DM)] * 3 + [(DM, H * D)]]
    qw, kw = (rng.uniform(0.5, 1.5, D).astype(np.float32) for _ in range(2))
    f = generate_rope_freqs(gh, gw)
    bufs = [DevBuf.of(a) for a in (x, mod, *w, qw, kw, f)]
    n = lib.anima_hip_attention_block_scratch_bytes(None, B, S, DM, H, D, mode)
    scratch = DevBuf(n)
    print(f"block B={B} S={S} mode={mode}", flush=True)
    _lib.check(lib.anima_hip_attention_block_dev(
        *[b.addr for b in bufs], None, B, S, DM, H, D, ct.c_float(1e-6), mode, scratch.addr, n,
        None), "attention_block_dev")
    out = bufs[0].get(x.shape)
    ref = oracle.attention_block(x, mod, *w, qw, kw, f, None, heads=H, head_dim=D,
                                 sdpa=lambda a, b, c: oracle.flash_sdpa(a, b, c, threads=8))
    d_ref = ref - x
    err = float(np.abs((out - x) - d_ref).max() / np.abs(d_ref).max())
    print(f"  rel err {err:.3e}", flush=True)
    assert np.isfinite(out).all() and err <= 1e-4
