"""The DiT's small kernels at sizes around their workgroups.

The MLP at hidden widths around the GELU pass's workgroups of 1 to 4 waves of 512
values (one wave and the next ragged, one workgroup of two, five of one, two of
three, three of four) against the oracle's model; tolerances of the whole DiT's tests (1e-4 in the f32 mode, 3e-2
in bf16); and a model of enough blocks that the launches of all AdaLN layers give
each lane group two rows, at a width whose rows and columns come out ragged."""
import os
import sys

import numpy as np
import pytest

import oracle
from anima_hip import rt
from anima_hip.dit import AnimaDiT, DeviceArray, DiTConfig

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))
import dit_weights  # noqa: E402


def check(cfg, mode):
    rt.init()
    w = dit_weights.make(cfg["mlp_hidden"], **cfg)
    rng = np.random.default_rng(cfg["mlp_hidden"])
    x = rng.standard_normal((2, 16, 1, 6, 10), dtype=np.float32)
    ctx = rng.standard_normal((2, 7, 64), dtype=np.float32)
    sigma = np.array([0.7, 0.3], np.float32)
    keep = [DeviceArray.of(a) for a in w.values()]
    table = {n: (d.ptr, "BF16" if a.ndim == 2 else "F32", a.shape)
             for (n, a), d in zip(w.items(), keep)}
    print(f"dit {cfg} mode={mode}", flush=True)
    with AnimaDiT(table, DiTConfig.anima_2b(**cfg), mode) as m:
        out = m.forward(x, sigma, ctx)
    ref = oracle.dit_forward(x, sigma, ctx, w, cfg["blocks"], cfg["heads"], 128)
    err = float(np.abs(out - ref).max() / np.abs(ref).max())
    print(f"  normwise error {err:.3e}", flush=True)
    assert err <= (3e-2 if mode == rt.BF16 else 1e-4)


@pytest.mark.parametrize("mode", [rt.F32, rt.BF16])
@pytest.mark.parametrize("hidden", [264, 776, 2056, 3072, 6144])
def test_mlp_widths(hidden, mode):
    check(dict(dim=256, blocks=2, heads=2, head_dim=128, mlp_hidden=hidden, ctx_dim=64), mode)


def test_many_adaln_rows():
    check(dict(dim=520, blocks=22, heads=2, head_dim=128, mlp_hidden=256, ctx_dim=64), rt.F32)
