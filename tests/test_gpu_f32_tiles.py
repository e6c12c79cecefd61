"""The FP32 MFMA tiles of F32 stacks (64 tokens x 64 weight rows x 32 columns): with k = E every expert holds
all T tokens, so T walks the edges of a tile (a wave's 16 activation rows, the 32-token halves, the tile), d and
d_ff those of the columns (whole tiles in pairs, an odd tile, a tile of 4 columns) and of the weight rows (32 gate
+ 32 up, 64 down, both ragged), and the down projection's K split. Held to the oracle (utils.cpp:704-748) at
1e-6 rel-L2: the layer's F32 sums are off by ~1.7e-7 on either path, four times that with room for short
sums, and no further off than the GEMV's are by more than a third (both are rounding noise of equal depth)."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import rel_l2, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 16, 17, 31, 32, 33, 63, 64, 65, 130])
@pytest.mark.parametrize("d,d_ff", [(256, 688), (100, 36), (1024, 1504), (96, 132)])
def test_f32_tiles(gpu, monkeypatch, d, d_ff, T):
    spec = em.LayerSpec(d=d, d_ff=d_ff, E=2, k=2, wtype=em.F32, seed=T, weight_std=0.1)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    print(f"f32 tiles d={d} d_ff={d_ff} T={T}", flush=True)
    want = run_oracle(hl, x)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemv")
    gemv = rel_l2(run_gpu(hl, x), want)
    monkeypatch.setenv("EMBER_MOE_PATH", "skinny")
    y = run_gpu(hl, x)
    err = rel_l2(y, want)
    print(f"  rel-L2 {err:.2e}, GEMV {gemv:.2e}", flush=True)
    assert np.isfinite(y).all()
    assert err < 1e-6 and err < 1.34 * gemv + 2e-8
    assert same_bits(y, run_gpu(hl, x))


@pytest.mark.parametrize("T", [20, 96])
def test_f32_tiles_routed_and_shared(gpu, T):
    """Unforced: segments of any length, a dense shared expert on the tiles too."""
    spec = em.LayerSpec(d=192, d_ff=320, E=8, k=2, wtype=em.F32, seed=T, weight_std=0.1, d_ff_shared=224)
    hl = em.make_host_layer(spec)
    dl = em.DeviceLayer.upload(hl)
    assert em.path(dl.desc, T) & em.PATH_TILES64 and em.path(dl.desc, T) & em.PATH_SHARED_MFMA
    x = em.make_input(spec, T)
    assert rel_l2(run_gpu(hl, x), run_oracle(hl, x)) < 1e-6


def _classes(a):
    """0 finite, 1 +Inf, 2 -Inf, 3 NaN."""
    return np.where(np.isnan(a), 3, np.where(np.isposinf(a), 1, np.where(np.isneginf(a), 2, 0)))


@pytest.mark.parametrize("T", [5, 40, 70])
@pytest.mark.parametrize("kind", ["inf", "nan", "overflow"])
@pytest.mark.parametrize("stack,col", [("down", 3), ("down", 170), ("down", 319), ("up", 0), ("up", 131), ("up", 255),
                                       ("gate", 70)])
def test_f32_tiles_keep_infinities(gpu, monkeypatch, stack, col, kind, T):
    """An infinite or NaN weight, or sums past the largest float, in an early, a middle and the last group of 64
    columns (the compensated sums' step), and in the last but one of an odd number of 32-column tiles: every output
    is finite, +Inf, -Inf or NaN as on the GEMV, and the finite ones hold the tiles' bar against it. One expert's rows
    only, with operands of one sign in the overflowing sums, so that no order of additions decides."""
    spec = em.LayerSpec(d=256, d_ff=320, E=2, k=2, wtype=em.F32, seed=11, weight_std=0.1)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    rows, K = (spec.d, spec.d_ff) if stack == "down" else (spec.d_ff, spec.d)
    w = getattr(hl, stack).view(np.float32).reshape(spec.E, rows, K)
    bad = [0, 33, rows - 1] if stack == "down" else [45]  # (one hidden value: its sign decides each output's)
    for r in bad:
        if kind == "overflow":  # two products of 3e38 a column group apart; the rest of the row stays
            x[:, [col % spec.d, (col + 64) % spec.d]] = 1.0
            w[1, r, [col, (col + 64) % K]] = np.float32(3e38)
        else:
            w[1, r, col] = np.inf if kind == "inf" else np.nan
    setattr(hl, stack, np.ascontiguousarray(w).view(np.uint8).reshape(-1))
    print(f"f32 tiles {kind} in {stack} column {col} T={T}", flush=True)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemv")
    want = run_gpu(hl, x)
    monkeypatch.setenv("EMBER_MOE_PATH", "skinny")
    y = run_gpu(hl, x)
    cls = _classes(want)
    assert cls.any() and (kind == "nan" or (cls != 3).any())
    assert np.array_equal(_classes(y), cls)
    ok = cls == 0
    if ok.any():
        assert rel_l2(y[ok], want[ok]) < 1e-6
