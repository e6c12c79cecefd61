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
    """Unforced: segments of any length, a dense shared expert (the GEMV up to 64 rows, tiles beyond)."""
    spec = em.LayerSpec(d=192, d_ff=320, E=8, k=2, wtype=em.F32, seed=T, weight_std=0.1, d_ff_shared=224)
    hl = em.make_host_layer(spec)
    dl = em.DeviceLayer.upload(hl)
    assert em.path(dl.desc, T) & em.PATH_TILES64
    x = em.make_input(spec, T)
    assert rel_l2(run_gpu(hl, x), run_oracle(hl, x)) < 1e-6
