"""The 256-token tiles' heights and the XCDs' runs of work: with k = E every expert holds all T tokens, so T walks
one tile, the rest of at most 32 rows past whole tiles (left as it is and, being more than a sixth of the tiles,
counted as light), and equal tiles in 32-row steps. A row's sums do not depend on its tile, so every
row's bits are those of the same token in a call of at most 256 tokens (one tile per expert), and the output holds
the oracle's bar (utils.cpp:704-748), with the down projection split over K or not."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import rel_l2, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [256, 257, 288, 289, 300, 513, 545, 700])
@pytest.mark.parametrize("wtype,pack,E", [(em.Q8_0, True, 2), (em.Q8_0, False, 3), (em.Q4_K, True, 2), (em.BF16, True, 2), (em.F16, False, 2)])
def test_tile_heights(gpu, monkeypatch, wtype, pack, E, T):
    spec = em.LayerSpec(d=256, d_ff=512, E=E, k=E, wtype=wtype, seed=5)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemm")
    monkeypatch.setenv("EMBER_KSPLIT", "1")
    print(f"tile heights {em.TYPE_NAMES[wtype]} pack={pack} T={T}", flush=True)
    y = run_gpu(hl, x, pack=pack)
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
    for a in range(0, T, 200):
        assert same_bits(y[a:a + 200], run_gpu(hl, x[a:a + 200], pack=pack)), a
    monkeypatch.setenv("EMBER_KSPLIT", "4")
    assert rel_l2(run_gpu(hl, x, pack=pack), y) < 1e-5


@pytest.mark.parametrize("T", [31, 32, 33, 96, 97, 129, 256, 300])
@pytest.mark.parametrize("wtype,pack,shared", [(em.BF16, True, 0), (em.F16, False, 0), (em.BF16, True, 192)])
def test_half_tiles_ragged(gpu, monkeypatch, wtype, pack, shared, T):
    """The BF16 / F16 256-token tiles: subtiles and activation loads past a tile's rows left out, weight rows past
    d_ff and d (320 = 2.5 x 128, 192 < 256), an even and an odd number of 32-column K tiles per part, a dense shared
    expert, against the oracle at the fp16 operands' 2e-3."""
    spec = em.LayerSpec(d=192, d_ff=320, E=3, k=3, wtype=wtype, seed=T, d_ff_shared=shared)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemm")
    monkeypatch.setenv("EMBER_MOE_SHARED_PATH", "gemm")
    print(f"half tiles {em.TYPE_NAMES[wtype]} T={T} shared={shared}", flush=True)
    y = run_gpu(hl, x, pack=pack)
    assert np.isfinite(y).all()
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
    assert same_bits(y, run_gpu(hl, x, pack=pack))


@pytest.mark.parametrize("T", [1050, 2048])
def test_xcd_runs_skewed(gpu, T):
    """Uniform and skewed segments of eight experts: full tiles, equal tiles and light rests mixed."""
    spec = em.LayerSpec(d=256, d_ff=512, E=8, k=2, wtype=em.Q8_0, seed=9, router_std=0.01 if T == 1050 else 0.2)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    y = run_gpu(hl, x, pack=True)
    assert np.isfinite(y).all()
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
