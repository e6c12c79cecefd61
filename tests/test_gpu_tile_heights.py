"""The 256-token tiles' heights and the XCDs' runs of work: with k = E every expert holds all T tokens, so T walks
one tile, the rest of at most 32 rows past whole tiles (left as it is and, every expert ending in one, counted as
light), and equal tiles in 32-row steps. EMBER_GEMM_SHORT=0 keeps the packs, whose rule for 64-row tiles takes
layers this small, on 256-row tiles. A row's sums do not depend on its tile, so every row's bits are those of the
same token in a call of at most 256 tokens (one tile per expert), and the output holds the oracle's bar
(utils.cpp:704-748), with the down projection split over K (Q8_0, Q4_K) or not."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import rel_l2, run_gpu, run_oracle, same_bits, tile_table_tail

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [256, 257, 288, 289, 300, 513, 545, 700])
@pytest.mark.parametrize("wtype,pack,E", [(em.Q8_0, True, 2), (em.Q8_0, False, 3), (em.Q4_K, True, 2), (em.BF16, True, 2),
                                          (em.F16, False, 2)])
def test_tile_heights(gpu, monkeypatch, wtype, pack, E, T):
    spec = em.LayerSpec(d=256, d_ff=512, E=E, k=E, wtype=wtype, seed=5)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemm")
    monkeypatch.setenv("EMBER_GEMM_SHORT", "0")
    monkeypatch.setenv("EMBER_KSPLIT", "1")
    print(f"tile heights {em.TYPE_NAMES[wtype]} pack={pack} T={T}", flush=True)
    y = run_gpu(hl, x, pack=pack)
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
    for a in range(0, T, 200):
        assert same_bits(y[a:a + 200], run_gpu(hl, x[a:a + 200], pack=pack)), a
    if wtype not in (em.BF16, em.F16):  # (whose 256-token tiles do not split K)
        monkeypatch.setenv("EMBER_KSPLIT", "4")
        assert rel_l2(run_gpu(hl, x, pack=pack), y) < 1e-5


@pytest.mark.parametrize("T", [31, 32, 33, 96, 97, 129, 256, 300])
@pytest.mark.parametrize("wtype,pack,shared", [(em.BF16, True, 0), (em.F16, False, 0), (em.BF16, True, 192)])
def test_half_tiles_ragged(gpu, monkeypatch, wtype, pack, shared, T):
    """The BF16 / F16 256-token tiles: subtiles and activation loads past a tile's rows left out, weight rows past
    d_ff and d (320 = 2.5 x 128, 192 < 256), 6 and 10 K tiles of 32 columns (no multiple of the
    ring's four stages), a dense shared expert, against the oracle at the fp16 operands' 2e-3."""
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


def _runs(counts):
    """write_tiles' rule: tile heights, the XCDs' runs in 4096ths of a tile, and whether they follow the tiles' time."""
    tiles, weight, light, short = [], [], 0, False
    for n in counts:
        nt = -(-n // 256)
        h = 256 if nt <= 1 or n - (nt - 1) * 256 <= 32 else -(-(-(-n // nt)) // 32) * 32
        rows = [min(h, n - i * h) for i in range(nt)]
        rest = nt > 1 and rows[-1] <= 32
        light, short = light + rest, short or (nt > 0 and min(h, n) <= 224)
        tiles += rows
        weight += [832] * (nt - 1) + [384 if rest else 832] if nt else []
    timed = 2 * light >= sum(n > 0 for n in counts) and not short
    total, pos = sum(weight), []
    for x in range(9):
        if not timed:
            pos.append(len(tiles) * 4096 * x // 8)
            continue
        r, i = total * x // 8, 0
        while i < len(weight) - 1 and r >= weight[i]:
            r, i = r - weight[i], i + 1
        pos.append(i * 4096 + min(r * 4096 // weight[i], 4096))
    return tiles, pos, timed


def _routed_to(counts, d, seed):
    """Tokens that a one-hot router sends to expert e counts[e] times, in a shuffled order."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((sum(counts), d)).astype(np.float32) * 0.5
    e = rng.permutation(np.repeat(np.arange(len(counts)), counts))
    x[:, :len(counts)] = 0.0
    x[np.arange(len(e)), e] = 8.0
    return x


@pytest.mark.parametrize("counts,timed", [
    ((270, 262, 256, 250), True),           # two rests for four experts
    ((530, 514, 512, 500, 0, 257), True),   # rests behind two whole tiles, an expert without rows
    ((288, 288, 288, 288), True),
    ((270, 256, 256, 250), False),          # one rest
    ((270, 262, 289, 270), False),          # a pair of 160-row tiles
    ((270, 262, 150, 270), False),          # a tile of 150 rows
    ((700, 33, 0, 290), False),             # three tiles of 256, 256, 188; pairs
])
@pytest.mark.parametrize("wtype,pack", [(em.Q8_0, True), (em.Q4_K, True), (em.Q8_0, False), (em.BF16, True), (em.F16, False)])
def test_xcd_runs(gpu, monkeypatch, wtype, pack, counts, timed):
    """The tiles' number and the runs that the dispatch leaves in the scratch (the count in its last 256 bytes, the runs 64
    bytes on), by the rule restated above, and the output of segments of just these lengths against the oracle."""
    import torch

    monkeypatch.setenv("EMBER_MOE_PATH", "gemm")
    monkeypatch.setenv("EMBER_GEMM_SHORT", "0")  # 256-row tiles whatever the rule for 64-row ones says
    monkeypatch.setenv("EMBER_TAIL_PARTS", "1")
    E = len(counts)
    spec = em.LayerSpec(d=256, d_ff=512, E=E, k=1, wtype=wtype, seed=9)
    hl = em.make_host_layer(spec)
    hl.router = np.ascontiguousarray(np.eye(E, 256, dtype=np.float32).reshape(-1))
    x = _routed_to(counts, 256, 9)
    T = len(x)
    dl = em.DeviceLayer.upload(hl)
    if pack:
        buf = torch.empty(em.prefill_pack_bytes(dl.desc), dtype=torch.uint8, device="cuda")
        em.prefill_pack(dl.desc, buf)
        dl.tensors["pack"] = buf
    print(f"xcd runs {em.TYPE_NAMES[wtype]} pack={pack} {counts}", flush=True)
    y, scratch = dl.forward(torch.from_numpy(x).cuda())
    torch.cuda.synchronize()
    assert em.path(dl.desc, T) & em.PATH_TILES256
    offsets = em.scratch_routing(dl.desc, T, scratch)["offsets"]
    assert np.array_equal(np.diff(offsets), counts)
    tiles, pos, by_time = _runs(counts)
    assert by_time == timed
    assert tile_table_tail(dl.desc, T, scratch) == (len(tiles), pos)
    assert rel_l2(y.cpu().numpy(), run_oracle(hl, x)) < 2e-3


@pytest.mark.parametrize("T", [1050, 2048])
def test_xcd_runs_skewed(gpu, monkeypatch, T):
    """Uniform and skewed segments of eight experts: full tiles, equal tiles and light rests mixed."""
    monkeypatch.setenv("EMBER_GEMM_SHORT", "0")
    spec = em.LayerSpec(d=256, d_ff=512, E=8, k=2, wtype=em.Q8_0, seed=9, router_std=0.01 if T == 1050 else 0.2)
    hl = em.make_host_layer(spec)
    x = em.make_input(spec, T)
    y, scratch, dl = run_gpu(hl, x, pack=True, whole=True)
    tiles, pos, _ = _runs(np.diff(em.scratch_routing(dl.desc, T, scratch)["offsets"]))
    assert tile_table_tail(dl.desc, T, scratch) == (len(tiles), pos)
    assert np.isfinite(y).all()
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
