"""Batches of more than 64 tokens on the prefill packs' 64-row tiles (the 256-token path's short ring), chosen by
the mean rows per expert, and a Q8_0 shared expert's batch on the dense 64-token tiles, its down projection split
over K. The routed tiles multiply the same fragments in the same order as the 256-row ones (EMBER_GEMM_SHORT=0):
bit-identical outputs. So do the shared expert's gate/up tiles; the K split of its down projection changes the
order of FP32 sums: rel-L2 of about sqrt(K) 2^-24 = 3e-6 at most for K <= 2048 against the 256-row tiles. Both are
held to the oracle (utils.cpp:704-748) at the 2e-3 rel-L2 bar of the FP16 tiles."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import rel_l2, run_oracle, same_bits, tile_table_tail


def _layer(kw, pack=True):
    import torch

    spec = em.LayerSpec(seed=67, **kw)
    hl = em.make_host_layer(spec)
    dl = em.DeviceLayer.upload(hl)
    if pack:
        buf = torch.empty(em.prefill_pack_bytes(dl.desc), dtype=torch.uint8, device="cuda")
        em.prefill_pack(dl.desc, buf)
        dl.tensors["pack"] = buf
    return spec, hl, dl


def _run(dl, x):
    import torch

    out, _ = dl.forward(torch.from_numpy(np.ascontiguousarray(x)).cuda())
    torch.cuda.synchronize()
    return out.cpu().numpy()


# (a selection bias of the scores' own spread skews the segments, so that some pass 64 rows)
WIDE = dict(d=512, d_ff=512, E=64, k=2, bias_std=0.02)  # 64 experts x 4 column tiles: a block for every CU
FEW = dict(d=512, d_ff=768, E=4, k=2, bias_std=0.15)
CASES = {
    # name: (spec kwargs, T): T k / E mean rows, the rule's ends and segments past 64 rows ("past" and "below": the batch
    # next to an end that keeps 256-row tiles)
    "q8_first": (dict(WIDE, wtype=em.Q8_0, bias_std=0.3), 65),
    "q8_last": (dict(WIDE, wtype=em.Q8_0), 1280),
    "q8_past": (dict(WIDE, wtype=em.Q8_0), 1281),
    "q4_last": (dict(WIDE, wtype=em.Q4_K), 1856),
    "q4_past": (dict(WIDE, wtype=em.Q4_K), 1857),
    "few_below": (dict(FEW, wtype=em.Q8_0), 104),
    "few_first": (dict(FEW, wtype=em.Q8_0), 105),
    "few_q4": (dict(FEW, wtype=em.Q4_K), 777),
    "all_on_one": (dict(d=512, d_ff=512, E=64, k=1, wtype=em.Q8_0, bias_std=50.0), 193),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_short_tiles_of_batches_same_bits(gpu, monkeypatch, name):
    kw, T = CASES[name]
    spec, hl, dl = _layer(kw)
    x = em.make_input(spec, T, seed=68)
    monkeypatch.setenv("EMBER_MOE_PATH", "gemm")
    monkeypatch.setenv("EMBER_TAIL_PARTS", "1")
    print(f"short tiles of a batch {name} T={T}", flush=True)
    import torch

    out, scratch = dl.forward(torch.from_numpy(np.ascontiguousarray(x)).cuda())
    torch.cuda.synchronize()
    y = out.cpu().numpy()
    counts = np.diff(em.scratch_routing(dl.desc, T, scratch)["offsets"])
    rows = 256 if name.endswith(("past", "below")) else 64
    assert tile_table_tail(dl.desc, T, scratch)[0] == int(np.sum(-(-counts // rows)))
    assert np.sum(-(-counts // 64)) > np.sum(-(-counts // 256))
    if rows == 64:
        monkeypatch.setenv("EMBER_GEMM_SHORT", "0")
        assert same_bits(y, _run(dl, x))
    err = rel_l2(y, run_oracle(hl, x))
    print(f"  rel-L2 vs oracle {err:.2e}", flush=True)
    assert err < 2e-3, err


@pytest.mark.gpu
@pytest.mark.parametrize("T", [9, 65, 200])
def test_q8_shared_expert_on_dense_tiles(gpu, monkeypatch, T):
    spec, hl, dl = _layer(dict(d=512, d_ff=512, E=8, k=2, wtype=em.Q8_0, d_ff_shared=1984), pack=False)
    x = em.make_input(spec, T, seed=69)
    print(f"Q8_0 shared expert T={T}", flush=True)
    y = _run(dl, x)
    monkeypatch.setenv("EMBER_MOE_SHARED_PATH", "skinny")
    assert same_bits(y, _run(dl, x))  # the path it takes by itself
    monkeypatch.setenv("EMBER_MOE_SHARED_PATH", "gemm")
    diff = rel_l2(y, _run(dl, x))
    print(f"  rel-L2 vs the 256-row tiles {diff:.2e}", flush=True)
    assert diff < 3e-6
    err = rel_l2(y, run_oracle(hl, x))
    assert err < 2e-3, err


def _desc(kw):
    spec = em.LayerSpec(**kw)
    L = em.Layer()
    for n, v in dict(d=spec.d, d_ff=spec.d_ff, E=spec.E, k=spec.k, d_ff_shared=spec.d_ff_shared).items():
        setattr(L, n, v)
    sh = ("gate_shared", "up_shared", "down_shared") if spec.d_ff_shared else ()
    for n in ("gate", "up", "down") + sh:
        setattr(L, n, 1 << 20)  # (never read)
        setattr(L, n.split("_")[0] + ("_shared_type" if "_" in n else "_type"), spec.wtype)
    L.router = 1 << 20
    return L


@pytest.mark.parametrize("kw,T", [
    (dict(d=2048, d_ff=1408, E=64, k=6, wtype=em.Q8_0, d_ff_shared=2816), 120),  # 33.2 MB without the K split's parts
    (dict(d=64, d_ff=64, E=8, k=4, wtype=em.F32), 6412),  # 4 KiB below the buffer's size without the tile table
])
def test_scratch_stays_within_the_no_allocation_buffer(kw, T):
    assert 0 < em.scratch_bytes(_desc(kw), T) <= 32 << 20


@pytest.mark.parametrize("T", [3, 16, 64, 100])
def test_q8_shared_expert_takes_no_room_for_gate_up_parts(T):
    """Only the down projection of a Q8_0 shared expert is split over K: beside its rows of h, y and converted x, the
    shared expert adds the down parts, which stay within its down weights' bytes, and no parts of gate / up dots."""
    kw = dict(d=2048, d_ff=1408, E=64, k=6, wtype=em.Q8_0)
    n, d = 2816, kw["d"]
    room = em.scratch_bytes(_desc(dict(kw, d_ff_shared=n)), T) - em.scratch_bytes(_desc(kw), T)
    rows = T * (4 * n + 4 * d + 2 * d + 4 + 2 * n + 4) + 8 * 256
    assert room <= rows + 2 * d * em.row_bytes(em.Q8_0, n), room  # (its parts, and room for a smaller batch's)


@pytest.mark.parametrize("kw,Ts", [
    (dict(d=2048, d_ff=1408, E=64, k=6, wtype=em.Q8_0, d_ff_shared=2816), range(1, 200)),
    (dict(d=512, d_ff=512, E=16, k=2, wtype=em.F32, d_ff_shared=2048), range(1, 1200, 7)),
])
def test_scratch_of_a_batch_serves_smaller_ones(kw, Ts):
    L = _desc(kw)
    sizes = [em.scratch_bytes(L, T) for T in Ts]
    assert sizes == sorted(sizes)
