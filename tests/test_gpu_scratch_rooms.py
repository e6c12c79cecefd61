"""Where a call keeps its F32 tile table and the parts of a Q8_0 or F32 shared expert's split down projection: a call
needs no more scratch for the parts (they take what y or h have to spare), and none more than the
allocation-free entry point's buffer for the table, and its path does not depend on that buffer's size. Numerics
against the oracle (utils.cpp:704-748): F32 1e-6 rel-L2 (the F32 tiles' bar), Q8_0 the FP16 tiles' 2e-3."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import rel_l2, run_oracle, same_bits
from test_gpu_short_tile_batches import _desc

LIMIT = 32 << 20
# one batch each whose table would pass the buffer (the batch before and after have theirs in a section, or no room)
TIGHT = [(dict(d=64, d_ff=64, E=8, k=4, wtype=em.F32), 6412),
         (dict(d=64, d_ff=64, E=8, k=4, wtype=em.F32, d_ff_shared=192), 5363)]


@pytest.mark.parametrize("kw,T", TIGHT)
def test_path_does_not_depend_on_the_no_allocation_buffer(kw, T):
    L = _desc(kw)
    assert em.scratch_bytes(L, T) == LIMIT
    assert {em.path(L, t) for t in (T - 1, T, T + 1, T + 200)} == {em.path(L, T - 2)}


@pytest.mark.parametrize("kw,Ts", [
    (dict(d=2048, d_ff=1408, E=64, k=6, wtype=em.Q8_0, d_ff_shared=2816), (13, 64, 100, 121)),
    (dict(d=512, d_ff=1024, E=16, k=2, wtype=em.F32, d_ff_shared=2048), (65, 100, 600)),
])
def test_shared_down_parts_take_no_scratch(kw, Ts):
    """Beside h, y, the converted activations and the tile table, the shared expert's rows add one y row each."""
    n, d = kw["d_ff_shared"], kw["d"]
    plain = _desc({k: v for k, v in kw.items() if k != "d_ff_shared"})
    half = 2 * n + 4 if kw["wtype"] == em.Q8_0 else 0
    for T in Ts:
        room = em.scratch_bytes(_desc(kw), T) - em.scratch_bytes(plain, T)
        assert room <= T * (4 * n + 4 * d + half + (2 * d + 4 if half else 0)) + 6 * 256 + 16 * T * kw["k"], T


def _run(dl, x, how):
    import torch

    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    out = torch.full_like(xd, float("nan"))
    if how == "noalloc":
        assert em.moe_ffn_noalloc(dl.desc, xd, x.shape[0], out) == 0
    else:
        need = em.scratch_bytes(dl.desc, x.shape[0])
        sc = torch.full((need,), 255, dtype=torch.uint8, device="cuda")  # (NaN wherever a part is read unwritten)
        if how == "timed":
            em.moe_ffn_timed(dl.desc, xd, x.shape[0], out, sc)
        else:
            assert em.moe_ffn(dl.desc, xd, x.shape[0], out, sc) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("kw,T", TIGHT + [
    (dict(d=36, d_ff=1024, E=48, k=1, wtype=em.F32), 0),                      # (K split 4 outside the window)
    (dict(d=512, d_ff=1024, E=16, k=2, wtype=em.F32, d_ff_shared=2048), 100)])  # parts in y, routed K split 2
def test_f32_rooms(gpu, kw, T):
    hl = em.make_host_layer(em.LayerSpec(seed=3, weight_std=0.1, **kw))
    dl = em.DeviceLayer.upload(hl)
    if not T:
        T = next(t for t in range(2500, 7000) if em.scratch_bytes(dl.desc, t) == LIMIT)
    x = em.make_input(hl.spec, T)
    print(f"f32 rooms {kw} T={T}", flush=True)
    y = _run(dl, x, "ffn")
    assert rel_l2(y, run_oracle(hl, x)) < 1e-6
    assert same_bits(y, _run(dl, x, "timed")) and same_bits(y, _run(dl, x, "noalloc"))


@pytest.mark.gpu
@pytest.mark.parametrize("kw,T", [
    (dict(d=512, d_ff=512, E=8, k=2, d_ff_shared=1024, wtype=em.F16, shared_type=em.Q8_0), 5),  # routed GEMV: 3 parts of y
    (dict(d=512, d_ff=512, E=8, k=2, d_ff_shared=1024), 40),    # routed tiles, unsplit
    (dict(d=256, d_ff=8192, E=4, k=1, d_ff_shared=1024), 30),   # routed K split 4: y is full, h behind the table
    (dict(d=1024, d_ff=64, E=4, k=1, d_ff_shared=2048), 9),     # fewer parts than the split asks for
])
def test_q8_rooms(gpu, monkeypatch, kw, T):
    hl = em.make_host_layer(em.LayerSpec(seed=4, **dict(dict(wtype=em.Q8_0), **kw)))
    dl = em.DeviceLayer.upload(hl)
    x = em.make_input(hl.spec, T)
    print(f"q8 rooms {kw} T={T}", flush=True)
    monkeypatch.setenv("EMBER_MOE_SHARED_PATH", "skinny")
    if T == 5:
        monkeypatch.setenv("EMBER_MOE_PATH", "gemv")
    assert em.path(dl.desc, T) & em.PATH_SHARED_MFMA
    y = _run(dl, x, "ffn")
    assert rel_l2(y, run_oracle(hl, x)) < 2e-3
    assert same_bits(y, _run(dl, x, "timed"))
    monkeypatch.setenv("EMBER_MOE_SHARED_PATH", "gemm")
    assert rel_l2(y, _run(dl, x, "ffn")) < 3e-6  # (unsplit: sqrt(K) 2^-24, K <= 2048)
