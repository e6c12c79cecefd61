"""Which kernels a layer call takes at the ends of the dispatch rules (ember_moe_path; no GPU): shapes at which a rule taken
from fewer shapes made calls slower than the kernels they took before it. The figures stand beside the rules."""
import pytest

import ember_moe as em
from test_gpu_short_tile_batches import _desc

KERNEL = em.PATH_GEMV | em.PATH_TILES64 | em.PATH_TILES256


def _kernel(kw, T):
    return em.path(_desc(kw), T) & KERNEL


F32 = dict(wtype=em.F32)


@pytest.mark.parametrize("kw,gemv,tiles", [
    (dict(F32, d=3072, d_ff=4096, E=16, k=4), 10, 12),
    (dict(F32, d=2048, d_ff=8192, E=16, k=2), 20, 24),
    (dict(F32, d=1024, d_ff=2816, E=8, k=2), 10, 12),
    (dict(F32, d=4096, d_ff=14336, E=8, k=2), 7, 8),
    (dict(F32, d=2048, d_ff=768, E=128, k=8), 20, 32),
    (dict(F32, d=1024, d_ff=2816, E=1, k=1), 18, 19),
    # with an F32 shared expert, both or neither
    (dict(F32, d=1024, d_ff=768, E=16, k=4, d_ff_shared=2048), 18, 19),
    (dict(F32, d=512, d_ff=1024, E=16, k=2, d_ff_shared=2048), 18, 19),
    (dict(F32, d=2048, d_ff=1408, E=64, k=6, d_ff_shared=2816), 18, 20),
    (dict(F32, d=2048, d_ff=768, E=128, k=2, d_ff_shared=1024), 64, 128),
])
def test_f32_gemv_and_tiles(kw, gemv, tiles):
    assert _kernel(kw, gemv) == em.PATH_GEMV
    assert _kernel(kw, tiles) == em.PATH_TILES64
    if "d_ff_shared" in kw:
        assert not em.path(_desc(kw), gemv) & em.PATH_SHARED_MFMA
        assert em.path(_desc(kw), tiles) & em.PATH_SHARED_MFMA


@pytest.mark.parametrize("wtype", [em.F16, em.BF16])
def test_one_half_expert_and_shared_lines(wtype):
    """A routed layer of one expert by its own blocks, not by the 800 rows of a shared expert beside routed launches."""
    def layer(pack=True, **kw):
        L = _desc(dict(kw, wtype=wtype))
        L.prefill_pack = 1 << 20 if pack and wtype == em.BF16 else None
        return L

    small, big = layer(d=1024, d_ff=2816, E=1, k=1), layer(d=4096, d_ff=14336, E=1, k=1)
    assert all(em.path(small, T) & KERNEL == em.PATH_TILES64 for T in (200, 801, 1024, 2816))
    assert em.path(small, 2817) & KERNEL == em.PATH_TILES256
    assert em.path(big, 512) & KERNEL == em.PATH_TILES64 and em.path(big, 513) & KERNEL == em.PATH_TILES256
    if wtype == em.BF16:  # without row exponents only the 64-token tiles have the split path
        assert em.path(layer(False, d=4096, d_ff=14336, E=1, k=1), 4000) & KERNEL == em.PATH_TILES64


@pytest.mark.gpu
@pytest.mark.parametrize("kw,rows,packed", [
    (dict(d=1792, d_ff=64, E=2, k=1, d_ff_shared=6400), 384, 704),     # 50 column tiles: 310 and 560 blocks
    (dict(d=256, d_ff=64, E=2, k=1, d_ff_shared=12288), 1600, 1600),   # one column tile of the down launch
])
def test_q8_shared_expert_line(gpu, monkeypatch, kw, rows, packed):
    """The largest batch whose Q8_0 shared expert takes the 64-token tiles: there the call has the bits of those forced,
    one row further the 256-token tiles' (the two differ: at these sizes the first split the down projection over
    K). Held to the FP16 tiles' 2e-3 against the oracle."""
    import numpy as np
    import torch

    from gpu_util import rel_l2, run_oracle, same_bits

    hl = em.make_host_layer(em.LayerSpec(seed=6, wtype=em.Q8_0, **kw))
    dl = em.DeviceLayer.upload(hl)
    pack = torch.empty(em.prefill_pack_bytes(dl.desc), dtype=torch.uint8, device="cuda")
    em.prefill_pack(dl.desc, pack)

    def run(x, path=None):
        monkeypatch.delenv("EMBER_MOE_SHARED_PATH", raising=False)
        if path:
            monkeypatch.setenv("EMBER_MOE_SHARED_PATH", path)
        out, _ = dl.forward(torch.from_numpy(np.ascontiguousarray(x)).cuda())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    for p, most in ((None, rows), (pack.data_ptr(), packed)):
        dl.desc.prefill_pack = p
        for T in (most, most + 1):
            x = em.make_input(hl.spec, T)
            print(f"q8 shared line {kw} T={T} pack={p is not None}", flush=True)
            y, y64, y256 = run(x), run(x, "skinny"), run(x, "gemm")
            assert not same_bits(y64, y256)
            assert same_bits(y, y64 if T == most else y256)
            if T == rows:
                assert rel_l2(y, run_oracle(hl, x)) < 2e-3
