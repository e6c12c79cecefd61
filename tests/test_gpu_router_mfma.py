"""Router logits on the FP64 matrix cores (from 65536 token x expert pairs on): bit-identical to the reference's
eight FP64 chains (cpu_dot.h:12-21, the oracle), for ragged tokens, experts and columns (a step of 32 columns cut at
its 8-column groups, a tail of 4) on both tile widths, with operands that show any other order of additions
(magnitudes over 2^60, cancelling pairs), subnormals, signed zeros, infinities and NaN."""
import numpy as np
import pytest

import ember_moe as em
from gpu_util import same_bits
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,d,E", [(1024, 64, 64), (655, 516, 101), (2000, 72, 33), (515, 300, 128), (1311, 100, 100),
                                   (4097, 96, 32), (1100, 264, 129)])
@pytest.mark.parametrize("kind", ["normal", "spread", "cancel", "special"])
def test_router_mfma_bits(gpu, T, d, E, kind):
    import torch

    assert T * E >= 65536
    rng = np.random.default_rng(T + d)
    x = rng.standard_normal((T, d)).astype(np.float32)
    R = rng.standard_normal((E, d)).astype(np.float32)
    if kind == "spread":
        x *= np.exp2(rng.integers(-60, 60, (T, d))).astype(np.float32)
        R *= np.exp2(rng.integers(-60, 60, (E, d))).astype(np.float32)
    elif kind == "cancel":
        x[:, 8:16] = -x[:, 0:8]
        R[:, 8:16] = R[:, 0:8]
        x[::3, 1::2] *= np.float32(2.0**40)
    elif kind == "special":
        x[5::97, 3] = np.inf
        x[7::89, d - 1] = np.nan
        x[1::5, ::2] = np.float32(1e-42)
        x[2::7] = -0.0
        R[3::11, 2] = -np.inf
    xd, Rd = torch.from_numpy(x).cuda(), torch.from_numpy(R).cuda()
    lg = torch.empty((T, E), dtype=torch.float32, device="cuda")
    print(f"router mfma T={T} d={d} E={E} {kind}", flush=True)
    assert em.router_logits(xd, T, d, E, Rd, lg) == 0
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        want = O.router_logits(x, R)
    assert same_bits(lg.cpu().numpy(), want)
