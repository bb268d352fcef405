"""MPO operators around the sizes at which their upload changes form (GPU):
kernel-argument blobs of 1 and 3 KB, the staged copy beyond, and operators too
dense for compressed rows.

The H_eff apply against a float64 einsum of the same inputs; FP64 1e-12
relative, FP32 2e-6 (as the other H_eff parity tests), back to back with a
second operator so that an upload overtaken by the next one would show.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mpo(rng, w, d, terms):
    """Automaton-like W[w, w, d, d]: identities in the corners, `terms` random
    local operators in the first row and last column, nothing else."""
    W = np.zeros((w, w, d, d))
    W[0, 0] = W[-1, -1] = np.eye(d)
    for k in range(1, w - 1):
        for row, col in ((0, k), (k, w - 1)):
            for _ in range(terms):
                W[row, col, rng.integers(d), rng.integers(d)] = rng.standard_normal()
    return W


# (w, d, terms): compressed operators of about 0.5, 1, 2.5, 3 and 6 KB, and a dense one
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("w,d,terms", [(3, 2, 2), (5, 2, 2), (7, 3, 2), (8, 3, 3), (8, 4, 4), (3, 2, 400)])
def test_apply(engine, prec, w, d, terms):
    import torch
    rng = np.random.default_rng(100 * w + terms)
    Dl, Dr = 19, 22
    envt = engine.env_dtype(prec)
    jobs = []
    for _ in range(2):
        W1, W2 = (rng.standard_normal((w, w, d, d)) if terms > 100 else _mpo(rng, w, d, terms) for _ in range(2))
        L, R = (torch.from_numpy(rng.standard_normal((w, D, D))).to(engine.device, envt) for D in (Dl, Dr))
        x = torch.from_numpy(rng.standard_normal((Dl, d, d, Dr))).to(engine.device)
        desc = engine.heff_desc(L[None].contiguous(), R[None].contiguous(), W1[None], W2[None], Dl, Dr, d, d, 0, prec)
        jobs.append((desc, L, R, W1, W2, x, engine.empty((1, x.numel()))))
    for desc, _, _, _, _, x, y in jobs:
        engine.heff_apply(desc, x, y)
    torch.cuda.synchronize()
    for _, L, R, W1, W2, x, y in jobs:
        t = np.einsum("lac,cstd->lastd", L.double().cpu().numpy(), x.cpu().numpy())
        t = np.einsum("lmps,lastd->maptd", W1, t)
        t = np.einsum("mrqt,maptd->rapqd", W2, t)
        ref = np.einsum("rapqd,rde->apqe", t, R.double().cpu().numpy())
        err = np.linalg.norm(y.cpu().numpy().reshape(ref.shape) - ref) / np.linalg.norm(ref)
        assert err < (1e-12 if prec == 0 else 2e-6), err
