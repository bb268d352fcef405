"""Krylov vector work at its edges (GPU): basis sizes across the batches of dot
products (1, 2, 4, 8, 16 and beyond, in both fields), vector lengths around the
workgroups' share and around the lengths where the number of workgroups
changes.

Lanczos energies after a fixed number of steps, the Ritz vector and the evolved
vector against
the same Lanczos recursion in plain torch FP64 on the same operator: energies
1e-12, evolved vectors 1e-11, Ritz vectors 1e-10 relative (rounding of a
recursion of <= 40 steps; a Ritz vector loses by the spectral gap).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _operator(engine, Dl, Dr, d, cplx, seed):
    """One-site H_eff with w = 1: y = L C R, Hermitian L and R, W = identity."""
    import torch
    rng = np.random.default_rng(seed)

    def herm(D):
        g = rng.standard_normal((D, D)) + (1j * rng.standard_normal((D, D)) if cplx else 0)
        return (g + g.conj().T) / np.sqrt(8.0 * D)

    def planes(a, pitch=None):
        p = np.stack([a.real, a.imag]) if cplx else np.asarray(a)[None]
        t = torch.from_numpy(np.ascontiguousarray(p)).to(engine.device)
        if pitch and pitch != t.shape[-1]:
            t = torch.nn.functional.pad(t, (0, pitch - t.shape[-1]))
        return t.contiguous()

    L, R = herm(Dl), herm(Dr)
    x = rng.standard_normal((Dl, d, Dr)) + (1j * rng.standard_normal((Dl, d, Dr)) if cplx else 0)
    Ld, Rd = planes(L[None], engine.env_pitch(Dl)), planes(R[None], engine.env_pitch(Dr))
    desc = engine.heff_desc(Ld, Rd, np.eye(d)[None, None, None], None, Dl, Dr, d, 0, int(cplx), 0)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to(engine.device) for a in (L, R, x)]
    return desc, planes(x).reshape(1 + int(cplx), -1), dev


def _lanczos(L, R, x, steps):
    import torch

    def apply(q):
        q = q.reshape(x.shape)
        return ((L @ q.reshape(x.shape[0], -1)).reshape(-1, x.shape[2]) @ R).reshape(-1)

    Q = [(x / torch.linalg.vector_norm(x)).reshape(-1)]
    al, be = [], []
    for k in range(steps):
        w = apply(Q[-1])
        al.append(float(torch.vdot(Q[-1], w).real))
        B = torch.stack(Q)
        for _ in range(2):
            w = w - (B.conj() @ w) @ B
        be.append(float(torch.linalg.vector_norm(w)))
        Q.append(w / be[-1])
    T = np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1)
    return torch.stack(Q[:-1]), T


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("Dl,Dr,d,steps", [(5, 3, 2, 3), (16, 16, 1, 5), (17, 15, 1, 9), (16, 17, 2, 17), (40, 31, 2, 33),
                                           (64, 64, 2, 40), (1024, 1023, 2, 4), (1024, 1025, 2, 4),
                                           (2048, 2047, 2, 3), (2048, 2049, 2, 3)])
def test_steps(engine, cplx, Dl, Dr, d, steps):
    import torch
    if cplx and Dl >= 1024:
        steps = 3
    desc, x, (L, R, x0) = _operator(engine, Dl, Dr, d, cplx, Dl + Dr)
    Q, T = _lanczos(L, R, x0, steps)
    ev, Z = np.linalg.eigh(T)
    y = x.clone()
    energy, iters = engine.lanczos(desc, y, steps, 1e-30)
    assert iters == steps
    assert abs(energy - ev[0]) < 1e-12 * max(1.0, abs(ev[0]))
    ref = torch.from_numpy(Z[:, 0].copy()).to(Q) @ Q
    got = torch.complex(y[0], y[1]) if cplx else y[0]
    sign = float(torch.sign(torch.vdot(ref, got).real))
    assert float(torch.linalg.vector_norm(sign * got - ref)) < 1e-10     # eigenvector: the gap's loss
    coeff = -0.3j if cplx else -0.3
    z = x.clone()
    engine.expm(desc, z, coeff, steps, 0.0, 0.0)
    col = (Z * np.exp(coeff * ev)) @ Z[0]
    ref = torch.linalg.vector_norm(x0) * (torch.from_numpy(col).to(Q) @ Q)
    got = torch.complex(z[0], z[1]) if cplx else z[0]
    assert float(torch.linalg.vector_norm(got - ref)) < 1e-12 * float(torch.linalg.vector_norm(ref)) * 10
