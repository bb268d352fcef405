"""Tridiagonalisation inside one workgroup (real orders up to 128, GPU): orders
at the edges of its 32-row groups and 64-column halves, zero sub-columns, and
the early stop against the complete reduction; the complex reduction at the
same orders.

Eigenpairs against the matrix itself, bounds of 10 n eps of its norm (the form
of LAPACK's own test ratios).
"""

import numpy as np
import pytest

from test_gpu_trd_resident import _check, _graded

pytestmark = pytest.mark.gpu

ORDERS = [2, 3, 4, 31, 32, 33, 34, 63, 64, 65, 66, 95, 96, 97, 126, 127, 128, 129]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", ORDERS)
@pytest.mark.parametrize("kind", ["graded", "dense", "blocks"])
def test_orders(engine, kind, n, cplx):
    import torch
    rng = np.random.default_rng(5 * n + cplx)
    if kind == "graded":
        A = _graded(rng, n, cplx)
    elif kind == "dense":
        A = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0)
        A = A + A.conj().T
    else:   # decoupled blocks and a diagonal part
        A = np.diag(np.arange(n) + 1.0).astype(complex if cplx else float)
        for at, size in ((0, n // 3), (n // 3 + 1, n // 4)):
            A[at:at + size, at:at + size] = _graded(rng, size, cplx) if size else 0.0
    A = torch.from_numpy(A).to(engine.device)
    if cplx:
        w, Z = engine.herm_eig(torch.stack([A.real, A.imag]).contiguous(), 1)
        Z = torch.complex(Z[0], Z[1])
    else:
        w, Z = engine.sym_eig(A, 1)
    _check(A, w, Z)


@pytest.mark.parametrize("field", [0, 1])
@pytest.mark.parametrize("m", [100, 128])
def test_early_stop(engine, field, m):
    """Rows and columns falling by 1e-20: the trailing block is below 2e-15 of
    the Gram matrix at the first check, so the reduction ends at column 96."""
    import torch
    rng = np.random.default_rng(m)
    n = m + 8
    r, c = 10.0 ** (-20.0 * np.arange(m) / m), 10.0 ** (-20.0 * np.arange(n) / n)
    Z = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if field else 0)
    M = r[:, None] * Z * c
    Md = torch.tensor(np.stack([M.real, M.imag]) if field else M[None], dtype=torch.float64, device=engine.device)
    out = {}
    try:
        for mode in (3, 1):
            engine.set_eigensolver(mode)
            engine.prof_enable(True)
            U, V, keep, disc, sv = engine.svd_split(field, Md, m, n, 1e-12, 0, 1, 0)
            torch.cuda.synchronize()
            trd_bytes = engine.prof_read_bytes()[4]
            engine.prof_enable(False)
            U, V = U.cpu().numpy(), V.cpu().numpy()
            out[mode] = (U[0] + 1j * U[1], V[0] + 1j * V[1]) if field else (U[0], V[0])
            out[mode] += (keep, disc, sv, trd_bytes)
    finally:
        engine.set_eigensolver(1)   # the default
    Uf, Vf, kf, df, sf, bf = out[3]
    Ue, Ve, ke, de, se, be = out[1]
    eps = 2.0 ** -52
    assert ke == kf
    assert abs(de - df) < 1e-14
    assert np.all(np.abs(se[:ke] - sf[:kf]) <= 1e-13 + 8 * eps / sf[:kf])
    assert np.linalg.norm(Uf @ Vf - Ue @ Ve) < (1e-12 + 100 * eps / sf[kf - 1]) * np.linalg.norm(Uf @ Vf)
    assert np.abs(Ue.conj().T @ Ue - np.eye(ke)).max() < 1e-12
    assert be < bf
