"""Blocked back-transformation: T factors of the reflector blocks

Orders at which the last block of reflectors (128 real, 64 complex) holds one
row, a 16-row leaf less or more by one, or a join level only partly, and inner
dimensions just below and above the lengths that are split.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


@pytest.fixture(scope="module")
def engine():
    from dmrgpy_amd.engine import get_engine
    return get_engine(0)


@pytest.mark.parametrize("cx,n", [(False, n) for n in (16, 17, 18, 34, 81, 130, 146, 194, 257, 258, 386)]
                         + [(True, n) for n in (16, 17, 18, 34, 50, 66, 82, 129, 130, 258)])
def test_eigenvectors(engine, cx, n):
    import torch
    rng = np.random.default_rng(11 * n + cx)
    A = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cx else 0.0)
    A = A + A.conj().T
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=engine.device)
    if cx:
        w, Z = engine.herm_eig(dev(np.stack([A.real, A.imag])), 1)
        Z = Z.cpu().numpy()
        Z = Z[0] + 1j * Z[1]
    else:
        w, Z = engine.sym_eig(dev(A), 1)
        Z = Z.cpu().numpy()
    w = w.cpu().numpy()
    # backward stable: residual and departure from orthonormality a small
    # multiple of n eps in norm (entrywise well inside it)
    tol = 20 * n * EPS
    assert np.abs(Z.conj() @ Z.T - np.eye(n)).max() <= tol
    assert np.abs(A @ Z.T - Z.T * w).max() <= tol * np.linalg.norm(A, 2)
