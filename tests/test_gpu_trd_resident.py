"""The register-resident tridiagonalisation at the edges of its variants (GPU):
orders at workgroup, column-chunk and row-block boundaries, the largest order
it takes and the first beyond (panels down to it), real and complex.

Eigenpairs against the matrix itself: residual, orthonormality and (against
numpy) eigenvalues within 10 n eps of the matrix norm, LAPACK's own form of
bound for these quantities.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REAL = [3, 14, 15, 16, 31, 255, 256, 257, 511, 513, 1024, 1025, 1537, 2049, 2561, 3072, 3073]
COMPLEX = [3, 6, 7, 8, 255, 257, 513, 1025, 1537, 1792, 1793]


def _check(A, w, Z):
    import torch
    n = A.shape[0]
    bound = 10 * n * np.finfo(np.float64).eps
    nrm = float(torch.linalg.matrix_norm(A))
    ZT = Z.transpose(-1, -2).contiguous()            # columns: eigenvectors
    res = float(torch.linalg.matrix_norm(A @ ZT - ZT * w)) / nrm
    eye = torch.eye(n, dtype=A.dtype, device=A.device)
    orth = float(torch.linalg.matrix_norm(Z.conj().contiguous() @ ZT - eye))
    assert res < bound, (n, res)
    assert orth < bound * np.sqrt(n), (n, orth)
    if n <= 600:
        ref = np.linalg.eigvalsh(A.cpu().numpy())
        assert np.abs(w.cpu().numpy() - ref).max() < bound * nrm


def _graded(rng, n, cplx):
    """Entries graded like a Gram matrix of a two-site tensor (eight decades)."""
    g = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0)
    s = np.exp(-np.linspace(0.0, 9.0, n))
    a = g * s[:, None] * s
    return a + a.conj().T


@pytest.mark.parametrize("n", REAL)
def test_real_orders(engine, n):
    import torch
    rng = np.random.default_rng(n)
    A = torch.from_numpy(_graded(rng, n, False)).to(engine.device)
    w, Z = engine.sym_eig(A, 1)
    _check(A, w, Z)


@pytest.mark.parametrize("n", COMPLEX)
def test_complex_orders(engine, n):
    import torch
    rng = np.random.default_rng(n)
    A = torch.from_numpy(_graded(rng, n, True)).to(engine.device)
    w, Z = engine.herm_eig(torch.stack([A.real, A.imag]).contiguous(), 1)
    _check(A, w, torch.complex(Z[0], Z[1]))


@pytest.mark.parametrize("cplx", [False, True])
def test_zero_subcolumns(engine, cplx):
    """Decoupled blocks and a diagonal part: zero sub-columns in mid reduction."""
    import torch
    rng = np.random.default_rng(3)
    n = 300
    A = np.zeros((n, n), dtype=complex if cplx else float)
    at = 0
    for size in (1, 40, 2, 97, 1, 60):
        A[at:at + size, at:at + size] = _graded(rng, size, cplx)
        at += size
    A[range(at, n), range(at, n)] = np.arange(n - at)
    A = torch.from_numpy(A).to(engine.device)
    if cplx:
        w, Z = engine.herm_eig(torch.stack([A.real, A.imag]).contiguous(), 1)
        Z = torch.complex(Z[0], Z[1])
    else:
        w, Z = engine.sym_eig(A, 1)
    _check(A, w, Z)
