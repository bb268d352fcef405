"""Divide and conquer on tridiagonal matrices (GPU): orders at block and level
boundaries, and the spectra that decide its deflation -- equal and clustered
eigenvalues, decoupled rows, tiny couplings, gradings, extreme scales.

The tridiagonal matrices go through sym_eig as dense matrices (their reduction
is trivial).  Residual, orthonormality and eigenvalues against numpy within
10 n eps of the matrix norm, LAPACK's own form of bound for these quantities.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _random(rng, n):
    return rng.standard_normal(n), rng.standard_normal(n - 1)


def _toeplitz(rng, n):
    return np.full(n, 2.0), np.full(n - 1, -1.0)


def _wilkinson(rng, n):
    return np.abs(np.arange(n) - (n - 1) / 2.0), np.ones(n - 1)


def _glued(rng, n):
    d, e = np.abs(np.arange(n) % 21 - 10.0), np.ones(n - 1)
    e[20::21] = 1e-9
    return d, e


def _graded(rng, n):
    d = np.exp(-36.0 * np.arange(n) / n) * (1 + 0.1 * rng.standard_normal(n))
    return d, 0.3 * np.sqrt(np.abs(d[1:] * d[:-1]))


def _decoupled(rng, n):
    d, e = rng.standard_normal(n), rng.standard_normal(n - 1)
    e[rng.random(n - 1) < 0.3] = 0.0
    return d, e


def _constant(rng, n):
    return np.full(n, 1.0), np.where(np.arange(n - 1) % 3 == 0, 1e-17, 1e-3)


def _multiple(rng, n):
    return np.round(rng.standard_normal(n)), 1e-15 * rng.standard_normal(n - 1)


def _diagonal(rng, n):
    return np.zeros(n), np.zeros(n - 1)


KINDS = [_random, _toeplitz, _wilkinson, _glued, _graded, _decoupled, _constant, _multiple, _diagonal]


def _check(engine, d, e, scale=1.0):
    import torch
    n = len(d)
    T = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    A = torch.from_numpy(T * scale).to(engine.device)
    w, Z = engine.sym_eig(A, 1)
    w, A = w / scale, torch.from_numpy(T).to(engine.device)
    bound = 10 * n * np.finfo(np.float64).eps
    nrm = max(float(torch.linalg.matrix_norm(A)), 1e-300)
    ZT = Z.T.contiguous()
    assert float(torch.linalg.matrix_norm(A @ ZT - ZT * w)) <= bound * nrm
    assert float(torch.linalg.matrix_norm(Z @ ZT - torch.eye(n, dtype=A.dtype, device=A.device))) <= bound * np.sqrt(n)
    assert np.abs(w.cpu().numpy() - np.linalg.eigvalsh(T)).max() <= bound * nrm


@pytest.mark.parametrize("kind", KINDS, ids=lambda k: k.__name__.strip("_"))
@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 64, 65, 129, 300, 1025])
def test_spectra(engine, kind, n):
    _check(engine, *kind(np.random.default_rng(n), n))


@pytest.mark.parametrize("scale", [1e-140, 1e-30, 1e140])
def test_scales(engine, scale):
    _check(engine, *_random(np.random.default_rng(1), 200), scale=scale)


@pytest.mark.parametrize("n", [2049, 4032, 4033])
def test_large(engine, n):
    """The largest order it takes, and the first beyond."""
    _check(engine, *_random(np.random.default_rng(n), n))
