"""Divide and conquer on matrices with a decoupled part far below the rest
(GPU): the squares of that part's entries, or of their ratios to its
eigenvalues, leave the range of doubles although the entries do not.

Orders of one block, two blocks and several levels; the small part first or
last, its coupling to the rest zero or as small as itself.  Residual,
orthonormality and eigenvalues within 10 n eps of the matrix norm, as in
test_gpu_tridiag_dc.py; the eigenvalues' reference is numpy's eigh, since its
values-only eigvalsh (LAPACK's square-root-free QL) is itself off by 1e-6 on
the couplings from 1e-300 to 1 below (1.00050083 for a largest eigenvalue of
1.0004998755617123 in 80 bits).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(engine, d, e):
    import torch
    n = len(d)
    T = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    A = torch.from_numpy(T).to(engine.device)
    w, Z = engine.sym_eig(A, 1)
    bound = 10 * n * np.finfo(np.float64).eps
    nrm = np.linalg.norm(T)
    ZT = Z.T.contiguous()
    assert float(torch.linalg.matrix_norm(A @ ZT - ZT * w)) <= bound * nrm
    assert float(torch.linalg.matrix_norm(Z @ ZT - torch.eye(n, dtype=A.dtype, device=A.device))) <= bound * np.sqrt(n)
    assert np.abs(w.cpu().numpy() - np.linalg.eigh(T)[0]).max() <= bound * nrm


@pytest.mark.parametrize("coupled", [False, True])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("scale", [1e-60, 1e-80, 1e-120, 1e-150, 1e-158, 1e-165, 1e-200, 1e-300])
@pytest.mark.parametrize("n", [8, 24, 100, 200])
def test_small_part(engine, n, scale, first, coupled):
    rng = np.random.default_rng(n)
    d, e = rng.standard_normal(n), rng.standard_normal(n - 1)
    h = n // 2
    if first:
        d[:h] *= scale
        e[:h - 1] *= scale
    else:
        d[h:] *= scale
        e[h:] *= scale
    e[h - 1] = scale if coupled else 0.0
    _check(engine, d, e)


@pytest.mark.parametrize("n", [12, 24, 200])
def test_falling_couplings(engine, n):
    """Equal diagonal entries and couplings from 1 down to 1e-300: every size
    of coupling is torn or merged somewhere."""
    _check(engine, np.ones(n), 10.0 ** (-300.0 * np.arange(n - 1) / n))
    _check(engine, np.zeros(n), 10.0 ** (-300.0 * np.arange(n - 1) / n)[::-1].copy())
