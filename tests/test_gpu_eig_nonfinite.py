"""Eigenproblems that hold NaN or infinity (GPU): the default eigensolver and
the splits built on it raise, also right after a finite call of the same order
(whose values the workspace still holds), and the next finite call returns what
it returned before.

Orders on each side of the divide and conquer's block (12), of the reductions
(128 / 129 real) and with several levels of merges; the bad entry on the
diagonal and in the corner that the reduction sees first.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _planes(engine, a):
    import torch
    p = np.stack([a.real, a.imag]) if np.iscomplexobj(a) else a[None]
    return torch.from_numpy(np.ascontiguousarray(p)).to(engine.device)


def _gauss(rng, shape, cplx):
    return rng.standard_normal(shape) + (1j * rng.standard_normal(shape) if cplx else 0)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [2, 8, 12, 13, 24, 100, 128, 129, 300, 1025])
def test_eigenpairs(engine, n, cplx, bad):
    import torch
    A = _gauss(np.random.default_rng(n), (n, n), cplx)
    A = A + A.conj().T
    eig = engine.herm_eig if cplx else (lambda a, mode: engine.sym_eig(a[0], mode))
    w, Z = eig(_planes(engine, A), 1)
    for r, c in ((n // 2, n // 2), (n - 1, 0)):
        B = A.copy()
        B[r, c] = B[c, r] = bad
        with pytest.raises(RuntimeError):
            eig(_planes(engine, B), 1)
        w2, Z2 = eig(_planes(engine, A), 1)
        assert torch.equal(w, w2) and torch.equal(Z, Z2)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("m,n", [(40, 36), (130, 120), (300, 420)])
def test_split(engine, m, n, cplx, bad):
    import torch
    rng = np.random.default_rng(m)
    s = np.exp(-9.0 * np.arange(m) / m)
    M = _gauss(rng, (m, n), cplx) * s[:, None]
    Md = _planes(engine, M)
    U, V, keep, disc, _ = engine.svd_split(int(cplx), Md, m, n, 1e-12, 0, 1, 0)
    B = M.copy()
    B[m // 2, n // 3] = bad
    with pytest.raises(RuntimeError):
        engine.svd_split(int(cplx), _planes(engine, B), m, n, 1e-12, 0, 1, 0)
    U2, V2, keep2, disc2, _ = engine.svd_split(int(cplx), Md, m, n, 1e-12, 0, 1, 0)
    assert keep == keep2 and disc == disc2 and torch.equal(U, U2) and torch.equal(V, V2)
