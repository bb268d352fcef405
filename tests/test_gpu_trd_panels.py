"""The tridiagonalisation by panels, and the in-register reduction that gives up
and leaves its matrix to the panels (GPU).

Both are forced from the host: panels by dmrg_set_reduction, a give-up by a
wait of zero, with which a workgroup ends its attempt the first time a word of
its peers is missing (every workgroup exits normally).  The counts of
dmrg_reduction_counts show that the path meant really ran.  Eigenpairs as in
test_gpu_trd_resident.py, early-stopping splits against the complete reduction
as in test_gpu_eig.py, and splits whose order starts in panels and ends in
registers, or stops within the panels.
"""

import numpy as np
import pytest

from test_gpu_eig import test_split_early_stop_matches_full_reduction as early_stop_matches
from test_gpu_trd_resident import _check, _graded

pytestmark = pytest.mark.gpu


@pytest.fixture
def reduction(engine):
    yield engine.set_reduction
    engine.set_reduction()   # the default


def _counted(engine, fn):
    before = engine.reduction_counts()
    fn()
    return tuple(b - a for a, b in zip(before, engine.reduction_counts()))[:4]


def _eig(engine, n, cplx):
    import torch
    A = torch.from_numpy(_graded(np.random.default_rng(n), n, cplx)).to(engine.device)
    if cplx:
        w, Z = engine.herm_eig(torch.stack([A.real, A.imag]).contiguous(), 1)
        Z = torch.complex(Z[0], Z[1])
    else:
        w, Z = engine.sym_eig(A, 1)
    _check(A, w, Z)


@pytest.mark.parametrize("cplx,n", [(False, n) for n in (2, 3, 32, 33, 34, 64, 65, 128, 129, 300, 1025, 2400)] +
                         [(True, n) for n in (2, 3, 32, 33, 65, 129, 300, 1025)])
def test_panels(engine, reduction, n, cplx):
    reduction(in_registers=False)
    assert _counted(engine, lambda: _eig(engine, n, cplx)) == (0, 0, 0, 1)


@pytest.mark.parametrize("cplx,n", [(False, 300), (False, 1025), (False, 2400), (False, 3200),
                                    (True, 300), (True, 1025), (True, 1900)])
def test_given_up(engine, reduction, n, cplx):
    reduction(wait_ms=0.0)
    assert _counted(engine, lambda: _eig(engine, n, cplx)) == (0, 0, 1, 1)


@pytest.mark.parametrize("setting", [{"in_registers": False}, {"wait_ms": 0.0}], ids=["panels", "given up"])
@pytest.mark.parametrize("field,shape", [(0, (330, 340)), (0, (2400, 2560)), (1, (340, 330)), (1, (1400, 1300))])
def test_early_stop(engine, reduction, field, shape, setting):
    reduction(**setting)
    single, registers, given_up, panels = _counted(engine, lambda: early_stop_matches(engine, field, shape))
    assert (single, registers, panels) == (0, 0, 4)   # two splits in each of two modes
    assert given_up == (2 if "wait_ms" in setting else 0)   # the second and fourth come after a failure


def test_back_off(engine, reduction):
    """After a failure the next 1, 2, 4 ... reductions go to the panels at once,
    until a setting or a success forgets it."""
    import torch
    A = torch.from_numpy(_graded(np.random.default_rng(0), 150, False)).to(engine.device)
    reduction(wait_ms=0.0)
    tried = [_counted(engine, lambda: engine.sym_eig(A, 1))[2] for _ in range(12)]
    assert tried == [1, 0, 1, 0, 0, 1, 0, 0, 0, 0, 1, 0]
    reduction()
    assert _counted(engine, lambda: engine.sym_eig(A, 1)) == (0, 1, 0, 0)


@pytest.mark.parametrize("field,shape", [(0, (3300, 3200)), (0, (3400, 3500)), (1, (2000, 2100))])
def test_early_stop_from_panels_to_registers(engine, field, shape):
    """Complete and stopped alike: panels down to the order that fits, then one
    launch; the stop comes in the registers (at about 45% of the order)."""
    assert _counted(engine, lambda: early_stop_matches(engine, field, shape)) == (0, 4, 0, 4)


@pytest.mark.parametrize("field,m", [(0, 3400), (1, 2100)])
def test_early_stop_within_the_panels(engine, field, m):
    """Rows and columns falling by 1e-10 in the first 150: the reduction stops
    before the order that fits the registers."""
    import torch
    rng = np.random.default_rng(m)
    n = m + 8
    r, c = (10.0 ** (-10.0 * np.arange(k) / 150) for k in (m, n))
    Z = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if field else 0)
    M = r[:, None] * Z * c
    Md = torch.from_numpy(np.ascontiguousarray(np.stack([M.real, M.imag]) if field else M[None])).to(engine.device)
    out = []
    counts = _counted(engine, lambda: out.append(engine.svd_split(field, Md, m, n, 1e-12, 0, 1, 0)))
    assert counts == (0, 0, 0, 1)
    U, V, keep, disc, sv = out[0]
    Ms = torch.complex(Md[0], Md[1]) if field else Md[0]
    ref = np.linalg.svd(M[:400, :400], compute_uv=False)   # the rest is below 1e-26 of it
    eps = 2.0 ** -52
    assert np.all(np.abs(sv[:keep] - ref[:keep]) <= ref[0] * (1e-13 + 8 * eps * ref[0] / ref[:keep]))
    Uc, Vc = (torch.complex(x[0], x[1]) if field else x[0] for x in (U, V))
    miss = float(torch.linalg.matrix_norm(Uc @ Vc - Ms) / torch.linalg.matrix_norm(Ms))
    assert miss <= 1.01 * np.sqrt(disc) + 1e-10
    gram = Uc.conj().T.contiguous() @ Uc
    assert float((gram - torch.eye(keep, dtype=gram.dtype, device=gram.device)).abs().max()) < 1e-12
