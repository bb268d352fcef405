"""GEMM kernels at the edges of their tiles, splits and dispatch lines (GPU).

Each size sits next to a line of the dispatch (direct-load 16 x 16 or 32 x 32
tiles with one or four waves per tile, LDS 64 x 64 or 128 x 128 tiles) or of a
tile (a remainder of one, an inner dimension just off a multiple of 16, rows
shorter than a vector).  Operands lie in buffers whose row padding and
surroundings are NaN, so a value read from outside an operand shows.

Tolerance (relative Frobenius against a float64 product of the same inputs):
4 sqrt(K) eps of the type, the growth of K roundings of random sign.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REAL = [(1, 1, 1), (16, 16, 16), (17, 15, 17), (33, 31, 65), (129, 3, 45), (3, 129, 15),
        (400, 400, 63), (417, 449, 64), (449, 417, 400), (1100, 1000, 33), (1537, 1473, 129), (2049, 1025, 80),
        (2050, 2046, 31)]
COMPLEX = [(1, 1, 1), (17, 15, 17), (65, 33, 100), (450, 420, 47), (1030, 1025, 90), (1030, 1025, 801)]


def _operand(rng, rows, cols, pitch, planes, dtype, device):
    import torch
    a = rng.standard_normal((planes, rows, cols))
    buf = torch.full((planes, rows + 2, pitch), float("nan"), dtype=dtype, device=device)
    t = torch.from_numpy(a).to(device=device, dtype=dtype)
    buf[:, 1:-1, :cols] = t
    return buf, t.double()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("field,shape", [(0, s) for s in REAL] + [(1, s) for s in COMPLEX])
@pytest.mark.parametrize("pad", [0, 3])
def test_gemm_edges(engine, prec, ta, tb, field, shape, pad):
    import torch
    M, N, K = shape
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    dt = torch.float64 if prec == 0 else torch.float32
    npl = 1 + field
    ra, ca = (K, M) if ta else (M, K)
    rb, cb = (N, K) if tb else (K, N)
    A, a = _operand(rng, ra, ca, ca + pad, npl, dt, engine.device)
    B, b = _operand(rng, rb, cb, cb + pad, npl, dt, engine.device)
    C, c0 = _operand(rng, M, N, N + pad, npl, dt, engine.device)
    lda, ldb, ldc = ca + pad, cb + pad, N + pad
    engine.gemm(prec, field, A[0, 1:], B[0, 1:], C[0, 1:], M, N, K, transA=ta, transB=tb, conjA=bool(field and ta),
                conjB=bool(field and tb), alpha=0.7, beta=0.3, lda=lda, ldb=ldb, ldc=ldc, planeA=A[0].numel(),
                planeB=B[0].numel(), planeC=C[0].numel())
    torch.cuda.synchronize()

    def matrix(t, trans):
        m = torch.complex(t[0], t[1]) if field else t[0]
        return (m.mH if trans else m).cpu().numpy()

    ref = 0.7 * matrix(a, ta) @ matrix(b, tb) + 0.3 * matrix(c0, False)
    out = matrix(C[:, 1:-1, :N].double(), False)
    eps = np.finfo(np.float64 if prec == 0 else np.float32).eps
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err < 4 * np.sqrt(max(K, 16)) * eps, err
    rest = C.clone()
    rest[:, 1:-1, :N] = float("nan")
    assert bool(torch.isnan(rest).all())      # nothing written outside C
