"""Direct-load products on 32 x 16 tiles (GPU): remainders of the tile in both
directions and of the k-step, every orientation, at shapes whose 32 x 16 tiles
fill rounds of the device better than 16 x 16 or 32 x 32 do.

Operands have NaN around them.  Tolerance as for the other tiles (relative
Frobenius against a float64 product): 4 sqrt(K) eps of the type, twice that for
complex, whose sums have twice the terms.
"""

import numpy as np
import pytest

from test_gpu_gemm_tiles import _operand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transA,transB", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("prec,field,M,N,K", [
    (0, 1, 600, 593, 47), (0, 1, 577, 608, 48), (1, 1, 600, 600, 65),
    (1, 0, 2400, 150, 100), (1, 0, 2369, 145, 31), (0, 1, 2259, 241, 801)])
def test_products(engine, transA, transB, prec, field, M, N, K):
    import torch
    rng = np.random.default_rng(M + N + K)
    dt = torch.float64 if prec == 0 else torch.float32
    npl = 1 + field
    ra, ca = (K, M) if transA else (M, K)
    rb, cb = (N, K) if transB else (K, N)
    A, a = _operand(rng, ra, ca, ca + 1, npl, dt, engine.device)
    B, b = _operand(rng, rb, cb, cb + 2, npl, dt, engine.device)
    C = torch.full((npl, M, N), float("nan"), dtype=dt, device=engine.device)
    engine.gemm(prec, field, A[:, 1:], B[:, 1:], C, M, N, K, transA=transA, transB=transB, lda=ca + 1, ldb=cb + 2,
                planeA=A[0].numel(), planeB=B[0].numel(), planeC=M * N)
    if field:
        a, b, c = torch.complex(a[0], a[1]), torch.complex(b[0], b[1]), torch.complex(C[0].double(), C[1].double())
    else:
        a, b, c = a[0], b[0], C[0].double()
    a = a.T.contiguous() if transA else a
    b = b.T.contiguous() if transB else b
    ref = a @ b
    tol = 4 * (1 + field) * np.sqrt(K) * float(torch.finfo(dt).eps)
    assert float((c - ref).norm() / ref.norm()) <= tol
