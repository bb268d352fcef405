"""FP32 products on 96 x 96 tiles (GPU): remainders of the tile and of its 32-deep
inner tile, every orientation, batches and row pitches, at shapes whose 96 x 96
tiles fill one or two rounds of the device better than 64 or 128 do.

Reference in FP64; entrywise bound (K + 2) eps |A||B| of FP32 accumulation in
any order.
"""

import pytest

pytestmark = pytest.mark.gpu

EPS32 = 2.0 ** -24


@pytest.mark.parametrize("transA,transB", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("M,N,K,batch,padA,padB", [
    (1536, 1536, 1, 1, 0, 0), (1536, 1533, 31, 1, 0, 0), (1537 - 95, 1440, 32, 1, 1, 3), (1441, 1535, 33, 1, 0, 5),
    (1500, 1499, 63, 1, 7, 0), (857, 857, 65, 6, 0, 0), (864, 769, 130, 6, 2, 1)])
def test_products(engine, transA, transB, M, N, K, batch, padA, padB):
    import torch
    gen = torch.Generator().manual_seed(M + N + K)
    rows = lambda r, c, pad: torch.randn(batch, r, c + pad, generator=gen, dtype=torch.float32).to(engine.device)
    A = rows(*((K, M) if transA else (M, K)), padA)
    B = rows(*((N, K) if transB else (K, N)), padB)
    C = torch.full((batch, M, N), float("nan"), dtype=torch.float32, device=engine.device)
    engine.gemm(1, 0, A, B, C, M, N, K, lda=A.shape[2], ldb=B.shape[2], transA=transA, transB=transB,
                strideA=A[0].numel(), strideB=B[0].numel(), strideC=M * N, batch=batch)
    a = A[:, :, :(M if transA else K)].double()
    b = B[:, :, :(K if transB else N)].double()
    a = a.transpose(1, 2).contiguous() if transA else a.contiguous()
    b = b.transpose(1, 2).contiguous() if transB else b.contiguous()
    for i in range(batch):
        err = (C[i].double() - a[i] @ b[i]).abs()
        assert bool((err <= (K + 2) * EPS32 * (a[i].abs() @ b[i].abs())).all())
