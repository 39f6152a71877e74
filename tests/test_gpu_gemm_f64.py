"""FP64 GEMM: every operand order at the edges of tiles and chunks, against torch in FP64."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _operand(rows, k, batch, trans, pad, off, gen):
    """batch x (rows x k), stored transposed when trans, with padded rows and an odd 8-byte offset."""
    r, c = (k, rows) if trans else (rows, k)
    buf = torch.full((off + batch * r * (c + pad),), float("nan"), dtype=torch.float64, device="cuda")
    x = buf[off:].view(batch, r, c + pad)
    x[:, :, :c] = torch.randn(batch, r, c, dtype=torch.float64, device="cuda", generator=gen)
    dense = x[:, :, :c].transpose(1, 2) if trans else x[:, :, :c]
    return x, dense.contiguous(), c + pad


def _gemm(A, lda, B, ldb, C, M, N, K, batch, ta, tb, alpha, beta, ksplit, kchunk, tile):
    from dftbaby_amd import _lib
    g = _lib.GemmArgs()
    g.A, g.B, g.C = A.data_ptr(), B.data_ptr(), C.data_ptr()
    g.lda, g.ldb, g.ldc = lda, ldb, N
    g.sA, g.sB, g.sC, g.cs2 = A.shape[1] * lda, B.shape[1] * ldb, M * N, 1
    g.M, g.N, g.K, g.batch = M, N, K, batch
    g.ksplit, g.kchunk, g.sCk = ksplit, kchunk, batch * M * N
    g.alpha, g.beta, g.a_trans, g.b_trans, g.tile = alpha, beta, ta, tb, tile
    _lib.call("dftb_gemm", ctypes.byref(g), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K,batch", [(1, 1, 1, 1), (16, 16, 16, 2), (17, 33, 15, 1), (80, 48, 97, 3), (39, 1025, 31, 1),
                                         (65, 79, 1000, 1), (255, 257, 63, 2), (513, 130, 201, 1), (3, 700, 5, 1)])
def test_gemm_f64_orders(M, N, K, batch, ta, tb):
    gen = torch.Generator(device="cuda").manual_seed(M * 1000 + N)
    A, Ad, lda = _operand(M, K, batch, ta, 3, 1, gen)
    # B(k, n): element (k, n) of a K x N operand, stored N x K when tb
    B, Bd, ldb = _operand(N, K, batch, not tb, 5, 1, gen)
    Bd = Bd.transpose(1, 2)
    # |error| <= (K + 2) eps sum |a b| element by element, for a chain of fused multiply-adds
    bound = (K + 2) * 2.3e-16 * (Ad.abs() @ Bd.abs())
    C0 = torch.randn(batch, M, N, dtype=torch.float64, device="cuda", generator=gen)
    C = C0.clone()
    _gemm(A, lda, B, ldb, C, M, N, K, batch, ta, tb, -0.5, 2.0, 1, K, 0)
    assert ((C - (2.0 * C0 - 0.5 * Ad @ Bd)).abs() <= bound + 1e-15 * (1 + C0.abs())).all()
    # one chain over ascending k, whatever the tile: the 128 x 128 tiling gives the same bits
    X, Y = torch.empty_like(C), torch.empty_like(C)
    _gemm(A, lda, B, ldb, X, M, N, K, batch, ta, tb, 1.0, 0.0, 1, K, 0)
    _gemm(A, lda, B, ldb, Y, M, N, K, batch, ta, tb, 1.0, 0.0, 1, K, 128)
    assert torch.equal(X, Y)
    if K > 32:   # slices of 32, the last one partial or empty
        ks = (K + 31) // 32 + 1
        P = torch.empty(ks, batch, M, N, dtype=torch.float64, device="cuda")
        _gemm(A, lda, B, ldb, P, M, N, K, batch, ta, tb, 1.0, 0.0, ks, 32, 0)
        assert ((P.sum(0) - Ad @ Bd).abs() <= 2 * bound).all()
