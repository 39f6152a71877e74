"""BF16x3 GEMM without a given tile: sizes that only some of the tiles can run (run with -m gpu)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _pair(x):
    hi = x.to(torch.bfloat16)
    return hi, (x - hi.double()).to(torch.bfloat16)


def _rows(x, ld):
    """x (rows x K) with its rows ld elements apart, a little more than what the last row needs."""
    buf = torch.empty((x.shape[0] - 1) * ld + x.shape[1] + 8, dtype=torch.bfloat16, device="cuda")
    view = buf.as_strided(x.shape, (ld, 1))
    view.copy_(x)
    return buf


# rows 2^23 or 2^24 apart: the 256 or 128 rows of a wide tile span 4 GiB, more than its 32-bit
# offsets reach, where the estimate of time prefers that tile (in A, then in B)
@pytest.mark.parametrize("M,N,K,batch,lda,ldb", [(100, 16384, 1024, 8, 1 << 23, 1088),
                                                 (16384, 100, 1024, 8, 1088, 1 << 24)])
def test_bf16x3_falls_back_to_a_tile_that_fits(M, N, K, batch, lda, ldb):
    """Against the FP64 product within the bound of the split (see test_gpu_gemm_bf16), and the bits
    of the 64 x 64 tile."""
    from dftbaby_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    # one set of rows for all of the batch: the batches differ in their start along K
    A = torch.randn(M, K + 8 * batch, dtype=torch.float64, device="cuda", generator=gen)
    B = torch.randn(N, K + 8 * batch, dtype=torch.float64, device="cuda", generator=gen)
    ops = [_rows(x, ld) for x, ld in zip((*_pair(A), *_pair(B)), (lda, lda, ldb, ldb))]
    outs = []
    for tile in (0, 64):
        C = torch.full((batch, M, N), float("nan"), dtype=torch.float64, device="cuda")
        a = _lib.GemmArgs()
        a.A, a.A2, a.B, a.B2 = (x.data_ptr() for x in ops)
        a.C = C.data_ptr()
        a.lda, a.ldb, a.ldc, a.sA, a.sB, a.sC, a.cs2 = lda, ldb, N, 8, 8, M * N, 1
        a.M, a.N, a.K, a.batch, a.ksplit, a.kchunk = M, N, K, batch, 1, 0
        a.alpha, a.beta, a.b_trans, a.in_type, a.out_type, a.tile = 1.0, 0.0, 1, 2, 0, tile
        assert lib.dftb_gemm(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        outs.append(C)
    assert torch.equal(*outs)
    for b in range(batch):
        x, y = A[:, 8 * b:8 * b + K], B[:, 8 * b:8 * b + K]
        bound = (3 * 2.0 ** -16 + 3 * (K / 32 + 32) * 2.0 ** -24) * (x.abs() @ y.abs().T)
        assert bool(((outs[0][b] - x @ y.T).abs() <= bound).all())
