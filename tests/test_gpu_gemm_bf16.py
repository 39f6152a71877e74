"""BF16x3 GEMM: the tile chosen by size (run with -m gpu)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _pair(x):
    hi = x.to(torch.bfloat16)
    return hi.contiguous(), (x - hi.double()).to(torch.bfloat16).contiguous()


# one tile's corner, a ragged edge of each tile, the ranges of the three choices, K below and
# above one stage of 32
@pytest.mark.parametrize("M,N,K,batch", [(1, 1, 8, 1), (8, 130, 40, 2), (176, 176, 744, 3), (257, 129, 1000, 1),
                                         (264, 520, 136, 9), (1248, 1248, 1000, 2), (1248, 1250, 264, 9),
                                         (600, 256, 2200, 30)])
def test_bf16x3_tiles(M, N, K, batch):
    """Against the FP64 product: each operand is a pair with relative error 2^-16, the dropped
    low x low term is below 2^-16, and each of the 3 K / 32 MFMA steps rounds in FP32.  The tile
    does not show in the bits."""
    from dftbaby_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, dtype=torch.float64, device="cuda", generator=gen)
    B = torch.randn(batch, N, K, dtype=torch.float64, device="cuda", generator=gen)
    ah, al = _pair(A)
    bh, bl = _pair(B)
    outs = []
    for tile in (0, 64, 256, 512):
        C = torch.full((batch, M, N), float("nan"), dtype=torch.float64, device="cuda")
        a = _lib.GemmArgs()
        a.A, a.A2, a.B, a.B2, a.C = (x.data_ptr() for x in (ah, al, bh, bl, C))
        a.lda, a.ldb, a.ldc, a.sA, a.sB, a.sC, a.cs2 = K, K, N, 0, N * K, M * N, 1
        a.M, a.N, a.K, a.batch, a.ksplit, a.kchunk = M, N, K, batch, 1, 0
        a.alpha, a.beta, a.b_trans, a.in_type, a.out_type, a.tile = 1.0, 0.0, 1, 2, 0, tile
        rc = lib.dftb_gemm(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        outs.append(C)
    ref = torch.stack([A @ b.T for b in B])
    bound = (3 * 2.0 ** -16 + 3 * (K / 32 + 32) * 2.0 ** -24) * torch.stack([A.abs() @ b.abs().T for b in B])
    assert bool(((outs[0] - ref).abs() <= bound).all())
    for C in outs[1:]:
        assert torch.equal(C, outs[0])
