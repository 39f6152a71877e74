"""Transition charges in the reference layout at odd sizes and addresses (run with -m gpu)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# rows shorter than a line, lines and blocks crossed, aligned and not, one to eight stripes of 256
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("nat,nmu,nocc,nvirt", [(3, 4, 1, 2), (8, 4, 5, 9), (24, 4, 33, 32), (20, 4, 257, 255), (6, 9, 300, 17),
                                                (5, 16, 513, 31), (4, 4, 2047, 1025), (3, 4, 64, 2049)])
def test_trans_charges_odd_rows(nat, nmu, nocc, nvirt, shift):
    """Against the definition in FP64: 2 nmu + 1 roundings of the sum per entry, norb of S C."""
    from dftbaby_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(nocc)
    rnd = lambda *s: torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)
    off = np.full(nat, nmu, dtype=np.int32)
    off[::3] = 1
    norb = int(off.sum())
    Co, Cv, S = rnd(norb, nocc), rnd(norb, nvirt), rnd(norb, norb)
    S = S + S.T
    nb = lib.dftb_trans_charges_workspace(norb, nocc, nvirt, nat)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    q = [torch.full((nat * a * b + 2,), 7.0, dtype=torch.float64, device="cuda")
         for a, b in ((nocc, nocc), (nocc, nvirt), (nvirt, nvirt))]
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.dftb_trans_charges(p(Co), p(Cv), p(S), off.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), nat, norb, nocc,
                                nvirt, *[p(x[shift:]) for x in q], p(ws), nb,
                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    at = np.repeat(np.arange(nat), off)
    for x, (X, Z) in zip(q, ((Co, Co), (Co, Cv), (Cv, Cv))):
        n = nat * X.shape[1] * Z.shape[1]
        got = x[shift:shift + n].view(nat, X.shape[1], Z.shape[1])
        for A in range(nat):
            r = torch.as_tensor(np.flatnonzero(at == A), device="cuda")
            ref = 0.5 * (X[r].T @ (S @ Z)[r] + (S @ X)[r].T @ Z[r])
            mag = X[r].abs().T @ (S.abs() @ Z.abs())[r] + (S.abs() @ X.abs())[r].T @ Z[r].abs()
            assert bool(((got[A] - ref).abs() <= (norb + 2 * nmu + 4) * 2.0 ** -52 * mag).all())
        # nothing beside the block
        assert bool((x[:shift] == 7.0).all()) and bool((x[shift + n:] == 7.0).all())
