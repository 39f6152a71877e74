"""Lowest eigenpairs at the sizes where the eigensolver changes its path."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("l,nev", [(1, 1), (2, 2), (3, 1), (63, 9), (64, 20), (65, 5), (127, 40), (136, 12), (137, 12),
                                   (138, 12), (139, 12), (200, 16), (641, 8), (1030, 6)])
def test_syevx_sizes(l, nev):
    from dftbaby_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(l)
    A = torch.randn(l, l, dtype=torch.float64, device="cuda", generator=g)
    A = torch.diag(torch.linspace(0.1, 1.0, l, dtype=torch.float64, device="cuda")) + 0.01 * (A + A.T)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    w = torch.empty(nev, dtype=torch.float64, device="cuda")
    V = torch.empty(l, nev, dtype=torch.float64, device="cuda")
    n = _lib.load().dftb_syevx_workspace(l, nev)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    _lib.call("dftb_syevx", p(A), l, l, nev, p(w), p(V), p(ws), n,
              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    ref = torch.linalg.eigvalsh(A)[:nev]
    # backward stable reduction: |dw| and residuals of a modest multiple of l eps |A|
    tol = 20 * l * 1.2e-16 * float(A.norm())
    assert float((w - ref).abs().max()) <= tol
    assert float((A @ V - V * w).norm(dim=0).max()) <= 10 * tol
    assert float((V.T @ V - torch.eye(nev, dtype=V.dtype, device="cuda")).abs().max()) <= 1e-10
