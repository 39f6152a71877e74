"""Sums over slices and the rank-dropping factor at their edges (run with -m gpu)."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _rnd(seed, *s):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)


@pytest.mark.parametrize("P,Q,n", [(1, 1, 1), (3, 2, 2048), (5, 7, 2048 * 31), (64, 3, 2048 * 32), (17, 40, 2048 * 33 + 5),
                                   (9, 9, 2048 * 64 + 1), (2, 70, 2048 * 75)])
def test_gram_slices(P, Q, n):
    """Below, at and above blocks of 32 slices, against torch: n roundings of the dot product."""
    from dftbaby_amd import _lib
    from dftbaby_amd.engine import Workspace, _p, _stream
    X, Y = _rnd(P, P, n), _rnd(Q + 100, Q, n)
    out = torch.full((P, Q + 3), 7.0, dtype=torch.float64, device="cuda")
    w, wn = Workspace(X.device).get(_lib.load().dftb_gram_workspace(P, Q, n))
    _lib.call("dftb_gram", _p(X), n, P, _p(Y), n, Q, n, _p(out), Q + 3, _p(w), wn, _stream())
    bound = n * 2.0 ** -52 * (X.abs() @ Y.abs().T)
    assert bool(((out[:, :Q] - X @ Y.T).abs() <= bound).all())
    assert bool((out[:, Q:] == 7.0).all())


@pytest.mark.parametrize("m", [2, 3, 17, 39, 52, 53, 70])
def test_orthonormalize_drops_dependent_rows(m):
    """Every third row a combination of two earlier ones (of the basis for the first): dropped and
    zeroed; the others orthonormal to the basis and each other (n roundings)."""
    from dftbaby_amd import _lib
    from dftbaby_amd.engine import Workspace, _p, _stream
    n, l = 4000, 5
    basis = torch.linalg.qr(_rnd(1, n, l))[0].T.contiguous()
    Q = _rnd(m, m, n)
    dep = [j for j in range(m) if j % 3 == 1]
    for j in dep:
        Q[j] = 2.0 * Q[j - 1] - 3.0 * (basis[2] if j == 1 else Q[j - 4])
    keep = torch.full((m,), -1, dtype=torch.int32, device="cuda")
    w, wn = Workspace(Q.device).get(_lib.load().dftb_orthonormalize_workspace(l, m, n))
    _lib.call("dftb_orthonormalize", _p(basis), l, _p(Q), m, n, 1e-8, _p(keep), _p(w), wn, _stream())
    ok = torch.ones(m, dtype=torch.bool, device="cuda")
    ok[dep] = False
    assert bool(((keep != 0) == ok).all())
    assert bool((Q[~ok] == 0.0).all())
    B = torch.cat([basis, Q[ok]])
    assert float((B @ B.T - torch.eye(len(B), dtype=torch.float64, device="cuda")).abs().max()) < n * 2.0 ** -52
