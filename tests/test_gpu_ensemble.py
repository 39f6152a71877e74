"""Persistent ensemble solver vs the oracle Davidson, molecule by molecule (run with -m gpu)."""
import numpy as np
import pytest

from conftest import ground_state
from oracle import tddftb_oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

MEMBERS = [("C8H10", 0.05, 1), ("C12H14", 0.05, 2), ("C8H10", 0.05, 3), ("C20H22", 0.05, 4), ("C12H14", 0.05, 5)]


def _oracle(gs, k, conv):
    r = O.solve_from_ground_state(gs, nstates=k, diag_conv=conv, diag_maxiter=100)
    return r["Omega"], r["XpY"]


@pytest.mark.parametrize("precision,conv,tol", [(0, 1e-8, 1e-9), (1, 1e-6, 1e-6)])
def test_ensemble_matches_oracle(precision, conv, tol):
    """FP64 to 1e-8 residual; FP32 exchange to the ensemble tolerance 1e-6 (the
    FP32 products put a floor near 1e-7 under the residual), energies within 1e-6 Ha."""
    from dftbaby_amd.ensemble import build_operators, solve_operators
    gss = [ground_state(n, 1, s, seed) for (n, s, seed) in MEMBERS]
    ops = build_operators(gss)
    k = 6
    res = solve_operators(ops, k, conv=conv, maxiter=100, precision=precision)
    for gs, w, xpy, it in zip(gss, res.Omega, res.XpY, res.iterations):
        ref_w, ref_xpy = _oracle(gs, k, 1e-8)
        assert np.abs(w - ref_w).max() < tol, (w, ref_w)
        for a, b in zip(xpy, ref_xpy):
            assert min(np.linalg.norm(a - b), np.linalg.norm(a + b)) < (1e-5 if precision == 0 else 1e-3)


def test_ensemble_reports_nonconvergence():
    from dftbaby_amd.ensemble import build_operators, solve_operators
    from dftbaby_amd.engine import ExcitedStatesNotConverged
    ops = build_operators([ground_state("C8H10", 1, 0.05, 1)])
    with pytest.raises(ExcitedStatesNotConverged):
        solve_operators(ops, 4, conv=1e-14, maxiter=1)


@pytest.mark.parametrize("copies", [1, 30, 100])
@pytest.mark.parametrize("precision,conv,tol", [(0, 1e-8, 1e-9), (1, 1e-6, 1e-6)])
def test_ensemble_batch_size_does_not_show(copies, precision, conv, tol):
    """A member's results are those of the oracle (energies within the bounds above) and the
    same bits alone and in a batch of any size."""
    from dftbaby_amd.ensemble import build_operators, solve_operators
    for name, n in (("C8H10", copies), ("C12H14", min(copies, 2))):
        gs = ground_state(name, 1, 0.05, 7)
        res = solve_operators(build_operators([gs] * n), 5, conv=conv, maxiter=100, precision=precision)
        ref_w, _ = _oracle(gs, 5, 1e-8)
        alone = solve_operators(build_operators([gs]), 5, conv=conv, maxiter=100, precision=precision)
        for w, xpy in zip(res.Omega, res.XpY):
            assert np.abs(w - ref_w).max() < tol, (w, ref_w)
            assert np.array_equal(w, alone.Omega[0]) and np.array_equal(xpy, alone.XpY[0])


@pytest.mark.parametrize("count", [150, 192, 300])
def test_large_ensembles(count):
    """Launches without helpers (150), with helpers that start as members end (192) and with more
    members than CUs (300): the bits of each member alone, and energies within the bound above."""
    from conftest import progress
    from dftbaby_amd.ensemble import build_operators, solve_operators
    kinds = [ground_state("C8H10", 1, 0.05, 7), ground_state("C12H14", 1, 0.05, 8), ground_state("C8H10", 1, 0.05, 9)]
    which = [1 if i % 50 == 7 else 2 * (i % 2) for i in range(count)]
    alone = [solve_operators(build_operators([gs]), 5, conv=1e-6, maxiter=100, precision=1) for gs in kinds]
    for gs, one in zip(kinds, alone):
        assert np.abs(one.Omega[0] - _oracle(gs, 5, 1e-8)[0]).max() < 1e-6
    ops = build_operators([kinds[i] for i in which])
    progress("%d operators" % count)
    res = solve_operators(ops, 5, conv=1e-6, maxiter=100, precision=1)
    for i, w, xpy, n in zip(which, res.Omega, res.XpY, res.iterations):
        assert n == alone[i].iterations[0]
        assert np.array_equal(w, alone[i].Omega[0]) and np.array_equal(xpy, alone[i].XpY[0])
