"""Host-side logic of the engine (no GPU needed)."""
import numpy as np


def test_initial_indices_match_stable_argsort():
    """The partial selection of the Davidson start (Solver.py:232-251 sorts all
    pairs) returns the same indices in the same order as a full stable argsort,
    including ties at the selection threshold."""
    from dftbaby_amd.engine import _initial_indices
    rng = np.random.default_rng(0)
    for _ in range(200):
        o, v = int(rng.integers(1, 30)), int(rng.integers(1, 30))
        vals = np.round(rng.random((o, v)) * rng.integers(1, 6), 1)
        lmax = int(rng.integers(1, o * v + 1))
        i, a = _initial_indices(vals, o, v, lmax)
        assert np.array_equal(i * v + a, np.argsort(vals.ravel(), kind="stable")[:lmax])


def test_zvector_solver_needs_the_gpu_operator():
    """Solver.Krylov_solver_Zvector takes the (A+B) operator object, not a Python
    callable (the products run on the GPU); the check precedes any device work."""
    import numpy as np
    import pytest
    from dftbaby_amd import Solver
    with pytest.raises(TypeError):
        Solver.Krylov_solver_Zvector(lambda x: x, np.ones((2, 3)), np.ones((2, 3, 1)), None)


def test_householder_steps_promise_no_separate_matrix():
    """syevx_block runs the Householder steps on W itself (X = W) for matrices beyond the LDS, so the
    function that takes both must not declare W free of aliases."""
    import os
    import re
    from conftest import ROOT
    src = open(os.path.join(ROOT, "dftbaby_amd", "csrc", "blockops.h")).read()
    assert re.search(r"hh_block_steps<\d+, \d+>\(W, [^;]*, W,", src)
    params = re.search(r"void hh_block_steps\(([^)]*)\)", src).group(1)
    assert re.search(r"double\s*\*\s*W\b", params) and not re.search(r"__restrict__\s+[XW]\b", params)


def test_tuned_tiles_hold_for_the_blocks_they_were_measured_on(monkeypatch):
    """Products of a few vectors take the library's tiles by size, not those tuned on a full block."""
    import torch
    from dftbaby_amd import engine
    tuned = {"tile_expand": 512, "tile_contract": 256, "nvec": 40}
    assert engine.tuned_tiles({}, 1) == (0, 0)
    assert engine.tuned_tiles(tuned) == engine.tuned_tiles(tuned, 20) == engine.tuned_tiles(tuned, 48) == (512, 256)
    assert engine.tuned_tiles(tuned, 1) == engine.tuned_tiles(tuned, 19) == (0, 0)

    # a product passes the size of its block on
    class Stop(Exception):
        pass

    def struct(self, *args):
        raise Stop(args[-1])

    op = engine.CasidaOperatorGPU.__new__(engine.CasidaOperatorGPU)
    op.N, op.device = 4, torch.device("cpu")
    monkeypatch.setattr(engine.CasidaOperatorGPU, "_struct", struct)
    for m in (1, 7):
        try:
            op.matvec(torch.zeros(m, 4, dtype=torch.float64))
        except Stop as e:
            assert e.args == (m,)


def test_tuning_measured_on_earlier_kernels_does_not_count(tmp_path):
    """A cache entry without the kernel generation in its key (128 x 128 FP64 tiles were the faster
    choice once) is not taken."""
    import json
    from types import SimpleNamespace
    from dftbaby_amd import autotune
    op = SimpleNamespace(nat=64, nocc=128, nvirt=128, exchange="ao", lc=1, tuning={}, prepare=lambda p: None)
    cache = tmp_path / "tuning.json"
    cache.write_text(json.dumps({"p0_ao_nat64_o128_v128": {"tile_expand": 128, "tile_contract": 128}}))
    assert autotune.autotune(op, 0, cache=str(cache)) == {} and not op.tuning
    cache.write_text(json.dumps({autotune._bucket(op, 0): {"tile_expand": 64}}))
    assert autotune.autotune(op, 0, cache=str(cache)) == {"tile_expand": 64}
