"""The dense LU of the Newton direct mode at the edges of its one-workgroup
form (LDS-resident up to 140 unknowns, 256 threads up to 64) and just beyond,
against numpy's LU: random matrices that need row exchanges, a zero leading
diagonal, rows of very different scale, and a singular matrix."""
import numpy as np
import pytest

import oracle
from ohmnivore_amd import _native as N
from ohmnivore_amd import solver

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return solver.HipBackend()


def dense_solve(be, d, b):
    n = d.shape[0]
    rows, cols = np.nonzero(d)
    a = oracle.from_triplet_arrays(n, n, rows, cols, d[rows, cols])
    x, _ = solver.newton_solve(be, a, b, linear_solver="dense", max_iterations=2, abs_tol=1e300)
    return x


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 100, 128, 139, 140, 141, 150])
@pytest.mark.parametrize("density", [1.0, 0.15])
def test_dense_lu_matches_numpy(be, n, density):
    rng = np.random.default_rng(n)
    d = rng.standard_normal((n, n)) * (rng.random((n, n)) < density)
    d += np.roll(np.eye(n), 1, axis=1) * 3.0      # nonsingular pattern off the diagonal
    d *= 10.0 ** rng.uniform(-3, 3, (n, 1))
    if n > 1:
        d[0, 0] = 0.0
    b = rng.standard_normal(n)
    x, ref = dense_solve(be, d, b), np.linalg.solve(d, b)
    # backward stable: a residual of order n eps |A| |x| per row
    assert np.all(np.abs(d @ x - b) <= 64 * n * 2.3e-16 * (np.abs(d) @ np.abs(ref) + np.abs(b)))
    # and no further from numpy's answer than the condition number explains
    assert np.abs(x - ref).max() <= 64 * n * 2.3e-16 * np.linalg.cond(d / np.abs(d).max(1)[:, None]) * np.abs(ref).max()


@pytest.mark.parametrize("n", [3, 64, 140, 141])
def test_dense_lu_singular(be, n):
    d = np.random.default_rng(n).standard_normal((n, n))
    d[:, n // 2] = 0.0
    with pytest.raises(N.OhmnivoreError, match="singular"):
        dense_solve(be, d, np.ones(n))
