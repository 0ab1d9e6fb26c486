"""The resident BiCGSTAB solve (one launch for the whole solve, workgroups of
at most 512 rows meeting through memory) against the FP64 LU and against the
multi-kernel pipeline, which a check_interval of one's own selects, at the
edges of its dispatch: one workgroup and several, a last workgroup of few
rows, row tiles of 4, 6 and 8 entries, rows longer than a tile, no
preconditioner, FP32 refinement, warm starts and breakdowns."""
import time

import numpy as np
import pytest

import oracle
from ohmnivore_amd import _native as N
from ohmnivore_amd import solver

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return solver.HipBackend()


def system(n, per_row, n_dense, seed):
    """Diagonally dominant, about per_row entries a row (neighbours and far
    columns), the first n_dense rows coupled to every third unknown."""
    rng = np.random.default_rng(seed)
    rows, cols, vals = [], [], []
    for d in range(1, (per_row - 1) // 2 + 1):
        step = 1 if d == 1 else max(2, n // (d + 1))
        i = np.arange(n - step) if n > step else np.arange(0)
        for r, c in ((i, i + step), (i + step, i)):
            rows.append(r)
            cols.append(c)
            vals.append(-rng.uniform(0.1, 1.0, r.shape[0]))
    for k in range(n_dense):
        c = np.arange(k + 1, n, 3)
        rows.append(np.full(c.shape[0], k))
        cols.append(c)
        vals.append(-rng.uniform(0.0, 0.01, c.shape[0]))
    rows, cols, vals = (np.concatenate(v) for v in (rows, cols, vals))
    diag = np.ones(n)
    np.add.at(diag, rows, np.abs(vals))
    return oracle.from_triplet_arrays(n, n, np.concatenate([rows, np.arange(n)]),
                                      np.concatenate([cols, np.arange(n)]),
                                      np.concatenate([vals, 2.0 * diag]))


def solve(be, a, b, prec, x0=None, **kw):
    m = be.upload_matrix(a.values, a.col_indices, a.row_pointers, a.nrows)
    p = None if prec == N.PREC_NONE else be.preconditioner(m, prec)
    bb, xx = be.new_buffer(a.nrows), be.new_buffer(a.nrows)
    be.upload_vec(b, bb)
    if x0 is not None:
        be.upload_vec(x0, xx)
    st = be.bicgstab(m, bb, xx, p, solver.bicgstab_params(warm_start=x0 is not None, **kw))
    return be.download_vec(xx), st


# relative residual 1e-13 and a condition number below 10: errors below 1e-11
TOL = dict(tolerance=1e-13, max_iterations=2000)


@pytest.mark.parametrize("n", [65, 511, 512, 513, 1024, 1025, 5000])
@pytest.mark.parametrize("per_row,n_dense", [(3, 0), (5, 1), (7, 2)])
@pytest.mark.parametrize("prec", [N.PREC_NONE, N.PREC_JACOBI, N.PREC_ISAI],
                         ids=["none", "jacobi", "isai"])
def test_resident_matches_lu_and_pipeline(be, n, per_row, n_dense, prec):
    a = system(n, per_row, n_dense, seed=n + per_row)
    b = np.random.default_rng(n).standard_normal(n)
    ref = oracle.sparse_lu_solve(a, b)
    scale = np.abs(ref).max()
    x, st = solve(be, a, b, prec, **TOL)
    y, _ = solve(be, a, b, prec, check_interval=8, **TOL)
    assert st.iterations > 0 and st.residual_norm < 1e-12
    assert np.abs(x - ref).max() < 1e-11 * scale
    assert np.abs(y - ref).max() < 1e-11 * scale
    # the answer does not depend on when workgroups meet
    assert solve(be, a, b, prec, **TOL)[0].tobytes() == x.tobytes()


@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_ISAI], ids=["jacobi", "isai"])
def test_resident_is_one_launch_per_solve(be, prec):
    a = system(3000, 5, 0, seed=5)
    b = np.ones(3000)
    _, st = solve(be, a, b, prec, **TOL)
    _, pl = solve(be, a, b, prec, check_interval=8, **TOL)
    assert st.dispatches < 8 < pl.dispatches


@pytest.mark.parametrize("n", [300, 1600])
@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_ISAI], ids=["jacobi", "isai"])
def test_resident_fp32_refinement_and_warm_start(be, n, prec):
    a = system(n, 5, 1, seed=n)
    b = np.random.default_rng(n).standard_normal(n)
    ref = oracle.sparse_lu_solve(a, b)
    x, _ = solve(be, a, b, prec, precision="fp32_ir", tolerance=1e-12, max_iterations=2000)
    assert np.abs(x - ref).max() < 1e-10 * np.abs(ref).max()
    y, st = solve(be, a, b, prec, x0=ref + 1e-6, **TOL)
    assert np.abs(y - ref).max() < 1e-11 * np.abs(ref).max()
    z, st0 = solve(be, a, b, prec, x0=y, tolerance=1e-9)
    assert st0.iterations == 0 and z.tobytes() == y.tobytes()
    assert st.iterations > 0


def test_resident_stops(be):
    """The iteration cap, a zero right-hand side and an unreachable one end as
    in the pipeline."""
    a = system(700, 5, 0, seed=1)
    b = np.ones(700)
    for kw in (dict(check_interval=8), {}):
        with pytest.raises(N.OhmnivoreError, match="did not converge within 2 iterations"):
            solve(be, a, b, N.PREC_JACOBI, tolerance=1e-14, max_iterations=2, **kw)
        with pytest.raises(N.OhmnivoreError, match="NaN/Inf|breakdown"):
            solve(be, a, np.where(np.arange(700) == 690, np.inf, b), N.PREC_JACOBI, **kw)
    x, st = solve(be, a, np.zeros(700), N.PREC_JACOBI)
    assert not x.any() and st.iterations == 0


def mesh(rows, cols, seed, supply=0):
    """A rows x cols five-point mesh of random conductances to neighbours and
    ground; with supply set the last unknown joins that many of the nodes."""
    rng = np.random.default_rng(seed)
    n = rows * cols
    idx = np.arange(n).reshape(rows, cols)
    pairs = [(idx[:, :-1].ravel(), idx[:, 1:].ravel()), (idx[:-1].ravel(), idx[1:].ravel())]
    if supply:
        at = rng.choice(n, supply, replace=False)
        pairs.append((np.full(supply, n), at))
        n += 1
    r, c, v = [], [], []
    for p, q in pairs:
        g = rng.uniform(0.5, 1.5, p.shape[0])
        r += [p, q]
        c += [q, p]
        v += [-g, -g]
    r, c, v = (np.concatenate(k) for k in (r, c, v))
    diag = rng.uniform(0.5, 1.5, n)
    np.add.at(diag, r, -v)
    return oracle.from_triplet_arrays(n, n, np.concatenate([r, np.arange(n)]),
                                      np.concatenate([c, np.arange(n)]),
                                      np.concatenate([v, diag]))


# The workgroups' halo under ISAI: formed by their spare threads (narrow
# meshes), fetched only (wide ones), with a row too long for a thread, and with
# a preconditioner of another pattern, whose halo finds no threads. The
# condition number is below 20 and the residual below 1e-12: errors below 1e-10.
@pytest.mark.parametrize("rows,cols,supply", [(33, 16, 0), (61, 47, 0), (61, 47, 20),
                                              (90, 70, 600), (70, 130, 5), (12, 700, 0)])
@pytest.mark.parametrize("precision", ["fp64", "fp32_ir"])
def test_resident_halo(be, rows, cols, supply, precision):
    a = mesh(rows, cols, seed=rows, supply=supply)
    b = np.random.default_rng(cols).standard_normal(a.nrows)
    ref = oracle.sparse_lu_solve(a, b)
    x, st = solve(be, a, b, N.PREC_ISAI, precision=precision, **TOL)
    assert st.residual_norm < 1e-12
    assert np.abs(x - ref).max() < 1e-10 * np.abs(ref).max()
    y, _ = solve(be, a, b, N.PREC_ISAI, precision=precision, **TOL)
    assert y.tobytes() == x.tobytes()


def test_resident_halo_of_another_pattern(be):
    a, other = mesh(61, 47, seed=1), system(61 * 47, 7, 0, seed=2)
    b = np.random.default_rng(3).standard_normal(a.nrows)
    for m, q in ((a, other), (other, a)):
        dm = be.upload_matrix(m.values, m.col_indices, m.row_pointers, m.nrows)
        dq = be.upload_matrix(q.values, q.col_indices, q.row_pointers, q.nrows)
        p = be.preconditioner(dq, N.PREC_ISAI)
        bb, xx = be.new_buffer(m.nrows), be.new_buffer(m.nrows)
        be.upload_vec(b, bb)
        st = be.bicgstab(dm, bb, xx, p, solver.bicgstab_params(**TOL))
        ref = oracle.sparse_lu_solve(m, b)
        assert st.residual_norm < 1e-12
        assert np.abs(be.download_vec(xx) - ref).max() < 1e-10 * np.abs(ref).max()


# A matrix of at most 64 KiB is one allocation and one copy (here up to about
# 1,480 rows), a larger one an allocation an array; either is tuned and solved.
@pytest.mark.parametrize("n", [1, 2, 41, 1400, 1600])
@pytest.mark.parametrize("prec", [N.PREC_NONE, N.PREC_JACOBI, N.PREC_ISAI],
                         ids=["none", "jacobi", "isai"])
def test_one_shot_solve(be, n, prec):
    a = system(n, 3, 0, seed=n)
    b = np.random.default_rng(n).standard_normal(n)
    ref = oracle.sparse_lu_solve(a, b)
    s = solver.GpuSolver(be, precond=prec, params=solver.bicgstab_params(**TOL))
    assert np.abs(s.solve_real(a, b) - ref).max() < 1e-11 * np.abs(ref).max()
    m = be.upload_matrix(a.values, a.col_indices, a.row_pointers, n)
    m.autotune()
    x, y = be.new_buffer(n), be.new_buffer(n)
    be.upload_vec(b, x)
    be.spmv(m, x, y)
    assert np.allclose(be.download_vec(y), oracle.spmv(a, b), rtol=1e-13, atol=1e-13)


def shuffled(a, seed):
    """a with its unknowns numbered in random order."""
    perm = np.random.default_rng(seed).permutation(a.nrows)
    r = np.repeat(np.arange(a.nrows), np.diff(a.row_pointers.astype(np.int64)))
    return oracle.from_triplet_arrays(a.nrows, a.nrows, perm[r], perm[a.col_indices], a.values)


@pytest.mark.parametrize("make,level", [(lambda: system(3000, 3, 0, seed=1), 1),
                                        (lambda: mesh(60, 50, seed=2), 0)], ids=["ladder", "mesh"])
def test_resident_isai_of_unordered_numbering(be, make, level):
    """Node numbers in random order: a workgroup's rows of M_L have more
    foreign columns (1,035 and 1,268) than its halo holds (768), so every row
    reads its own. Condition and residual as in test_resident_halo."""
    a = shuffled(make(), seed=1)
    b = np.random.default_rng(a.nrows).standard_normal(a.nrows)
    ref = oracle.sparse_lu_solve(a, b)
    m = be.upload_matrix(a.values, a.col_indices, a.row_pointers, a.nrows)
    p = be.preconditioner(m, N.PREC_ISAI, level)
    bb, out = be.new_buffer(a.nrows), []
    be.upload_vec(b, bb)
    for _ in range(2):
        xx = be.new_buffer(a.nrows)
        st = be.bicgstab(m, bb, xx, p, solver.bicgstab_params(**TOL))
        assert st.dispatches < 8 and st.residual_norm < 1e-12
        out.append(be.download_vec(xx))
    assert np.abs(out[0] - ref).max() < 1e-10 * np.abs(ref).max()
    assert out[0].tobytes() == out[1].tobytes()


@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_ISAI], ids=["jacobi", "isai"])
def test_large_unordered_systems_take_the_pipeline(be, prec):
    """Beyond a few thousand rows a matrix in random order is the pipeline's in
    64 bits; in row order, or in 32 bits, the resident solve's."""
    a = mesh(100, 90, seed=4) if prec == N.PREC_JACOBI else system(9000, 3, 0, seed=4)
    b = np.random.default_rng(5).standard_normal(a.nrows)
    for q, resident in ((a, True), (shuffled(a, 6), False)):
        ref = oracle.sparse_lu_solve(q, b)
        x, st = solve(be, q, b, prec, **TOL)
        assert np.abs(x - ref).max() < 1e-10 * np.abs(ref).max()
        assert (st.dispatches < 8) == resident
        y, st = solve(be, q, b, prec, precision="fp32_ir", **TOL)
        assert np.abs(y - ref).max() < 1e-10 * np.abs(ref).max()
        assert st.dispatches < 40


@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_ISAI], ids=["jacobi", "isai"])
def test_more_than_two_long_rows_take_the_pipeline(be, prec):
    """Rows longer than a tile are summed one after the other by their whole
    workgroup: two of them stay in the resident solve, three do not."""
    b = np.random.default_rng(8).standard_normal(2000)
    for n_long, resident in ((2, True), (3, False)):
        a = system(2000, 3, n_long, seed=n_long)
        ref = oracle.sparse_lu_solve(a, b)
        x, st = solve(be, a, b, prec, **TOL)
        assert np.abs(x - ref).max() < 1e-11 * np.abs(ref).max()
        assert (st.dispatches < 8) == resident


@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_ISAI], ids=["jacobi", "isai"])
def test_resident_solve_that_gives_up(be, prec, monkeypatch):
    """One workgroup stays away: the others give the solve up when their first
    wait has lasted 0.2 s, and the pipeline goes on from the start it left, to the
    pipeline's own answer; the next solves leave the resident form out for a
    second. Nothing is written by the solve that gave up: the warm start is
    still there."""
    n = 3000
    a = system(n, 5, 0, seed=5)
    b = np.random.default_rng(7).standard_normal(n)
    ref = oracle.sparse_lu_solve(a, b)
    x0 = ref + 1e-3 * np.random.default_rng(8).standard_normal(n)
    pipe, sp = solve(be, a, b, prec, x0=x0, check_interval=8, **TOL)
    monkeypatch.setenv("OHM_RESIDENT_ABSENT", "1")
    try:
        x, st = solve(be, a, b, prec, x0=x0, **TOL)
        assert st.dispatches > 8 and st.iterations == sp.iterations
        assert x.tobytes() == pipe.tobytes()
        monkeypatch.delenv("OHM_RESIDENT_ABSENT")
        _, later = solve(be, a, b, prec, x0=x0, **TOL)
        assert later.dispatches > 8  # not tried
    finally:
        time.sleep(1.05)
    _, again = solve(be, a, b, prec, x0=x0, **TOL)
    assert again.dispatches < 8
