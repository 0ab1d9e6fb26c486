"""Batched solves on resident workgroups (one launch per group of systems)
against the LU of every system and against the batch engine's own kernels,
which a check_interval of one's own selects: real and complex, one workgroup
per system and several, uneven sizes, one and two groups, rows longer than a
tile, no preconditioner."""
import threading
import time

import numpy as np
import pytest

import oracle
from ohmnivore_amd import _native as N
from ohmnivore_amd import circuit as ir
from ohmnivore_amd import solver
from tests.test_gpu_resident import system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return solver.HipBackend()


def lu(a, c, sigma, b):
    m = ir.CsrMatrix(a.nrows, a.ncols, a.values + sigma * c, a.col_indices, a.row_pointers)
    if not np.iscomplexobj(m.values):
        return oracle.sparse_lu_solve(m, b)
    n = m.nrows  # the complex system as a real one of twice the size
    rows = np.repeat(np.arange(n), np.diff(m.row_pointers.astype(np.int64)))
    cols, re, im = m.col_indices.astype(np.int64), m.values.real, m.values.imag
    big = oracle.from_triplet_arrays(
        2 * n, 2 * n, np.concatenate([rows, rows, rows + n, rows + n]),
        np.concatenate([cols, cols + n, cols, cols + n]), np.concatenate([re, -im, im, re]))
    x = oracle.sparse_lu_solve(big, np.concatenate([b.real, b.imag]))
    return x[:n] + 1j * x[n:]


@pytest.mark.parametrize("complex_", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("sizes,per_row,n_dense", [
    ([65, 300, 512], 3, 0),            # a workgroup each
    ([513, 40, 1300, 1], 5, 1),        # several, and a system of one row
    ([640, 641, 1025], 7, 2),
    ([1600] * 60, 3, 0),               # two groups at 512 rows a workgroup
    ([33] * 300, 3, 0)],               # more systems than compute units
    ids=["single", "uneven", "wide", "groups", "many"])
@pytest.mark.parametrize("prec", [N.PREC_JACOBI, N.PREC_NONE], ids=["jacobi", "none"])
def test_batch_resident_matches_lu(be, complex_, sizes, per_row, n_dense, prec):
    rng = np.random.default_rng(len(sizes) + per_row)
    mats = {n: system(n, per_row, n_dense, seed=n) if n > 1 else
            oracle.from_triplet_arrays(1, 1, np.array([0]), np.array([0]), np.array([2.0]))
            for n in set(sizes)}
    caps = {n: np.abs(m.values) * rng.uniform(0.1, 0.2, m.values.shape[0]) *
            (np.repeat(np.arange(n), np.diff(m.row_pointers.astype(np.int64))) ==
             m.col_indices) for n, m in mats.items()}
    systems, rhs = [], []
    for k, n in enumerate(sizes):
        m = mats[n]
        sigma = (1j * (1 + k % 7)) if complex_ else 0.5 * (k % 5)
        systems.append((m.row_pointers, m.col_indices, m.values, caps[n], sigma))
        b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if complex_ else 0)
        rhs.append(b)
    bt = solver.Batch(be, systems, complex_)
    prm = dict(tolerance=1e-13, max_iterations=2000)
    x = bt.solve(np.concatenate(rhs), params=solver.bicgstab_params(**prm), precond=prec)
    its = [r.iterations for r in bt.last_results]
    y = bt.solve(np.concatenate(rhs), params=solver.bicgstab_params(check_interval=8, **prm),
                 precond=prec)
    assert min(its) >= 1
    again = bt.solve(np.concatenate(rhs), params=solver.bicgstab_params(**prm), precond=prec)
    assert again.tobytes() == x.tobytes()
    for k in list(range(len(sizes)))[:8] + [len(sizes) - 1]:
        m = mats[sizes[k]]
        ref = lu(m, caps[sizes[k]], systems[k][4], rhs[k])
        scale = np.abs(ref).max()
        # relative residual 1e-13, condition below 10 (row scale up to 7)
        assert np.abs(bt.split(x)[k] - ref).max() < 1e-11 * scale
        assert np.abs(bt.split(y)[k] - ref).max() < 1e-11 * scale


def test_batch_resident_one_system_fails_alone(be):
    """A system whose right-hand side is not finite ends by itself; the
    iteration cap is per system."""
    m = system(700, 5, 0, seed=3)
    bt = solver.Batch(be, [(m.row_pointers, m.col_indices, m.values, None, 0.0)] * 3, False)
    b = np.tile(np.random.default_rng(0).standard_normal(700), 3)
    b[700] = np.inf
    x = bt.solve(b, params=solver.bicgstab_params(tolerance=1e-12), raise_on_failure=False)
    ok = [r.converged for r in bt.last_results]
    assert ok == [True, False, True]
    assert bt.split(x)[0].tobytes() == bt.split(x)[2].tobytes()
    bt.solve(b[:700].repeat(1).tolist() * 3, params=solver.bicgstab_params(
        tolerance=1e-14, max_iterations=2), raise_on_failure=False)
    assert [r.iterations for r in bt.last_results] == [2, 2, 2]


def launches(be, sizes, per_row, complex_, n_dense=0):
    """Kernel launches of one batched solve, checked against the first LU."""
    rng = np.random.default_rng(sizes[0])
    systems, rhs = [], []
    for k, n in enumerate(sizes):
        m = system(n, per_row, n_dense, seed=n)
        diag = np.repeat(np.arange(n), np.diff(m.row_pointers.astype(np.int64))) == m.col_indices
        systems.append((m.row_pointers, m.col_indices, m.values, np.abs(m.values) * 0.1 * diag,
                        1j if complex_ else 0.5))
        rhs.append(rng.standard_normal(n) + (1j * rng.standard_normal(n) if complex_ else 0))
    bt = solver.Batch(be, systems, complex_)
    prm = solver.bicgstab_params(tolerance=1e-13, max_iterations=2000)
    before = be.counters()[0]
    x = bt.solve(np.concatenate(rhs), params=prm)
    n = be.counters()[0] - before
    ref = lu(m if len(sizes) == 1 else system(sizes[0], per_row, n_dense, seed=sizes[0]),
             systems[0][3], systems[0][4], rhs[0])
    assert np.abs(bt.split(x)[0] - ref).max() < 1e-11 * np.abs(ref).max()
    return n


# Small batches, above all complex ones, are faster in one workgroup of the
# engine's own, which is one launch where the resident solve is four; so are
# two long rows up to 256, and two launches of less than 1,200 rows a system.
@pytest.mark.parametrize("sizes,per_row,complex_,n_dense,resident", [
    ([23], 3, False, 0, False), ([24], 3, False, 0, True), ([640] * 3, 3, False, 0, True),
    ([1024], 3, True, 0, False), ([1025, 9], 3, True, 0, True),
    ([256], 3, False, 2, False), ([257], 3, False, 2, True), ([700], 3, False, 2, False),
    ([1399], 3, True, 1, False), ([1400], 3, True, 1, True),
    ([700] * 140, 3, False, 0, False), ([1200] * 90, 3, False, 0, True)],
    ids=lambda v: str(v[:2]) + f"x{len(v)}" if isinstance(v, list) else None)
def test_batch_path_by_size(be, sizes, per_row, complex_, n_dense, resident):
    n = launches(be, sizes, per_row, complex_, n_dense)
    assert (n > 5) == resident, n


def test_batch_resident_from_several_threads(be):
    """Batches of four threads, each with its own backend: two fill most of the
    device and take turns, two small ones run beside them. Each gives the
    answer it gives alone."""
    jobs = []
    for n, k in ((1300, 60), (1300, 50), (2000, 2), (700, 5)):
        m = system(n, 5, 0, seed=n)
        mine = solver.HipBackend()
        bt = solver.Batch(mine, [(m.row_pointers, m.col_indices, m.values, None, 0.0)] * k, False)
        jobs.append((mine, bt, np.random.default_rng(n + k).standard_normal(n * k)))
    prm = solver.bicgstab_params(tolerance=1e-13, max_iterations=2000)
    alone = [bt.solve(b, params=prm).tobytes() for _, bt, b in jobs]
    out = [[] for _ in jobs]

    def work(k):
        for _ in range(8):
            out[k].append(jobs[k][1].solve(jobs[k][2], params=prm).tobytes())

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert [set(o) for o in out] == [{x} for x in alone]


@pytest.mark.parametrize("complex_", [False, True], ids=["real", "complex"])
def test_batch_resident_that_gives_up(be, complex_, monkeypatch):
    """A workgroup of each system stays away: after 0.2 s the others give up,
    the systems come back as they were and the engine's own kernels solve them, bit for bit as when they are asked to."""
    sizes = [1300, 1500, 1100]
    m = {n: system(n, 5, 0, seed=n) for n in sizes}
    bt = solver.Batch(be, [(m[n].row_pointers, m[n].col_indices, m[n].values, 0.1 * m[n].values,
                            1j if complex_ else 0.5) for n in sizes], complex_)
    b = np.random.default_rng(4).standard_normal(sum(sizes)) * (1 + 1j if complex_ else 1)
    prm = dict(tolerance=1e-12, max_iterations=2000)
    own = bt.solve(b, params=solver.bicgstab_params(check_interval=8, **prm))
    monkeypatch.setenv("OHM_RESIDENT_ABSENT", "1")
    try:
        x = bt.solve(b, params=solver.bicgstab_params(**prm))
        assert x.tobytes() == own.tobytes()
        monkeypatch.delenv("OHM_RESIDENT_ABSENT")
        before = be.counters()[0]
        y = bt.solve(b, params=solver.bicgstab_params(**prm))
        assert y.tobytes() == own.tobytes() and be.counters()[0] - before < 6  # not tried
    finally:
        time.sleep(1.05)
    before = be.counters()[0]
    z = bt.solve(b, params=solver.bicgstab_params(**prm))
    assert be.counters()[0] - before > 5
    assert np.abs(z - own).max() < 1e-10 * np.abs(own).max()
