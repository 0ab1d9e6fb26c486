"""The partitioned banded AC solve at the edges of its part counts: the
reduced system fetches a few parts ahead and the residual sum deals the parts
to 16 waves, so part counts around both (and one part alone) are solved and
compared with the one-lane LU of whole systems and the oracle."""
import numpy as np
import pytest

import oracle
from ohmnivore_amd import circuit as ir
from ohmnivore_amd import solver

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return solver.HipBackend()


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 7, 15, 16, 17, 33])
def test_part_counts(be, parts, monkeypatch):
    # part boundaries move by at most 16 rows, so 64 k - 31 rows make k parts
    rows = 64 * parts - 31
    m = solver.compile(ir.rlc_ladder((rows - 2) // 3, ir.SplitMix64(parts)))
    assert abs(m.size - rows) <= 3
    freqs = 10.0 ** np.linspace(0.0, 9.0, 70)     # one full wave and a part of one
    x = {}
    for r in ("0", "64"):
        monkeypatch.setenv("OHM_AC_PART_ROWS", r)
        res = solver.AcPlan(be, [m]).solve(freqs, keep_x=True)
        assert float(res.residual_norms.max()) < 1e-12
        x[r] = res.x[0]
    scale = np.abs(x["0"]).max(axis=1)
    assert float((np.abs(x["64"] - x["0"]).max(axis=1) / scale).max()) < 1e-10
    ref = oracle.ac_sweep(m, freqs)
    assert np.allclose(x["64"], ref, rtol=1e-6, atol=1e-9)


@pytest.mark.parametrize("sections,n_freqs,rows", [
    (20, 3, 64),          # the smallest part
    (5000, 61, 224),      # sqrt(3 x 15,002) up to a multiple of 32
    (5000, 1, 224),
])
def test_rows_per_part_rule(be, sections, n_freqs, rows, monkeypatch):
    monkeypatch.delenv("OHM_AC_PART_ROWS", raising=False)
    be.set_autotune(False)
    try:
        plan = solver.AcPlan(be, [solver.compile(ir.rlc_ladder(sections, ir.SplitMix64(1)))])
        res = plan.solve(10.0 ** np.linspace(0.0, 9.0, n_freqs))
    finally:
        be.set_autotune(True)
    st = plan.stats()
    assert st["rows_per_part"] == rows and st["redone_systems"] == 0
    assert float(res.residual_norms.max()) < 1e-12


def test_tuned_rows_hold_for_sweeps_like_the_first(be, monkeypatch):
    """A plan tuned on one frequency keeps its rows per part for sweeps of a few;
    400 frequencies, where the rule says twice as many rows, take the rule's."""
    monkeypatch.delenv("OHM_AC_PART_ROWS", raising=False)
    mnas = [solver.compile(ir.rlc_ladder(4000, ir.SplitMix64(k))) for k in range(16)]
    plan = solver.AcPlan(be, mnas)
    rows = []
    for n in (1, 3, 400, 2):
        res = plan.solve(10.0 ** np.linspace(0.0, 9.0, n))
        assert float(res.residual_norms.max()) < 1e-12
        rows.append(plan.stats()["rows_per_part"])
    # sqrt(3 x 12,002) and 16 x 12,002 x 400 / (64 x 3,072), up to multiples of 32
    assert rows[0] in (0, 96, 192, 288, 384, 768)
    assert rows[1] == rows[0] == rows[3] and rows[2] == 416


def test_tuning_counts_the_host_side(be, monkeypatch):
    """300 circuits of 62 rows: parts of 32 rows save a few us on the device and
    cost 60 in tables, so the tuned plan has whole systems."""
    monkeypatch.delenv("OHM_AC_PART_ROWS", raising=False)
    ms = [solver.compile(ir.rlc_ladder(20, ir.SplitMix64(k))) for k in range(4)]
    plan = solver.AcPlan(be, [ms[k % 4] for k in range(300)])
    for _ in range(2):
        res = plan.solve(10.0 ** np.linspace(0.0, 9.0, 61))
    assert plan.stats()["rows_per_part"] == 0
    assert float(res.residual_norms.max()) < 1e-12
