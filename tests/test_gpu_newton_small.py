"""Newton runs of circuits of at most 64 unknowns in one workgroup against the
general path (OHM_FUSED_SMALL=0), bit for bit: each preconditioner, dense LU
steps, shared device nodes (serial limiting), forcing, the iteration cap on
both sides of a launch's 64 iterations, and failures."""
import numpy as np
import pytest

from ohmnivore_amd import _native as N
from ohmnivore_amd import circuit as ir
from ohmnivore_amd import solver
from tests.test_gpu_dc import cmos_chain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return solver.HipBackend()


def mixed():
    """Diode, BJT and MOSFET sharing nodes, so that limiting runs serially."""
    c = ir.Circuit()
    c.add_diode_model("D", 1e-14, 1.0)
    c.add_bjt_model("Q", is_=1e-15, bf=100.0)
    c.add_mosfet_model("M", vto=0.7, kp=1e-4, lam=0.02, nmos=True)
    c.vsource("V1", "a", "0", dc=3.0)
    for k in range(4):
        c.resistor(f"R{k}", "a", f"n{k}", 1e3 * (k + 1))
        c.diode(f"D{k}", f"n{k}", "0", "D")
        c.diode(f"E{k}", f"n{k}", f"n{(k + 1) % 4}", "D")
        c.bjt(f"Q{k}", f"n{k}", f"n{(k + 1) % 4}", "0", "Q")
        c.mosfet(f"M{k}", f"n{k}", f"n{(k + 2) % 4}", "0", "M")
    return c


CIRCUITS = {"mesh7x8": lambda: ir.diode_mesh(7, 8, seed=3),        # 60 unknowns
            "mesh6x10": lambda: ir.diode_mesh(6, 10, seed=4),      # 64, the largest
            "mesh61": lambda: ir.diode_mesh(1, 61, seed=5),        # 65, general path
            "chain": lambda: cmos_chain(12), "mixed": mixed,
            "amplifier": lambda: ir.amplifier_array(12, seed=5)}


def outcome(be, m, monkeypatch, fused, **kw):
    monkeypatch.setenv("OHM_FUSED_SMALL", "1" if fused else "0")
    ctx = solver.NewtonContext(be, m.g, m.b_dc, m.diode_descriptors, m.bjt_descriptors,
                               m.mosfet_descriptors)
    try:
        st = ctx.run(**kw)
        got = (st.newton_iterations, st.bicgstab_iters_per_newton, st.max_diff)
    except N.OhmnivoreError as e:
        got = (e.kind, str(e))
    return got + (ctx.x().tobytes(),)


@pytest.mark.parametrize("name", CIRCUITS)
@pytest.mark.parametrize("kw", [
    dict(), dict(precond=N.PREC_ISAI), dict(precond=N.PREC_JACOBI), dict(precond=N.PREC_NONE),
    dict(forcing="ew1", forcing_max=0.9, forcing_safeguard="always", bicgstab_tolerance=1e-6),
    dict(linear_solver="dense"), dict(max_iterations=3), dict(abs_tol=0.0, max_iterations=64),
    dict(abs_tol=0.0, max_iterations=65), dict(abs_tol=0.0, max_iterations=130),
    dict(bicgstab_max_iterations=2)],
    ids=["auto", "isai", "jacobi", "none", "forcing", "dense", "cap3", "cap64", "cap65", "cap130",
         "subsolve_cap"])
def test_small_newton_matches_general_path(be, name, kw, monkeypatch):
    m = solver.compile(CIRCUITS[name]())
    args = dict(abs_tol=1e-10, bicgstab_tolerance=1e-9, max_iterations=60)
    args.update(kw)
    assert outcome(be, m, monkeypatch, True, **args) == outcome(be, m, monkeypatch, False, **args)


def test_small_newton_from_a_guess_and_after_an_update(be, monkeypatch):
    m = solver.compile(CIRCUITS["mesh7x8"]())
    out = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("OHM_FUSED_SMALL", fused)
        ctx = solver.NewtonContext(be, m.g, m.b_dc, m.diode_descriptors)
        kw = dict(abs_tol=1e-10, bicgstab_tolerance=1e-9, max_iterations=80)
        ctx.run(**kw)
        x0 = ctx.x()
        ctx.update(base_b=m.b_dc * 1.1)
        ctx.run(initial_guess=x0, **kw)
        x1 = ctx.x()
        gg, gk, lam, _ = ctx.adjoint(np.linspace(0, 1, m.size))
        out[fused] = (x0.tobytes(), x1.tobytes(), lam)
    assert out["1"][:2] == out["0"][:2]
    # the adjoint's ILU sweeps start from factors of the run's last refresh
    assert np.allclose(out["1"][2], out["0"][2], rtol=1e-8, atol=1e-10 * np.abs(out["0"][2]).max())


def random_mosfets(nodes, count, seed):
    r = np.random.default_rng(seed)
    c = ir.Circuit()
    c.add_mosfet_model("M", vto=0.7, kp=1e-4, lam=0.02, nmos=True)
    c.vsource("V1", "a", "0", dc=2.0)
    for k in range(nodes):
        c.resistor(f"R{k}", "a" if k == 0 else f"n{k - 1}", f"n{k}", 150.0)
        c.resistor(f"S{k}", f"n{k}", "0", 1e4)
    for k in range(count):
        c.mosfet(f"M{k}", *(f"n{r.integers(nodes)}" for _ in range(3)), "M")
    return c


def shared_diodes(count):
    c = ir.Circuit()
    c.add_diode_model("D", 1e-14, 1.0)
    c.vsource("V1", "a", "0", dc=2.0)
    for k in range(8):
        c.resistor(f"R{k}", "a" if k == 0 else f"n{k - 1}", f"n{k}", 150.0)
    for k in range(count):
        c.diode(f"D{k}", f"n{k % 8}", "0", "D")
    return c


# Where one workgroup is the slower one a run is the general path's: serial
# limiting of many diodes, and large ISAI factors. Dense steps stay.
@pytest.mark.parametrize("make,kw,small", [
    (lambda: shared_diodes(512), dict(precond=N.PREC_ISAI), True),
    (lambda: shared_diodes(513), dict(precond=N.PREC_ISAI), False),
    (lambda: shared_diodes(513), dict(linear_solver="dense"), True),
    (lambda: random_mosfets(58, 60, 1), dict(precond=N.PREC_ISAI), True),
    (lambda: random_mosfets(58, 200, 1), dict(precond=N.PREC_ISAI), False),
    (lambda: random_mosfets(58, 200, 1), dict(precond=N.PREC_JACOBI), True),
    (lambda: random_mosfets(30, 900, 1), dict(precond=N.PREC_ISAI), True)],
    ids=["512diodes", "513diodes", "513dense", "sparse", "dense_factors", "jacobi", "few_unknowns"])
def test_small_newton_path_by_size(be, make, kw, small, monkeypatch):
    m = solver.compile(make())
    args = dict(abs_tol=1e-9, bicgstab_tolerance=1e-9, max_iterations=60, **kw)
    monkeypatch.setenv("OHM_FUSED_SMALL", "1")
    ctx = solver.NewtonContext(be, m.g, m.b_dc, m.diode_descriptors, m.bjt_descriptors,
                               m.mosfet_descriptors)
    ctx.run(**args)
    before = be.counters()[0]
    st = ctx.run(**args)
    launches = be.counters()[0] - before
    assert (launches < 4 * st.newton_iterations) == small, (launches, st.newton_iterations)
    assert outcome(be, m, monkeypatch, True, **args) == outcome(be, m, monkeypatch, False, **args)
