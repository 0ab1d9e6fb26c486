"""The work that users of this framework have it do, as timed cases.

Each case is one call (or the few calls) a circuit-simulation program makes
through the public Python entry points, with what such a program holds
beforehand (compiled circuits, plans, device contexts) made in ``prepare``:

- ``dc_linear``    a linear operating point: GpuSolver.solve_real from host
                   arrays, a new matrix every call (LinearSolver's contract);
- ``dc_chain``     a CMOS inverter chain's .DC through the continuation cascade;
- ``newton``       newton_solve in one shot on a small diode mesh;
- ``newton_ctx``   Newton again on a device-resident context (a large mesh);
- ``tran_grid``    backward-Euler steps of an RC power grid, one instance;
- ``tran_mc``      the same for several Monte Carlo instances at once;
- ``tran_chain``   .TRAN of an inverter chain: a Newton solve per timestep;
- ``ac_grid``      .AC of an RC mesh (wide band: batched BiCGSTAB);
- ``ac_ladder``    .AC of RLC ladders in one shot, every phasor to the host;
- ``ac_plan``      a sweep of many ladders on a resident plan, a few read back;
- ``adjoint``      operating point and its gradients: forward and backward.

Sizes run from circuits of a few dozen unknowns, where launches and latency
are the cost, to the power grid and mesh of the benchmark.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ohmnivore_amd import _native as N
from ohmnivore_amd import adjoint as A
from ohmnivore_amd import circuit as ir
from ohmnivore_amd import dc, netlist, solver, transient

H = 1e-12          # timestep of the grid transients, the benchmark's 1 ps
GRID_STEPS = 10


def listed() -> list[dict]:
    return [
        # a hand-drawn circuit: a few dozen unknowns, the smallest call there is
        {"name": "dc_linear_40", "path": "dc_linear", "sections": 40, "precision": "fp64"},
        # the 10,000-section resistor ladder of the benchmark
        {"name": "dc_linear_10000", "path": "dc_linear", "sections": 10_000, "precision": "fp64"},
        # the middle of the 10-200 stage family of CMOS inverter chains, .DC
        {"name": "dc_chain_50", "path": "dc_chain", "stages": 50},
        # a small nonlinear mesh of odd sides, solved once
        {"name": "newton_61x47", "path": "newton", "rows": 61, "cols": 47},
        # the 256 x 256 diode mesh of the benchmark on a resident context
        {"name": "newton_ctx_256x256", "path": "newton_ctx", "rows": 256, "cols": 256},
        # the 512 x 512 power grid of the benchmark, ISAI
        {"name": "tran_grid_512x512", "path": "tran_grid", "rows": 512, "cols": 512,
         "precond": "isai", "precision": "fp64"},
        # Monte Carlo: 8 instances of a medium grid stepped together
        {"name": "tran_mc_8x128x128", "path": "tran_mc", "rows": 128, "cols": 128,
         "instances": 8},
        # a short inverter chain's .TRAN, the MOSFETs in the time loop
        {"name": "tran_chain_20", "path": "tran_chain", "stages": 20, "steps": 30},
        # a mesh that no band solver takes, over a log sweep
        {"name": "ac_grid_45x41", "path": "ac_grid", "rows": 45, "cols": 41, "freqs": 21},
        # one ladder's .AC from the command line: 61 points, all phasors back
        {"name": "ac_ladder_1x5000", "path": "ac_ladder", "circuits": 1, "sections": 5000,
         "freqs": 61},
        # a design sweep: 48 uneven ladders of 1,000-64,000 sections x 101 points
        {"name": "ac_plan_48x101", "path": "ac_plan", "circuits": 48, "lo": 1000, "hi": 64_000,
         "freqs": 101},
        # operating point and gradients of a 1,024-stage amplifier array
        {"name": "adjoint_1024", "path": "adjoint", "stages": 1024},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng) -> dict:
    path = rng.choice(["dc_linear", "dc_chain", "newton", "newton_ctx", "tran_grid", "tran_mc",
                       "tran_chain", "ac_grid", "ac_ladder", "ac_plan", "adjoint"])
    if path == "dc_linear":
        return {"path": path, "sections": _log_int(rng, 20, 20_000),
                "precision": rng.choice(["fp64", "fp64", "fp32_ir"])}
    if path == "dc_chain":
        return {"path": path, "stages": _log_int(rng, 5, 60)}
    if path == "newton":
        return {"path": path, "rows": _log_int(rng, 7, 70), "cols": _log_int(rng, 7, 70)}
    if path == "newton_ctx":
        return {"path": path, "rows": _log_int(rng, 24, 256), "cols": _log_int(rng, 24, 256)}
    if path == "tran_grid":
        return {"path": path, "rows": _log_int(rng, 24, 512), "cols": _log_int(rng, 24, 512),
                "precond": rng.choice(["isai", "jacobi"]),
                "precision": rng.choice(["fp64", "fp64", "fp64", "fp32_ir"])}
    if path == "tran_mc":
        return {"path": path, "rows": _log_int(rng, 20, 160), "cols": _log_int(rng, 20, 160),
                "instances": rng.randint(2, 8)}
    if path == "tran_chain":
        return {"path": path, "stages": _log_int(rng, 3, 24), "steps": rng.randint(10, 30)}
    if path == "ac_grid":
        return {"path": path, "rows": _log_int(rng, 9, 64), "cols": _log_int(rng, 9, 64),
                "freqs": rng.randint(5, 21)}
    if path == "ac_ladder":
        return {"path": path, "circuits": rng.randint(1, 4),
                "sections": _log_int(rng, 100, 5000), "freqs": rng.randint(11, 81)}
    if path == "ac_plan":
        lo = _log_int(rng, 500, 4000)
        return {"path": path, "circuits": _log_int(rng, 1, 48), "lo": lo,
                "hi": _log_int(rng, lo, 64_000), "freqs": rng.randint(5, 101)}
    return {"path": path, "stages": _log_int(rng, 12, 2048)}


# ------------------------------------------------------------- circuits ----
def _chain(stages: int, seed: int, analysis: str) -> str:
    """A CMOS inverter chain netlist; supply and model cards vary with the seed."""
    r = np.random.default_rng([seed, 11])
    vdd = 5.0 * (1 + 0.05 * (r.random() - 0.5))
    kn, kp = 1.1e-4 * (1 + 0.2 * (r.random() - 0.5)), 5.5e-5 * (1 + 0.2 * (r.random() - 0.5))
    vin = (f"VIN in 0 DC {vdd:.6g}" if analysis == "dc"
           else f"VIN in 0 PULSE(0 {vdd:.6g} 10n 1n 1n 50n 100n)")
    lines = ["* CMOS inverter chain",
             f".MODEL NMOD NMOS(VTO=0.7 KP={kn:.6g} LAMBDA=0.04)",
             f".MODEL PMOD PMOS(VTO=-0.7 KP={kp:.6g} LAMBDA=0.04)",
             f"VDD vdd 0 DC {vdd:.6g}", vin]
    for i in range(1, stages + 1):
        gate = "in" if i == 1 else f"out_{i - 1}"
        lines += [f"MP{i} out_{i} {gate} vdd vdd PMOD", f"MN{i} out_{i} {gate} 0 0 NMOD"]
    return "\n".join(lines + [".DC", ".END", ""])


def _rc_mesh(rows: int, cols: int, seed: int) -> ir.Circuit:
    """An RC mesh driven at one corner through 50 ohm by a 1 V AC source."""
    r = np.random.default_rng([seed, 12])
    ckt = ir.Circuit()
    ckt.vsource("V1", "in", "0", ac=(1.0, 0.0))
    ids = ckt.nodes(f"n{i}_{j}" for i in range(rows) for j in range(cols)).reshape(rows, cols)
    ckt.resistor("RS", "in", "n0_0", 50.0)
    a = np.concatenate([ids[:, :-1].ravel(), ids[:-1].ravel()])
    b = np.concatenate([ids[:, 1:].ravel(), ids[1:].ravel()])
    ckt.resistors(a, b, 10.0 ** r.uniform(2, 4, a.shape[0]))
    gnd = np.full(rows * cols, ckt.node("0"), np.int32)
    ckt.capacitors(ids.ravel(), gnd, 10.0 ** r.uniform(-13, -11, rows * cols))
    return ckt


def _ladders(case: dict, seed: int):
    rng = ir.SplitMix64(1000 + seed)
    k = case["circuits"]
    if case["path"] == "ac_ladder":
        sections = [max(2, int(case["sections"] * (1 - 0.1 * j))) for j in range(k)]
    else:  # uneven, spread over [lo, hi]: the sizes belong to the case, not the seed
        step = (math.sqrt(5) - 1) / 2
        sections = [int(case["lo"] + (case["hi"] - case["lo"]) * ((0.5 + j * step) % 1.0))
                    for j in range(k)]
    return [ir.rlc_ladder(s, rng) for s in sections], sections


def _freqs(case: dict) -> np.ndarray:
    nf = case["freqs"]
    if case["path"] == "ac_grid":
        return 10.0 ** (4.0 + 5.0 * np.arange(nf) / max(nf - 1, 1))
    return 10.0 ** (9.0 * np.arange(nf) / max(nf - 1, 1))


def _grid(case: dict, seed: int):
    ckt = ir.rc_grid(case["rows"], case["cols"],
                     max(4, case["rows"] * case["cols"] // 256), seed=3000 + seed)
    for w in ckt.tran.values():   # the sinks switch on within the steps taken
        w.td *= GRID_STEPS * H / 1e-9
    mna = solver.compile(ckt)
    x0 = np.zeros(mna.size)   # no sink conducts at t = 0: every node sits at the supply
    x0[:mna.n_nodes] = 1.0
    return ckt, mna, x0


def _instances(case: dict, seed: int, mna):
    r = np.random.default_rng([seed, 13])
    cg = transient.c_on_g(mna)
    return [(mna.g.values * (1 + 0.05 * (r.random() - 0.5)),
             cg * (1 + 0.2 * r.random(cg.shape[0]))) for _ in range(case["instances"])]


def _amplifier(case: dict, seed: int):
    ckt = ir.amplifier_array(case["stages"], seed=5000 + seed)
    return ckt, solver.compile(ckt)


# -------------------------------------------------------------- prepare ----
_BACKEND = None


def _backend() -> solver.HipBackend:
    """The program's one backend."""
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = solver.HipBackend()
    return _BACKEND


NEWTON_KW = dict(abs_tol=1e-9, bicgstab_tolerance=1e-10)
MESH_KW = dict(abs_tol=1e-10, max_iterations=100, bicgstab_tolerance=1e-8)
# the benchmark's settings for the large mesh
MESH_CTX_KW = dict(abs_tol=1e-10, max_iterations=100, bicgstab_tolerance=1e-6,
                   bicgstab_max_iterations=20_000, forcing="ew1", forcing_max=0.9,
                   forcing_safeguard="always", bicgstab_floor=1e-18)


def prepare(case: dict, seed: int) -> dict:
    be, path = _backend(), case["path"]
    if path == "dc_linear":
        m = solver.compile(ir.resistor_ladder(case["sections"], seed=100 + seed))
        prm = solver.bicgstab_params(tolerance=1e-13, max_iterations=200_000,
                                     precision=case["precision"])
        return {"path": path, "mna": m,
                "solver": solver.GpuSolver(be, precond=N.PREC_JACOBI, params=prm)}
    if path == "dc_chain":
        ckt = netlist.parse(_chain(case["stages"], seed, "dc")).to_circuit()
        return {"path": path, "mna": solver.compile(ckt)}
    if path == "newton":
        return {"path": path,
                "mna": solver.compile(ir.diode_mesh(case["rows"], case["cols"], seed=200 + seed))}
    if path == "newton_ctx":
        m = solver.compile(ir.diode_mesh(case["rows"], case["cols"], seed=200 + seed))
        return {"path": path, "ctx": solver.NewtonContext(be, m.g, m.b_dc, m.diode_descriptors)}
    if path in ("tran_grid", "tran_mc"):
        ckt, mna, x0 = _grid(case, seed)
        src, pwl = transient.source_table(ckt, mna)
        inst = _instances(case, seed, mna) if path == "tran_mc" else None
        tr = transient.Transient(be, mna, src, pwl, instances=inst)
        isai = case.get("precond") == "isai"
        return {"path": path, "tran": tr, "x0": x0,
                "precond": N.PREC_ISAI if isai else N.PREC_JACOBI,
                "probes": np.arange(0, mna.size, max(1, mna.size // 64)),
                "params": solver.bicgstab_params(tolerance=1e-10, max_iterations=20_000,
                                                 precision=case.get("precision", "fp64"))}
    if path == "tran_chain":
        ckt = netlist.parse(_chain(case["stages"], seed, "tran")).to_circuit()
        return {"path": path, "ckt": ckt, "mna": solver.compile(ckt), "steps": case["steps"]}
    if path == "ac_grid":
        return {"path": path, "mnas": [solver.compile(_rc_mesh(case["rows"], case["cols"], seed))],
                "freqs": _freqs(case),
                "params": solver.bicgstab_params(tolerance=1e-10, max_iterations=100_000)}
    if path == "ac_ladder":
        ckts, _ = _ladders(case, seed)
        return {"path": path, "mnas": [solver.compile(c) for c in ckts], "freqs": _freqs(case),
                "params": solver.bicgstab_params(tolerance=1e-10, max_iterations=100_000)}
    if path == "ac_plan":
        ckts, _ = _ladders(case, seed)
        plan = solver.AcPlan(be, [solver.compile(c) for c in ckts])
        return {"path": path, "plan": plan, "freqs": _freqs(case),
                "read": list(range(0, case["circuits"], 8))}
    ckt, mna = _amplifier(case, seed)
    prob = A.DcProblem(be, ckt, mna)
    return {"path": path, "problem": prob, "outs": torch.from_numpy(A.output_nodes(ckt, mna)),
            "g": torch.from_numpy(prob.g0.copy()), "kp": torch.from_numpy(prob.kp0.copy())}


# ------------------------------------------------------------------ run ----
def run(state: dict):
    be, path = _backend(), state["path"]
    if path == "dc_linear":
        m = state["mna"]
        return state["solver"].solve_real(m.g, m.b_dc)
    if path == "dc_chain":
        return dc.run(be, state["mna"], **NEWTON_KW).x
    if path == "newton":
        m = state["mna"]
        x, _ = solver.newton_solve(be, m.g, m.b_dc, m.diode_descriptors, **MESH_KW)
        return x
    if path == "newton_ctx":
        state["ctx"].run(**MESH_CTX_KW)
        return state["ctx"].x()
    if path in ("tran_grid", "tran_mc"):
        r = state["tran"].run(H, GRID_STEPS * H, method="be", x0=state["x0"],
                              probes=state["probes"], params=state["params"],
                              precond=state["precond"])
        return {"times": r.times, "waves": r.waves, "x_final": r.x_final}
    if path == "tran_chain":
        r = transient.run(be, state["ckt"], state["mna"], 1e-9, state["steps"] * 1e-9,
                          dc_kw=NEWTON_KW).result
        return {"times": r.times, "waves": r.waves}
    if path in ("ac_grid", "ac_ladder"):
        r = solver.ac_sweep_circuits(be, state["mnas"], state["freqs"], params=state["params"])
        return r.x
    if path == "ac_plan":
        plan, f = state["plan"], state["freqs"]
        r = plan.solve(f)
        return {"status": r.records["status"],
                "x": [plan.x(c, f.shape[0] // 2, 1) for c in state["read"]]}
    g = state["g"].clone().requires_grad_(True)
    kp = state["kp"].clone().requires_grad_(True)
    x = A.DcOperatingPoint.apply(g, kp, state["problem"])
    A.objective(x, state["outs"]).backward()
    return {"x": x.detach(), "grad_g": g.grad, "grad_kp": kp.grad}


# ----------------------------------------------------------------- work ----
def work(case: dict) -> dict:
    """Inputs once and results once: matrices at 12 bytes an entry, device
    cards at their descriptor sizes, solutions at 8 (16) bytes an unknown; a
    transient reads the matrix and writes a state every step. Flops: one
    multiply-add per matrix entry of one product (a solve needs at least one)."""
    path = case["path"]
    if path == "dc_linear":
        n, reps, cplx = case["sections"] + 2, 1, 1
        nnz = 3 * n
    elif path in ("dc_chain", "tran_chain"):
        n = case["stages"] + 4
        nnz, reps, cplx = 6 * n, case.get("steps", 1), 1
    elif path in ("newton", "newton_ctx", "tran_grid", "tran_mc"):
        n = case["rows"] * case["cols"] + 4
        nnz, reps, cplx = 5 * n, 1, 1
        if path in ("tran_grid", "tran_mc"):
            reps = GRID_STEPS * case.get("instances", 1)
    elif path == "ac_grid":
        n = case["rows"] * case["cols"] + 2
        nnz, reps, cplx = 5 * n, case["freqs"], 2
    elif path in ("ac_ladder", "ac_plan"):
        # a direct solve of every (circuit, frequency) system: its unknowns
        # written once each; the band rows of a circuit read once
        if path == "ac_ladder":
            sections = [max(2, int(case["sections"] * (1 - 0.1 * j)))
                        for j in range(case["circuits"])]
        else:
            step = (math.sqrt(5) - 1) / 2
            sections = [int(case["lo"] + (case["hi"] - case["lo"]) * ((0.5 + j * step) % 1.0))
                        for j in range(case["circuits"])]
        rows = sum(3 * s + 2 for s in sections)
        return {"bytes": 64.0 * rows + 16.0 * rows * case["freqs"],
                "flops": 40.0 * rows * case["freqs"]}
    else:
        n = 2 * case["stages"] + 2
        return {"bytes": 2 * 12.0 * 4 * n + 8.0 * 6 * n, "flops": 4.0 * 4 * n}
    return {"bytes": (12.0 * nnz + 16.0 * cplx * n) * reps, "flops": 2.0 * cplx * cplx * nnz * reps}


def tolerance(case: dict):
    """Every solve stops on a residual, so two correct implementations agree
    to that residual times the conditioning of the circuit. Figures: about
    four times the largest distance from ``exact`` over listed and drawn cases."""
    return {"rel": {"dc_linear": 1e-9,    # residual 1e-13, far nodes decayed
                    "dc_chain": 1e-8,     # Newton stops at 1e-9 V
                    "newton": 1e-8, "newton_ctx": 1e-8,
                    "tran_grid": 1e-9, "tran_mc": 1e-9,   # residual 1e-10 a step
                    "tran_chain": 1e-8,
                    "ac_grid": 4e-6,      # residual 1e-10 against the source's row
                    "ac_ladder": 1e-9,    # direct; resonances at the sweep's ends
                    "ac_plan": 1e-11, "adjoint": 1e-10}[case["path"]]}


# ---------------------------------------------------------------- exact ----
def _xv(x, idx):
    return np.where(idx == ir.SENTINEL, 0.0, x[np.minimum(idx, x.shape[0] - 1).astype(np.int64)])


def _add(mat, r, c, v):
    ok = (r != ir.SENTINEL) & (c != ir.SENTINEL)
    np.add.at(mat, (r[ok].astype(np.int64), c[ok].astype(np.int64)), v[ok])


def _add1(vec, r, v):
    ok = r != ir.SENTINEL
    np.add.at(vec, r[ok].astype(np.int64), v[ok])


def _soft(v_ov):
    """Smoothed overdrive of the level-1 MOSFET and its slope."""
    vt = 0.02585
    a = v_ov / vt
    with np.errstate(over="ignore"):
        e = np.exp(np.minimum(a, 20.0))
    mid = vt * np.log1p(e)
    return (np.where(a > 20, v_ov, np.where(a < -20, vt * e, mid)),
            np.where(a > 20, 1.0, np.where(a < -20, e, e / (1 + e))))


def _mosfet(x, m, kp=None):
    f = {k: m[k].astype(np.float64) for k in ("polarity", "vto", "kp", "lambda")}
    kp = f["kp"] if kp is None else kp
    vd, vg, vs = _xv(x, m["drain_idx"]), _xv(x, m["gate_idx"]), _xv(x, m["source_idx"])
    vgs, vds = f["polarity"] * (vg - vs), f["polarity"] * (vd - vs)
    ov, sig = _soft(vgs - f["vto"])
    lam = 1 + f["lambda"] * vds
    tri = vds < ov
    inner = np.where(tri, ov * vds - 0.5 * vds * vds, 0.5 * ov * ov)
    i = kp * inner * lam
    gm = np.where(tri, kp * vds * lam * sig, kp * ov * lam * sig)
    gds = np.where(tri, kp * (ov - vds) * lam, 0.0) + kp * inner * f["lambda"]
    return f["polarity"] * i, gm, gds


def _residual(gd, b, x, m, mosfet_kp=None):
    """F(x) and its Jacobian: G x + i(x) - b, dense."""
    jac = gd.copy()
    res = gd @ x - b
    d = m.diode_descriptors
    if len(d):
        a, c = d["anode_idx"], d["cathode_idx"]
        i_s, nvt = d["is_val"].astype(np.float64), d["n_vt"].astype(np.float64)
        e = np.exp(np.clip((_xv(x, a) - _xv(x, c)) / nvt, -80, 80))
        g, i = i_s * e / nvt, i_s * (e - 1)
        _add1(res, a, i)
        _add1(res, c, -i)
        for r, cc, s in ((a, a, 1), (c, c, 1), (a, c, -1), (c, a, -1)):
            _add(jac, r, cc, s * g)
    q = m.bjt_descriptors
    if len(q):
        f = {k: q[k].astype(np.float64) for k in ("polarity", "is_val", "bf", "br", "nf_vt", "nr_vt")}
        ci, bi, ei = q["collector_idx"], q["base_idx"], q["emitter_idx"]
        vc, vb, ve = _xv(x, ci), _xv(x, bi), _xv(x, ei)
        ef = np.exp(np.clip(f["polarity"] * (vb - ve) / f["nf_vt"], -80, 80))
        er = np.exp(np.clip(f["polarity"] * (vb - vc) / f["nr_vt"], -80, 80))
        i_f, i_r = f["is_val"] * (ef - 1), f["is_val"] * (er - 1)
        gf, gr = f["is_val"] * ef / f["nf_vt"], f["is_val"] * er / f["nr_vt"]
        af, ar, kf = f["bf"] / (f["bf"] + 1), 1 / (f["br"] + 1), 1 / (f["bf"] + 1)
        ic, ib = f["polarity"] * (af * i_f - ar * i_r), f["polarity"] * (kf * i_f + ar * i_r)
        _add1(res, ci, ic)
        _add1(res, bi, ib)
        _add1(res, ei, -(ic + ib))
        dic = {"c": ar * gr, "b": af * gf - ar * gr, "e": -af * gf}
        dib = {"c": -ar * gr, "b": kf * gf + ar * gr, "e": -kf * gf}
        for t, idx in (("c", ci), ("b", bi), ("e", ei)):
            _add(jac, ci, idx, dic[t])
            _add(jac, bi, idx, dib[t])
            _add(jac, ei, idx, -(dic[t] + dib[t]))
    t = m.mosfet_descriptors
    if len(t):
        i, gm, gds = _mosfet(x, t, mosfet_kp)
        di, gi, si = t["drain_idx"], t["gate_idx"], t["source_idx"]
        _add1(res, di, i)
        _add1(res, si, -i)
        for idx, v in ((di, gds), (gi, gm), (si, -(gm + gds))):
            _add(jac, di, idx, v)
            _add(jac, si, idx, -v)
    return res, jac


def _lin(a, b):
    return torch.linalg.solve(torch.from_numpy(a), torch.from_numpy(b)).numpy()


def _operating_point(m, b, x, limit=0.3, kp=None):
    """Step-limited Newton to rounding, over rising sources where a plain run
    does not settle."""
    gd = m.g.to_dense()

    def newton(bb, x):
        for k in range(200):
            res, jac = _residual(gd, bb, x, m, kp)
            try:
                dx = _lin(jac, -res)
            except RuntimeError:    # a node that every device has let go of
                return None
            big = np.max(np.abs(dx[:m.n_nodes]))
            x = x + dx * min(1.0, limit / big if big > 0 else 1.0)
            if big < 1e-13:
                return x
            if big < 1e-10 and k > 60:
                return x
        return None

    y = newton(b, x)
    if y is None:
        y = np.zeros(m.size)
        for s in np.linspace(0.05, 1.0, 20):
            y = newton(s * b, y)
            if y is None:
                return None
    return y


def _sources_at(ckt, mna, t):
    """b(t): each source's value at its branch row or its two nodes."""
    b = np.zeros(mna.size)
    comps, index = ckt.components, {nm: i for i, nm in enumerate(mna.node_names)}
    branch = 0
    for k in range(comps.shape[0]):
        kind = int(comps["kind"][k])
        if kind == ir.L:
            branch += 1
        if kind not in (ir.V, ir.I):
            continue
        w = ckt.tran.get(k)
        dcv = float(comps["value"][k]) if int(comps["flags"][k]) & ir.HAS_DC else 0.0
        v = w(t) if w is not None else dcv
        if kind == ir.V:
            b[mna.n_nodes + branch] += v
            branch += 1
        else:
            for node, s in ((int(comps["node"][k][0]), -1.0), (int(comps["node"][k][1]), 1.0)):
                nm = ckt.node_names[node]
                if not ir.is_ground(nm):
                    b[index[nm]] += s * v
    return b


def _sparse(m, values):
    n = m.size
    return torch.sparse_csr_tensor(torch.from_numpy(m.g.row_pointers.astype(np.int64)),
                                   torch.from_numpy(m.g.col_indices.astype(np.int64)),
                                   torch.from_numpy(values), (n, n), dtype=torch.float64)


def _grid_exact(ckt, mna, x0, gv, cv, probes):
    """Backward Euler of a grid whose only branches are supply pads: the free
    nodes' matrix is symmetric positive definite, solved by conjugate
    gradients to rounding."""
    n, nn = mna.size, mna.n_nodes
    a = gv + cv / H
    am, cm = _sparse(mna, a), _sparse(mna, cv / H)
    rows = np.repeat(np.arange(n), np.diff(mna.g.row_pointers.astype(np.int64)))
    cols = mna.g.col_indices.astype(np.int64)
    on = (rows == cols)
    diag = np.zeros(n)
    diag[rows[on]] = a[on]
    pad_of = {}     # branch row -> (pad node, its coefficient)
    for r in range(nn, n):
        ks = [k for k in range(int(mna.g.row_pointers[r]), int(mna.g.row_pointers[r + 1]))
              if mna.g.values[k] != 0.0]
        pad_of[r] = (int(cols[ks[0]]), gv[ks[0]])
    free = np.ones(n, dtype=bool)
    free[nn:] = False
    for node, _ in pad_of.values():
        free[node] = False
    fm, inv = torch.from_numpy(free.astype(np.float64)), torch.from_numpy(
        np.where(free, 1.0 / np.where(diag == 0, 1.0, diag), 0.0))
    x = torch.from_numpy(x0.copy())
    times, waves, t = [0.0], [x.numpy()[probes].copy()], 0.0
    tstop = GRID_STEPS * H
    while t < tstop:
        h = min(H, tstop - t)
        if h < H / 10000.0 * 0.5:
            break
        t = t + h
        rhs = torch.from_numpy(_sources_at(ckt, mna, t)) + cm @ x * (H / h)
        y = x.clone()
        for r, (node, coef) in pad_of.items():
            y[node] = rhs[r] / coef
        y[nn:] = 0.0
        res = (rhs - am @ y) * fm
        z = inv * res
        p, rz, stop = z.clone(), torch.dot(res, z), 1e-15 * float(torch.linalg.norm(rhs[:nn]))
        for _ in range(3000):
            ap = (am @ p) * fm
            al = rz / torch.dot(p, ap)
            y += al * p
            res -= al * ap
            if float(torch.linalg.norm(res)) < stop:
                break
            z = inv * res
            rz, old = torch.dot(res, z), rz
            p = z + (rz / old) * p
        left = rhs - am @ y
        for r, (node, _) in pad_of.items():   # pad current closes its node's balance
            k = [k for k in range(int(mna.g.row_pointers[node]), int(mna.g.row_pointers[node + 1]))
                 if cols[k] == r][0]
            y[r] = left[node] / gv[k]
        x = y
        times.append(t)
        waves.append(x.numpy()[probes].copy())
    return np.array(times), np.array(waves), x.numpy()


def _ladder_exact(mna, ckt, freqs):
    """An RLC ladder's phasors from the input admittances of its tails."""
    comps = ckt.components
    v = comps["value"]
    r, l, c = (v[comps["kind"] == k] for k in (ir.R, ir.L, ir.C))
    s = r.shape[0]
    w = 2 * np.pi * np.asarray(freqs)
    gmin = 1e-12     # the shunt the compiler puts on every node diagonal
    tail = np.zeros((s, w.shape[0]), dtype=np.complex128)   # admittance right of a_{k+1}
    y = np.zeros(w.shape[0], dtype=np.complex128)
    for k in range(s - 1, -1, -1):
        y = y + 1j * w * c[k] + gmin
        tail[k] = y
        yb = gmin + y / (1 + 1j * w * l[k] * y)              # at b_k
        y = yb / (1 + r[k] * yb)
    x = np.zeros((w.shape[0], mna.size), dtype=np.complex128)
    index = {nm: i for i, nm in enumerate(mna.node_names)}
    va = np.ones(w.shape[0], dtype=np.complex128)
    x[:, index["a1"]] = va
    il = np.zeros((s, w.shape[0]), dtype=np.complex128)
    iv = None
    for k in range(s):
        yt = tail[k]
        yb = gmin + yt / (1 + 1j * w * l[k] * yt)
        vb = va / (1 + r[k] * yb)
        if k == 0:
            iv = -(va * gmin + (va * yb) / (1 + r[k] * yb))
        i = vb * yt / (1 + 1j * w * l[k] * yt)
        va = i / yt
        x[:, index[f"b{k + 1}"]] = vb
        x[:, index[f"a{k + 2}"]] = va
        il[k] = i
    nl = 0
    for j, comp in enumerate(mna.extra["branch_components"]):
        if int(comps["kind"][comp]) == ir.V:
            x[:, mna.n_nodes + j] = iv
        else:
            x[:, mna.n_nodes + j] = il[nl]
            nl += 1
    return x


def exact(case: dict, seed: int):
    path = case["path"]
    if path == "dc_linear":
        if case["sections"] > 10_200:
            return None
        m = solver.compile(ir.resistor_ladder(case["sections"], seed=100 + seed))
        return _lin(m.g.to_dense(), m.b_dc)
    if path == "dc_chain":
        m = solver.compile(netlist.parse(_chain(case["stages"], seed, "dc")).to_circuit())
        return _operating_point(m, m.b_dc, np.zeros(m.size))
    if path in ("newton", "newton_ctx"):
        if case["rows"] * case["cols"] > 3000:
            return None
        m = solver.compile(ir.diode_mesh(case["rows"], case["cols"], seed=200 + seed))
        # from below the diodes' turn-on everywhere: each step is limited
        return _operating_point(m, m.b_dc, np.zeros(m.size), limit=0.1)
    if path in ("tran_grid", "tran_mc"):
        ckt, mna, x0 = _grid(case, seed)
        probes = np.arange(0, mna.size, max(1, mna.size // 64))
        inst = (_instances(case, seed, mna) if path == "tran_mc"
                else [(mna.g.values, transient.c_on_g(mna))])
        if mna.size * len(inst) > 300_000:
            return None
        got = [_grid_exact(ckt, mna, x0, g, c, probes) for g, c in inst]
        return {"times": got[0][0], "waves": np.stack([w for _, w, _ in got], axis=1),
                "x_final": np.stack([x for _, _, x in got])}
    if path == "tran_chain":
        ckt = netlist.parse(_chain(case["stages"], seed, "tran")).to_circuit()
        m = solver.compile(ckt)
        x = _operating_point(m, m.b_dc, np.zeros(m.size))
        if x is None:
            return None
        # no capacitors: every step is the operating point at its own time
        times, waves, t = [0.0], [x], 0.0
        tstop = case["steps"] * 1e-9
        while t < tstop:
            h = min(1e-9, tstop - t)
            if h < 1e-9 / 10000.0 * 0.5:
                break
            t = t + h
            x = _operating_point(m, _sources_at(ckt, m, t), x)
            if x is None:
                return None
            times.append(t)
            waves.append(x)
        return {"times": np.array(times), "waves": np.array(waves)[:, None, :]}
    if path == "ac_grid":
        if case["rows"] * case["cols"] > 2000:
            return None
        m = solver.compile(_rc_mesh(case["rows"], case["cols"], seed))
        g, c = m.g.to_dense(), m.c.to_dense()
        return [np.stack([_lin(g + 2j * np.pi * f * c, m.b_ac) for f in _freqs(case)])]
    if path in ("ac_ladder", "ac_plan"):
        ckts, sections = _ladders(case, seed)
        f = _freqs(case)
        read = range(0, case["circuits"], 8) if path == "ac_plan" else range(case["circuits"])
        if sum(sections[c] for c in read) > 300_000:
            return None
        if path == "ac_plan":
            f = f[case["freqs"] // 2: case["freqs"] // 2 + 1]
        xs = [_ladder_exact(solver.compile(ckts[c]), ckts[c], f) for c in read]
        return {"status": None, "x": xs} if path == "ac_plan" else xs
    if case["stages"] > 1100:
        return None
    ckt, m = _amplifier(case, seed)
    x = _operating_point(m, m.b_dc, np.zeros(m.size))
    if x is None:
        return None
    res, jac = _residual(m.g.to_dense(), m.b_dc, x, m)
    outs = A.output_nodes(ckt, m)
    dj = np.zeros(m.size)
    dj[outs] = 2 * (x[outs] - 0.9)
    lam = _lin(np.ascontiguousarray(jac.T), dj)
    comps, index = ckt.components, {nm: i for i, nm in enumerate(m.node_names)}
    sel = np.nonzero(comps["kind"] == ir.R)[0]
    ends = np.array([[ir.SENTINEL if ir.is_ground(ckt.node_names[int(e)]) else
                      index[ckt.node_names[int(e)]] for e in comps["node"][k][:2]] for k in sel],
                    dtype=np.uint32)
    gg = -(_xv(lam, ends[:, 0]) - _xv(lam, ends[:, 1])) * (_xv(x, ends[:, 0]) - _xv(x, ends[:, 1]))
    t = m.mosfet_descriptors
    unit, _, _ = _mosfet(x, t, np.ones(len(t)))
    gk = -(_xv(lam, t["drain_idx"]) - _xv(lam, t["source_idx"])) * unit
    return {"x": x, "grad_g": gg, "grad_kp": gk}
