"""What a user of the engine has it do on the GPU, as cases with inputs, one pass
through the public entry points, and the work that pass cannot do without.

A case names a kind of call and its sizes; the devices are the n-FinFETs of
decks/make_finfet.py (mesh lines per nm, gate length, fin width, carriers, bias),
the shipped FinFET deck, and a box of bulk silicon.  The kinds:

  step      Engine.step: deposit, Poisson solve, fields, flight; the transient
  heat      Engine.heat_step: the heating phase (no solve, heat tallied)
  batch     Batch.step: a bias sweep of devices sharing the mesh
  bulk      fly_step in a uniform field: transport in bulk silicon
  deposit   Engine.deposit: the tallies of a population, on the host
  seams     the step taken through its separate entry points with host arrays
  poisson   one solve with host vectors, cold or warm, in each of its forms
  qc        Engine.qc_potential: the quantum correction of a host potential
"""
import ctypes
import math
import os
import sys
import tempfile

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "c-mc_electron_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import emcgpu  # noqa: E402
from emcgpu import abi  # noqa: E402


# ---------------------------------------------------------------- the cases
def _finfet(name, kind, refine, electrons, holes, lg=15, wfin=5, vd=0.5, vg=0.7, **kw):
    return {"name": name, "kind": kind, "refine": refine, "electrons": electrons, "holes": holes, "lg": lg,
            "wfin": wfin, "vd": vd, "vg": vg, **kw}


def listed():
    return [
        # the smallest device of the tests and sweeps: a step is a chain of short kernels
        _finfet("step_20x40x12", "step", 1, 20000, 2000, steps=20, relax=100, phims=-0.46),
        # the benchmark's device, the largest here: two million carriers, 639 k nodes
        _finfet("step_80x160x48", "step", 4, 2000000, 500000, steps=10, relax=30, phims=-0.46),
        # the shipped deck: 50 x 64 x 28 cells of uneven width, 766 k carriers and
        # more after each refresh; fifty steps hold one MultipleRefresh
        {"name": "step_shipped_deck", "kind": "step", "deck": "finfet_shipped", "steps": 50, "relax": 50},
        # a step with the quantum correction, and the solve in FP64 throughout
        _finfet("step_quantum_40x72x22", "step", 2, 60000, 6000, lg=11, wfin=4, steps=5, relax=20, phims=-0.46,
                qc=True, fp32=0),
        # the heating phase: flight and deposit without a solve, heat tallied
        _finfet("heat_60x138x42", "heat", 3, 300000, 30000, lg=21, wfin=7, steps=20, relax=20, phims=-0.46),
        # bias points of one mesh stepped as one batch, electrons by bias
        _finfet("sweep_16x_20x40x12", "batch", 1, 50000, 5000, electrons_high=500000, points=16, steps=10, relax=20,
                phims=0.3),
        # drift in bulk silicon at 100 kV/cm: many scattering events a step, and
        # the population read back for its means
        {"name": "bulk_100kV", "kind": "bulk", "cells": 8, "cell_nm": 4, "carriers": 100000, "dt": 2e-15,
         "field": 1e7, "steps": 5},
        # the tallies of one population as host arrays
        _finfet("deposit_40x86x26", "deposit", 2, 250000, 25000, lg=18, wfin=6, phims=-0.46),
        # the solver seams with the host's vectors in between
        _finfet("seams_40x80x24", "seams", 2, 50000, 5000, relax=5, phims=-0.46),
        # one solve from zero on a mesh of odd sizes
        _finfet("poisson_cold_60x126x33", "poisson", 3, 60000, 6000, lg=17, wfin=4, form="cold", phims=-0.46),
        # one small solve from the last potential, without allocation (a serving loop)
        _finfet("poisson_warm_20x35x11", "poisson", 1, 20000, 2000, lg=10, wfin=4, form="noalloc", phims=-0.46),
        # the effective potential of a given potential
        _finfet("quantum_60x120x36", "qc", 3, 1000, 100, phims=-0.46),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: meshes of 20 x 35 x 11 to 60 x 165 x 45 cells, 10 k to 600 k
    electrons, gate lengths of 10 to 30 nm and fins of 4 to 8 nm, as the serving
    and sweep workloads take them."""
    kind = rng.choice(["step", "step", "step", "heat", "batch", "bulk", "deposit", "seams", "poisson", "poisson", "qc"])
    if kind == "bulk":
        return {"kind": kind, "cells": rng.randint(2, 12), "cell_nm": rng.randint(2, 6),
                "carriers": _log_int(rng, 8000, 200000), "dt": rng.choice([1e-16, 5e-16, 2e-15]),
                "field": 10 ** rng.uniform(5, 7.3), "steps": rng.randint(1, 8)}
    refine = 1 if kind == "batch" else rng.choice([1, 1, 2, 2, 3])
    electrons = _log_int(rng, 10000, 600000 if kind in ("step", "heat", "deposit") else 100000)
    c = {"kind": kind, "refine": refine, "electrons": electrons, "holes": max(200, electrons // 10),
         "lg": rng.randint(10, 30), "wfin": rng.randint(4, 8), "vd": round(rng.uniform(0.05, 0.8), 3),
         "vg": round(rng.uniform(0.0, 0.8), 3), "phims": rng.choice([-0.46, 0.3])}
    if kind == "step":
        c.update(steps=rng.randint(2, 12), relax=rng.randint(5, 40), fp32=rng.choice([2, 2, 2, 0, 1]),
                 qc=refine < 3 and rng.random() < 0.2)
    elif kind == "heat":
        c.update(steps=rng.randint(5, 20), relax=rng.randint(5, 20))
    elif kind == "batch":
        c.update(points=rng.randint(3, 20), steps=rng.randint(3, 10), relax=10, electrons_high=4 * electrons)
    elif kind == "seams":
        c.update(relax=rng.randint(2, 8))
    elif kind == "poisson":
        c.update(form=rng.choice(["cold", "warm", "noalloc", "mixed", "fp64"]))
    return c


# ---------------------------------------------------------------- decks and engines
# The band tables are built once per process and shared while any engine holds
# them: a program that runs device after device keeps one engine for them.
_TABLES = {}


def _keep_tables(qc):
    if qc not in _TABLES:
        d = tempfile.mkdtemp(prefix="emc_tables_")
        _TABLES[qc] = emcgpu.Engine(emcgpu.write_deck(d, refine=1, electrons=100, holes=10, qc=int(qc)), device=0)


def _deck(case, **kw):
    args = dict(refine=case["refine"], electrons=case["electrons"], holes=case["holes"], lg=case["lg"],
                wfin=case["wfin"], vd=case["vd"], vg=case["vg"], phims=case["phims"], total_step=100000,
                stat_step=1000, qc=int(case.get("qc", case["kind"] == "qc")), quantum_start_step=0)
    args.update(kw)
    return emcgpu.write_deck(tempfile.mkdtemp(prefix="emc_case_"), **args)


def _bulk_deck(case):
    """A periodic box of lightly doped silicon; its one contact is not used."""
    n, h = case["cells"], case["cell_nm"]
    d, L = tempfile.mkdtemp(prefix="emc_case_"), n * h
    with open(os.path.join(d, "lgrid.txt"), "w") as f:
        for _ in range(3):
            f.write("%d\n" % (n + 1))
            f.writelines("%.10g\n" % (q * h * 1e-3) for q in range(n + 1))
    with open(os.path.join(d, "ldg.txt"), "w") as f:
        f.write(f"""default_par_number 1 1
region 0 {L} 0 {L} 0 {L} SILICON
donor 0 {L} 0 {L} 0 {L} 1e21
acceptor 0 {L} 0 {L} 0 {L} 0
motioncube 0 {L} 0 {L} 0 {L} PASS PASS PASS PASS PASS PASS
motionplane 0 0 0 {L} 0 {L} UP PERIOD
motionplane {L} {L} 0 {L} 0 {L} DOWN PERIOD
motionplane 0 {L} 0 0 0 {L} LEFT PERIOD
motionplane 0 {L} {L} {L} 0 {L} RIGHT PERIOD
motionplane 0 {L} 0 {L} 0 0 FRONT PERIOD
motionplane 0 {L} 0 {L} {L} {L} BACK PERIOD
contact
  1 0
  0 {L} 0 0 0 {L}
  0
end
""")
    with open(os.path.join(d, "input.txt"), "w") as f:
        f.write(f"""gridFile=lgrid.txt
device_file_name=ldg.txt
total_step=100000
ElectronNumber={case['carriers']}
HoleNumber={case['carriers'] // 2}
Temperature=300
dt={case['dt']:g}
stat_step=1000
stat_heat_step=1000
heat_steps=0
Flag_QuantumCorrection=0
Flag_MultipleRefresh=0
Flag_compute_heat=0
Flag_SurfaceScatter=0
mr_step=10
""")
    return os.path.join(d, "input.txt")


class State:
    """An engine or batch and what the program holds beside it."""

    def __init__(self, case):
        self.case, self.kind, self.eng, self.at = case, case["kind"], None, 0

    def __del__(self):
        for e in [getattr(self, "batch", None)] + list(getattr(self, "engines", [])) + [self.eng]:
            if e is not None:
                e.close()


def _engine(inp, seed, **kw):
    return emcgpu.Engine(inp, device=0, seed=1 + seed, **kw)


def prepare(case, seed):
    s = State(case)
    kind = s.kind
    _keep_tables(bool(case.get("qc", kind == "qc")))
    rng = np.random.default_rng(seed)
    if kind == "bulk":
        s.eng = _engine(_bulk_deck(case), seed)
        s.eng.particles_init()
        m = s.eng.mesh
        f = emcgpu.CellFieldArrays(m.ncell)
        # V/m along a direction of the seed, in the engine's units
        v = rng.normal(size=3)
        v *= case["field"] / m.field0 / np.linalg.norm(v)
        for a, b, x in (("ex", "hx", v[0]), ("ey", "hy", v[1]), ("ez", "hz", v[2])):
            getattr(f, a)[:] = x
            getattr(f, b)[:] = x
        f.rho[:] = 0.5 * s.eng.mesh_arrays()["da"]
        s.eng.fields_set(f)
        return s
    if kind == "batch":
        # bias points of a sweep: the electrons grow with the gate voltage
        k = case["points"]
        s.engines = []
        for q in range(k):
            g = q / max(1, k - 1)
            ne = int(case["electrons"] + (case["electrons_high"] - case["electrons"]) * g)
            inp = _deck(case, electrons=ne, holes=ne // 10, vg=0.8 * g, vd=0.05 + 0.75 * ((q * 5) % k) / k)
            e = _engine(inp, seed * 64 + q)
            s.engines.append(e)
            e.particles_init()
        s.batch = emcgpu.Batch(s.engines)
        s.batch.step(case["relax"])
        return s
    if "deck" in case:
        inp = os.path.join(emcgpu.DECK_DIR, case["deck"], "input.txt")
    else:
        inp = _deck(case)
    fp32 = {"fp64": 0, "mixed": 1}.get(case.get("form"), case.get("fp32"))
    s.eng = e = _engine(inp, seed, poisson_fp32=fp32)
    if kind == "qc":
        # a potential like a solved one: a drop along y, the channel, noise
        m = e.mesh
        j, i, k = np.meshgrid(np.arange(m.pny), np.arange(m.pnx), np.arange(m.pnz), indexing="ij")
        ph = rng.uniform(0, 2 * np.pi, 3)
        s.pot = (rng.uniform(5, 25) * j / m.pny + 4 * np.sin(2 * np.pi * i / m.pnx + ph[0]) +
                 3 * np.cos(2 * np.pi * k / m.pnz + ph[1]) + 0.1 * rng.normal(size=j.shape)).reshape(-1)
        return s
    e.particles_init()
    if kind == "poisson":
        s.rhs = e.rhs_from_charge(e.deposit()[0])
        s.x0 = None
        if case["form"] != "cold":
            # the solution of the charge a few steps before
            s.x0 = e.poisson_solve(s.rhs)[0]
            e.step(2)
            s.rhs = e.rhs_from_charge(e.deposit()[0])
        return s
    if kind != "deposit":
        e.step(case["relax"])
        e.tallies_reset()
    if kind == "heat":
        e.step(5)  # the window whose mean potential the phase runs in
        e.heat_begin()
        e.tallies_reset()
    if kind == "seams":
        s.pot = e.potential()
        s.at = case["relax"]
    return s


# ---------------------------------------------------------------- one pass
def _tallies(t):
    """The counts of a step as they are, its contact sums in physical units."""
    c = np.ctypeslib.as_array(t.contact)
    return {"counts": np.array([t.n_catch, t.n_gen, t.n_phonon, t.n_impurity, t.n_events, t.n_mr_gen]),
            "drops": np.array(t.drops), "contact_n": c[:, [0, 3]].copy(), "contact_sums": c[:, [1, 2, 4]] / abi.FX_CONTACT}


def run(state):
    s, case, e = state, state.case, state.eng
    if s.kind == "step":
        t = e.step(case["steps"])
        r, lc = e.currents()
        return {"tallies": _tallies(t), "potential": e.potential(), "r": r / abi.FX_CONTACT, "l": lc / abi.FX_CONTACT}
    if s.kind == "heat":
        t = e.heat_step(case["steps"])
        w = e.stat_window()
        return {"tallies": _tallies(t), "heat_e": w["heat_e"] / abi.FX_HEAT, "heat_h": w["heat_h"] / abi.FX_HEAT,
                "cell_count": w["cell_count"], "r": w["rcur"] / abi.FX_CONTACT, "l": w["lcur"] / abi.FX_CONTACT}
    if s.kind == "batch":
        t = [_tallies(t) for t in s.batch.step(case["steps"])]
        out = {k: np.stack([x[k] for x in t]) for k in t[0]}
        out["potential"] = np.stack([q.potential() for q in s.engines])
        return out
    if s.kind == "bulk":
        t = [_tallies(e.fly_step(s.at + q))["counts"] for q in range(case["steps"])]
        s.at += case["steps"]
        p = e.download()
        out = {f: getattr(p, f) for f in abi.PARTICLE_F64 + abi.PARTICLE_I32}
        return {"counts": np.stack(t), **out}
    if s.kind == "deposit":
        q, st, cq, cn = e.deposit()
        return {"node_q": q, "node_stat": st, "cell_q": cq, "cell_n": cn}
    if s.kind == "seams":
        q, _, cq, _ = e.deposit()
        rhs = e.rhs_from_charge(q)
        s.pot = e.poisson_solve(rhs, x0=s.pot)[0]
        m = e.mesh_arrays()
        rho = np.maximum(cq[2 * e.mesh.ncell:] / abi.FX_Q / m["cvol"], 0.5 * m["da"])
        f = e.compute_field(s.pot, rho)
        t = e.fly_step(s.at)
        s.at += 1
        return {"potential": s.pot, "tallies": _tallies(t), **{k: getattr(f, k) for k in abi.CELL_FIELDS}}
    if s.kind == "poisson":
        if case["form"] == "mixed":
            return e.poisson_solve_mixed(s.rhs, s.x0)[0]
        if case["form"] == "noalloc":
            return e.poisson_solve_noalloc(s.rhs, s.x0)[0]
        return e.poisson_solve(s.rhs, s.x0)[0]
    return e.qc_potential(s.pot)


# ---------------------------------------------------------------- the work of a pass
def _sizes(case):
    """(nodes, cells, carriers, nodes of the quantum region) of a device, the
    carriers as sampled (the deck's counts and one of each type per silicon cell)."""
    if case["kind"] == "bulk":
        n = case["cells"]
        return (n + 1) ** 3, n ** 3, 1.5 * case["carriers"], 0
    if "deck" in case:
        return 51 * 65 * 29, 50 * 64 * 28, 1000000, 0
    r, ly, w = case["refine"], case["lg"] + 25, case["wfin"]
    nx, ny, nz = 20 * r, ly * r, (w + 7) * r
    si = r ** 3 * ly * (10 * w + 9 * (w + 7))
    return ((nx + 1) * (ny + 1) * (nz + 1), nx * ny * nz, case["electrons"] + case["holes"] + 2 * si,
            (10 * r + 1) * (ly * r + 1) * (w * r + 1))


def _qc_terms(case):
    """Source nodes in the window of one target (4 standard deviations of 0.5 nm on
    each side, and the node beyond)."""
    r = case["refine"]
    return (4 * r + 2) ** 2 * (4 * r + 2)


def work(case):
    nn, nc, npart, nq = _sizes(case)
    # a carrier's state read and written; the deposit reads its position, charge,
    # energy, cell and state again
    fly = (152 * npart, 300.0 * npart)
    dep = (44 * npart + 8 * (11 * nn + 4 * nc), 200.0 * npart)
    # a solve reads right-hand side, start and operator once and writes the solution;
    # its operations: the matrix and the cycle of each of six iterations
    sol = (8 * 8 * nn, 6 * 120.0 * nn)
    fld = (8 * nn + 8 * 8 * nc, 150.0 * nc)
    qc = (16 * nn, 5.0 * nq * _qc_terms(case)) if case.get("qc") or case["kind"] == "qc" else (0, 0)
    kind = case["kind"]
    if kind == "bulk":
        parts, k, once = [fly], case["steps"], 90 * npart
    elif kind == "heat":
        parts, k, once = [fly, dep, fld], case["steps"], 8 * 4 * nn
    elif kind == "deposit":
        parts, k, once = [dep], 1, 0
    elif kind == "poisson":
        parts, k, once = [sol], 1, 0
    elif kind == "qc":
        parts, k, once = [qc], 1, 0
    elif kind == "batch":
        n = case["points"]
        mean = npart + 0.55 * (case["electrons_high"] - case["electrons"])
        parts = [(152 * n * mean, 300.0 * n * mean), (44 * n * mean + 8 * n * (11 * nn + 4 * nc), 200.0 * n * mean),
                 (n * sol[0], n * sol[1]), (n * fld[0], n * fld[1])]
        k, once = case["steps"], 8 * n * nn
    else:
        parts, k, once = [fly, dep, sol, fld, qc], case.get("steps", 1), 8 * nn
    return {"bytes": float(k * sum(p[0] for p in parts) + once), "flops": float(k * sum(p[1] for p in parts))}


# ---------------------------------------------------------------- in 64 bits
_MATERIAL = {"oxide": 2, "silicon": 3}  # as the mesh view numbers them
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_DEV)


def _exact_poisson(m, ma, rhs):
    """Conjugate gradients to 1e-14 on the seven-point operator, diagonal scaling."""
    shp = (m.pny, m.pnx, m.pnz)
    b = _t(rhs).reshape(shp)
    diag, cx, cy, cz = (_t(ma[k]).reshape(shp) for k in ("diag", "cx", "cy", "cz"))
    free = torch.tensor(np.array(ma["node_kind"]) == 0, device=_DEV).reshape(shp)

    def op(x):
        y = diag * x
        for c, ax in ((cy, 0), (cx, 1), (cz, 2)):
            n = x.shape[ax] - 1
            w = c.narrow(ax, 0, n)
            y.narrow(ax, 0, n).add_(w * x.narrow(ax, 1, n))
            y.narrow(ax, 1, n).add_(w * x.narrow(ax, 0, n))
        return y

    x = torch.where(free, torch.zeros_like(b), b)
    r = torch.where(free, b - op(x), torch.zeros_like(b))
    d = torch.where(free, 1.0 / diag, torch.zeros_like(b))
    z = d * r
    p, rz, stop = z.clone(), (r * z).sum(), 1e-14 * float(b.norm())
    for it in range(4000):
        q = torch.where(free, op(p), torch.zeros_like(p))
        a = rz / (p * q).sum()
        x += a * p
        r -= a * q
        if it % 20 == 0 and float(r.norm()) <= stop:
            break
        z = d * r
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x.reshape(-1).cpu().numpy()


def _exact_qc(m, ma, pot):
    """The effective potential, one axis after another: for each of the four box
    shapes that a source can have on an axis, a matrix of erf differences."""
    nx, ny, nz = m.pnx, m.pny, m.pnz
    cell = lambda a: np.asarray(a).reshape(m.cny, m.cnx, m.cnz)  # noqa: E731

    def corners(mask):
        out = np.zeros((ny, nx, nz), bool)
        for j in (0, 1):
            for i in (0, 1):
                for k in (0, 1):
                    out[j:j + m.cny, i:i + m.cnx, k:k + m.cnz] |= mask
        return out

    mat = cell(ma["material"])
    si, ox = corners(mat == _MATERIAL["silicon"]), corners(mat == _MATERIAL["oxide"])
    solid, region = si | ox, corners(cell(ma["qcregion"]) != 0)
    v = np.where(solid, pot.reshape(ny, nx, nz) - np.where(ox & ~si, m.qc_eb, 0.0), 0.0)
    src = _t(v)
    shape, mats = [], []
    for ax, (l, dl, q) in enumerate(((ma["ly"], ma["dy"], 1), (ma["lx"], ma["dx"], 0), (ma["lz"], ma["dz"], 2))):
        th, r, n = m.qc_theta[q], m.qc_ratio[q] * m.qc_theta[q], len(l)
        edge = np.zeros((ny, nx, nz), bool)
        lo, hi = edge.copy(), edge.copy()
        at = lambda a, b: tuple(slice(a, b) if x == ax else slice(None) for x in range(3))  # noqa: E731
        lo[at(0, 1)] = True
        lo[at(1, None)] = ~solid[at(0, -1)]
        hi[at(-1, None)] = True
        hi[at(0, -1)] = ~solid[at(1, None)]
        shape.append(torch.tensor(lo.astype(np.int64) + 2 * hi, device=_DEV))
        # the window of each target: from the node before the first one within r
        # to the first one beyond
        w = np.zeros((n, n), bool)
        a = 0
        for p in range(n):
            a = a + int(np.searchsorted(l[a:max(a, p)], l[p] - r, side="left"))
            b = int(np.searchsorted(l, l[p] + r, side="right"))
            a = max(0, a - 1)
            w[p, a:min(b, n - 1) + 1] = True
        below = np.concatenate(([0.0], dl)) * 0.5
        above = np.concatenate((dl, [0.0])) * 0.5
        s2 = math.sqrt(2.0) * th
        tgt = _t(l)[:, None] / s2
        for c in range(4):
            e1 = _t(l - r if c & 1 else l - below) / s2
            e2 = _t(l + r if c & 2 else l + above) / s2
            d = torch.erf(e2[None, :] - tgt) - torch.erf(e1[None, :] - tgt)
            mats.append(torch.where(torch.tensor(w, device=_DEV), d, torch.zeros_like(d)))
    out = torch.zeros_like(src)
    zero = torch.zeros_like(src)
    for cy in range(4):
        for cx in range(4):
            for cz in range(4):
                here = (shape[0] == cy) & (shape[1] == cx) & (shape[2] == cz)
                x = torch.where(here, src, zero)
                x = torch.tensordot(mats[cy], x, dims=([1], [0]))
                x = torch.tensordot(mats[4 + cx], x, dims=([1], [1])).permute(1, 0, 2)
                out += torch.tensordot(x, mats[8 + cz], dims=([2], [1]))
    got = 0.125 * out.cpu().numpy()
    return np.where(region, got, pot.reshape(ny, nx, nz)).reshape(-1)


def exact(case, seed):
    """The solves and the effective potential on the mesh the engine lays out, in
    plain torch; the other cases follow single carriers through random draws."""
    if case["kind"] not in ("poisson", "qc"):
        return None
    s = prepare(case, seed)
    m, ma = s.eng.mesh, {k: np.array(v) for k, v in s.eng.mesh_arrays().items()}
    return _exact_poisson(m, ma, s.rhs) if s.kind == "poisson" else _exact_qc(m, ma, s.pot)
