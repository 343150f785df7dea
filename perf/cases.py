"""Performance cases of the ReaxFF engine: what its users have it do, from the 24-atom force call to the 192,000-atom MD run.

Every case goes through the public entry points (reaxamd.Engine, reaxamd.serving) with seeded synthetic systems of this
repository's own workloads (reaxamd.systems): liquid water, CH4 : O2 = 1 : 2 gas, random carbon. Kinds:

  force    one step of an external MD program (the LAMMPS plugin's calls): new positions, the charge update with its history,
           energies, gradient and virial (with per-atom tallies where the program writes them)
  charges  the charges of new positions from no history, solved tightly
  md       a chunk of the engine's own MD loop, then the state a program writes out
  pack     the same for many independent systems in one context
  request  one whole request of the server: a system's setup, its MD and its results
"""
import math
import os
import random
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "metal-reax_amd"))

import reaxamd  # noqa: E402
from reaxamd import serving, systems  # noqa: E402

FIELDS = {"water": "ffield.cho_standin", "gas": "ffield.cho_standin", "carbon": "ffield.C2013"}
PERIOD = 16   # positions of a force case's trajectory
EQUIL = 100   # steps from the generated start before an MD case's state is handed over


def listed():
    return [
        # the smallest unit cell a plugin user evaluates, in the default (FP64) precision: launches and round trips only
        {"name": "force_water_24_fp64", "kind": "force", "system": "water", "size": 2, "precision": "fp64", "peratom": False},
        # a small gas cell in single precision whose program dumps per-atom energies and virials
        {"name": "force_gas_450_fp32_peratom", "kind": "force", "system": "gas", "size": 50, "precision": "fp32", "peratom": True},
        # a mid-sized, odd-sided liquid cell driven by an external program in the GPU default (mixed) precision
        {"name": "force_water_6591_mixed", "kind": "force", "system": "water", "size": 13, "precision": "mixed", "peratom": False},
        # the large plugin step in the reference's default (FP64) precision
        {"name": "force_water_24000_fp64", "kind": "force", "system": "water", "size": 20, "precision": "fp64", "peratom": False},
        # charges alone, tight, from no history: a new configuration's first solve, and the check of a running one
        {"name": "charges_water_3000_mixed", "kind": "charges", "system": "water", "size": 10, "precision": "mixed"},
        # the small water workload (648 atoms): the latency of a step
        {"name": "md_water_648_mixed", "kind": "md", "system": "water", "size": 6, "precision": "mixed", "steps": 100},
        # an odd-sided liquid in FP64
        {"name": "md_water_10125_fp64", "kind": "md", "system": "water", "size": 15, "precision": "fp64", "steps": 25},
        # the main workload of the benchmark
        {"name": "md_water_24000_mixed", "kind": "md", "system": "water", "size": 20, "precision": "mixed", "steps": 25},
        # the random-carbon workload: bonded terms and list churn, charges fixed
        {"name": "md_carbon_30000_mixed", "kind": "md", "system": "carbon", "size": 30000, "precision": "mixed", "steps": 25},
        # a large box (32-bit columns)
        {"name": "md_water_192000_mixed", "kind": "md", "system": "water", "size": 40, "precision": "mixed", "steps": 4},
        # batched small systems (100 to 3000 atoms, half water, half gas) advanced together
        {"name": "pack_40_mixed", "kind": "pack", "count": 40, "nmax": 3000, "precision": "mixed", "steps": 20},
        # one gas request of the server on a kept context
        {"name": "request_gas_1503_mixed", "kind": "request", "system": "gas", "size": 167, "precision": "mixed", "steps": 40},
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    precision = rng.choice(("fp64", "mixed", "mixed", "fp32"))
    kind = rng.choice(("force", "force", "force", "charges", "md", "md", "md", "md", "pack", "request"))
    if kind == "pack":
        return {"kind": kind, "count": between(4, 48), "nmax": between(300, 3000), "precision": precision, "steps": between(4, 24)}
    system = rng.choice(("water", "water", "gas", "carbon") if kind == "md" else ("water", "water", "gas"))
    top = 40 if kind == "md" else 20 if kind == "force" else 13
    size = between(2, top) if system == "water" else between(11, 700) if system == "gas" else between(1000, 30000)
    case = {"kind": kind, "system": system, "size": size, "precision": precision}
    if kind == "force":
        case["peratom"] = rng.random() < 0.25
    if kind in ("md", "request"):
        atoms = _atoms(case)
        case["steps"] = max(2, min(between(10, 100), 500000 // atoms))
    return case


def _atoms(case):
    if case["kind"] == "pack":
        return sum(3 * k ** 3 if kind == "water" else 9 * k for kind, k in _pack_sizes(case))
    return {"water": 3 * case["size"] ** 3, "gas": 9 * case["size"], "carbon": case["size"]}[case["system"]]


def _pack_sizes(case):
    """(kind, size) of a pack's members: atoms log-uniform in [100, nmax], alternately water and gas; fixed by the case."""
    rng = random.Random(case["count"])
    out = []
    for k in range(case["count"]):
        n = math.exp(rng.uniform(math.log(100), math.log(case["nmax"])))
        out.append(("water", max(2, round((n / 3) ** (1 / 3)))) if k % 2 == 0 else ("gas", max(1, round(n / 9))))
    return out


def _system(kind, size, seed):
    if kind == "water":
        return systems.water_box(size, seed=seed)
    if kind == "gas":
        return systems.ch4_o2_gas(9 * size, density=0.3, seed=seed)
    return systems.random_carbon(size, density=1.0, dmin=1.2, seed=seed)


def _field(kind):
    return systems.load_ffield(os.path.join(REPO, "tests", "golden", FIELDS[kind]))


def _engine(case, kind):
    e = reaxamd.Engine(0)
    e.pair_style(["NULL", "precision", case["precision"]] + (["checkqeq", "no"] if kind == "carbon" else []))
    e.pair_coeff(_field(kind), ["C"] if kind == "carbon" else list(systems.ELEMENTS))
    return e


def _charges_on(e):
    e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))


def _trajectory(w, seed):
    """Positions along a smooth closed path: each atom swings about its place at thermal speed (300 K, dt 0.25 fs)."""
    v = systems.maxwell_boltzmann(w.masses(), 300.0, seed=seed + 1)
    a = v * 0.25 * PERIOD / (2 * math.pi)
    return [np.ascontiguousarray(w.x + a * math.sin(2 * math.pi * k / PERIOD)) for k in range(PERIOD)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "request":
        w = _system(case["system"], case["size"], seed)
        req = serving.Request(rid=0, system=w, steps=case["steps"], t_target=2500.0, dt=0.1, seed=seed + 1)
        return {"case": case, "engine": _engine(case, case["system"]), "request": req, "field": _field(case["system"])}
    if kind in ("force", "charges"):
        w = _system(case["system"], case["size"], seed)
        e = _engine(case, case["system"])
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        _charges_on(e)
        return {"case": case, "engine": e, "path": _trajectory(w, seed), "at": 0}
    # MD: from the generated start with strong coupling first, then the run's own thermostat
    e = _engine(case, "water" if kind == "pack" else case["system"])
    carbon = kind == "md" and case["system"] == "carbon"
    hot = 4000.0 if carbon else 2500.0 if kind == "pack" or case["system"] == "gas" else 300.0
    if kind == "pack":
        members = [_system(s, size, 1000 * seed + k) for k, (s, size) in enumerate(_pack_sizes(case))]
        e.set_systems(members)
        v = np.concatenate([systems.maxwell_boltzmann(m.masses(), hot, seed=seed + 1) for m in members])
    else:
        w = _system(case["system"], case["size"], seed)
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        v = systems.maxwell_boltzmann(w.masses(), hot, seed=seed + 1)
    masses = np.array([0.0, systems.MASS["C"]] if carbon else [0.0] + [systems.MASS[el] for el in systems.ELEMENTS])
    if not carbon:
        _charges_on(e)
    how = {"dt": 0.1 if hot == 2500.0 else 0.25, "t_target": hot, "skin": 2.0, "qeq_every": 0 if carbon else 1, "qeq_imax": 200,
           "qeq_tol": 1e-6}
    e.md_setup(v, masses, t_damp=5.0, **how)
    e.md_run(EQUIL)
    e.md_setup(e.state()[1], masses, t_damp=25.0, **how)
    return {"case": case, "engine": e}


def run(state):
    case, e = state["case"], state["engine"]
    kind = case["kind"]
    if kind == "request":
        return serving.run_one(e, state["field"], state["request"], case["precision"])
    if kind in ("force", "charges"):
        e.set_positions(state["path"][state["at"]])
        state["at"] = (state["at"] + 1) % PERIOD
        # (the relative residual a solve stops at is not kept: it is what rounding leaves of a difference)
        if kind == "charges":
            e.qeq_reset_history()
            q, iters, _ = e.qeq_charges(imax=1000, tol=1e-10)
            return {"charges": q, "iters": iters}
        q, iters, _ = e.qeq_charges()
        return dict(e.compute(peratom=case["peratom"]), charges=q, iters=iters)
    thermo = e.md_run(case["steps"])
    x, v, q = e.state()
    out = {"positions": x, "velocities": v, "charges": q, "thermo": thermo}
    if kind == "pack":
        out["systems"] = e.system_results()
    return out


def work(case):
    """The list-based model of a step (bench.py): per atom its state, gradient and energies; the half matrix of the pairs within
    10 A written once and read once per product (two systems per product); the bonds' state. Operations: the pair terms, the
    matrix entries and the products."""
    n = _atoms(case)
    steps = case.get("steps", 1)
    carbon = case.get("system") == "carbon"
    dens = {"water": 0.1003, "gas": 0.0203, "carbon": 0.0501}
    if case["kind"] == "pack":
        half = sum((3 * k ** 3 if s == "water" else 9 * k) * dens[s] for s, k in _pack_sizes(case)) / n
    else:
        half = dens[case["system"]]
    n_f = 0.5 * half * 4.0 / 3.0 * math.pi * 1000.0
    word = 8 if case["precision"] == "fp64" else 4
    products = 0 if carbon else {"charges": 30, "force": 8}.get(case["kind"], 8)
    matrix = 0 if carbon else (word + 4) * n_f * (1 + products)
    state = 200.0 + 4 * n_f + 240.0 * 3
    flops = n_f * (80.0 + (0 if carbon else 40.0 + 8.0 * products)) + 3000.0
    if case["kind"] == "charges":
        state, flops = 24.0 + 4 * n_f, n_f * (40.0 + 8.0 * products)
    return {"bytes": n * steps * (state + matrix), "flops": n * steps * flops}


# ---- the same in 64 bits, from the formulas: charges, van der Waals, Coulomb and polarisation energies ---------------------------
def _parameters():
    """General parameters and the elements' and pairs' non-bonded parameters of the C/H/O field."""
    lines = _field("water").splitlines()
    gp = [float(line.split()[0]) for line in lines[2:2 + int(lines[1].split()[0])]]
    at = 2 + len(gp)
    nt = int(lines[at].split()[0])
    at += 4
    rows = [[lines[at + 4 * k + r].split() for r in range(4)] for k in range(nt)]
    el = {"r": [float(r[0][4]) for r in rows], "eps": [float(r[0][5]) for r in rows], "gamma": [float(r[0][6]) for r in rows],
          "alpha": [float(r[1][0]) for r in rows], "gw": [float(r[1][1]) for r in rows], "chi": [float(r[1][5]) for r in rows],
          "eta": [2.0 * float(r[1][6]) for r in rows]}
    el = {k: torch.tensor(v, dtype=torch.float64) for k, v in el.items()}
    mix = {"D": torch.sqrt(torch.outer(el["eps"], el["eps"])), "rv": 2.0 * torch.sqrt(torch.outer(el["r"], el["r"])),
           "alpha": torch.sqrt(torch.outer(el["alpha"], el["alpha"])), "gw": torch.sqrt(torch.outer(el["gw"], el["gw"])),
           "shield": torch.outer(el["gamma"], el["gamma"]) ** -1.5}
    at += 4 * nt
    at += 2 + 2 * int(lines[at].split()[0])
    for line in lines[at + 1:at + 1 + int(lines[at].split()[0])]:
        f = line.split()
        for i, j in ((int(f[0]) - 1, int(f[1]) - 1), (int(f[1]) - 1, int(f[0]) - 1)):
            for key, value in (("D", float(f[2])), ("rv", 2.0 * float(f[3])), ("alpha", float(f[4]))):
                if value > 0:
                    mix[key][i, j] = value
    return gp, el, mix


def _taper(r, cut):
    x = r / cut
    return 1.0 + x ** 4 * (-35.0 + x * (84.0 + x * (-70.0 + 20.0 * x)))


def exact(case, seed):
    if case["kind"] not in ("force", "charges") or _atoms(case) > 8000:
        return None
    w = _system(case["system"], case["size"], seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gp, el, mix = _parameters()
    cut, p = gp[12], gp[28]
    t = torch.tensor(w.types.astype(np.int64) - 1, device=dev)
    mix = {k: v.to(dev) for k, v in mix.items()}
    box = torch.tensor(w.hi - w.lo, dtype=torch.float64, device=dev)
    x = torch.tensor(_trajectory(w, seed)[0], dtype=torch.float64, device=dev)
    x = x - torch.floor(x / box) * box
    n = len(t)
    H = torch.zeros((n, n), dtype=torch.float64, device=dev)   # Coulomb matrix without its unit, all images
    e_vdw = 0.0
    reach = [int(math.ceil(cut / float(b))) for b in box]
    shifts = [(a, b, c) for a in range(-reach[0], reach[0] + 1) for b in range(-reach[1], reach[1] + 1)
              for c in range(-reach[2], reach[2] + 1)]
    for lo in range(0, n, 1024):
        hi = min(n, lo + 1024)
        for s in shifts:
            image = x + torch.tensor(s, dtype=torch.float64, device=dev) * box
            r = torch.sqrt(sum((image[None, :, d] - x[lo:hi, None, d]) ** 2 for d in range(3)))
            i, j = torch.nonzero((r <= cut) & (r > 1e-8), as_tuple=True)
            if not len(i):
                continue
            r = r[i, j]
            ti, tj, tap = t[lo + i], t[j], _taper(r, cut)
            H[lo + i, j] += tap / (r ** 3 + mix["shield"][ti, tj]) ** (1.0 / 3.0)
            f = (r ** p + mix["gw"][ti, tj] ** -p) ** (1.0 / p)
            a = mix["alpha"][ti, tj] * (1.0 - f / mix["rv"][ti, tj])
            e_vdw += float((0.5 * tap * mix["D"][ti, tj] * (torch.exp(a) - 2.0 * torch.exp(0.5 * a))).sum())
    H, t = H.cpu(), t.cpu()
    b = torch.stack([-el["chi"][t], -torch.ones(n, dtype=torch.float64)], 1)
    st = torch.linalg.solve(14.4 * H + torch.diag(el["eta"][t]), b)
    q = st[:, 0] - st[:, 0].sum() / st[:, 1].sum() * st[:, 1]
    out = {"charges": q.numpy(), "iters": None}
    if case["kind"] == "force":
        e = {k: None for k in reaxamd.TERMS}
        e.update(e_vdW=e_vdw, e_ele=float(0.5 * 332.06371 * (q @ (H @ q))),
                 e_pol=float((23.02 * (el["chi"][t] * q + 0.5 * el["eta"][t] * q * q)).sum()))
        out.update(energy=e, grad=None, virial=None)
        if case["peratom"]:
            out.update(eatom=None, vatom=None)
    return out
