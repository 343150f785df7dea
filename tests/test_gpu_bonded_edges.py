"""Bonded kernels at the edges of their work splits, FP64 and mixed, against the FP64 oracle: dense carbon (diamond with random
displacements: 94 atoms within bond_cut, so that numbers within bond_cut pass 64 and share places in the sums, 4 to 6 bonds per
atom, several hundred torsions per wave) at sizes below and above the line where a wave takes several atoms, with the last wave
partly filled, and atom counts around a wave.

Bars as tests/test_gpu_variants.py: FP64 each term within 1e-9 of max(1, |E|), gradient within 1e-7 kcal/mol/A; mixed 1e-4
kcal/mol per atom and 4e-3 / 9e-4 kcal/mol/A (largest, RMS). Those hold for forces of the order of 100 kcal/mol/A; rounding grows
with the terms, so the gradient bars are scaled by the largest reference gradient over 100."""
import os

import numpy as np
import pytest

from helpers import new_engine
from reaxamd import systems
from oracle.oracle import Oracle

TERMS = ("e_bond", "e_ov", "e_un", "e_lp", "e_ang", "e_pen", "e_coa", "e_tor", "e_con", "e_vdW")
BASIS = np.array([[0, 0, 0], [0, 2, 2], [2, 0, 2], [2, 2, 0], [1, 1, 1], [1, 3, 3], [3, 1, 3], [3, 3, 1]]) / 4.0


def diamond(cells, drop, seed, a=3.567, sigma=0.08):
    g = np.stack(np.meshgrid(*[np.arange(c) for c in cells], indexing="ij"), -1).reshape(-1, 3)
    x = ((g[:, None] + BASIS[None]) * a).reshape(-1, 3)
    rng = np.random.default_rng(seed)
    x = x + rng.normal(size=x.shape) * sigma
    return x[rng.permutation(len(x))[drop:]], np.array(cells) * a


@pytest.mark.gpu
@pytest.mark.parametrize("cells,drop", [((2, 2, 2), 1), ((2, 2, 3), 31), ((3, 3, 3), 0), ((9, 10, 9), 17)])
def test_dense_carbon(cells, drop):
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ffield.C2013")) as fh:
        ff = fh.read()
    x, L = diamond(cells, drop, seed=sum(cells))
    n = len(x)
    types, tags, q = np.ones(n, dtype=np.int32), np.arange(1, n + 1), np.zeros(n)
    box12 = [0, 0, 0, L[0], 0, 0, 0, L[1], 0, 0, 0, L[2]]
    ref = Oracle(ff).compute(x, types - 1, tags, box12, (True, True, True), q=q)
    for prec in ("fp64", "mixed"):
        e = new_engine(ff, ["C"], prec, extra=("checkqeq", "no"))
        e.set_box(np.zeros(3), L)
        e.set_atoms(types, tags, x)
        e.set_charges(q)
        r = e.compute(rebuild=True, census=True)
        cen = e.census()
        e.close()
        d = (r["grad"] - np.asarray(ref["grad"])) / max(1.0, np.abs(ref["grad"]).max() / 100.0)
        if prec == "fp64":
            for k in TERMS:
                assert abs(r["energy"][k] - ref["energy"][k]) <= 1e-9 * max(1.0, abs(ref["energy"][k])), (n, k)
            assert np.abs(d).max() <= 1e-7, n
        else:
            assert abs(sum(r["energy"].values()) - sum(ref["energy"].values())) / n <= 1e-4, n
            assert np.abs(d).max() <= 4e-3 and np.sqrt((d ** 2).mean()) <= 9e-4, n
        for k, name in enumerate(("bonds", "angle_sets", "torsions")):
            assert np.array_equal(cen[k], np.asarray(ref["census"][name])), (n, prec, name)


@pytest.mark.gpu
@pytest.mark.parametrize("a,cells,drop", [(3.2, (2, 3, 3), 0), (3.0, (2, 2, 3), 5)])
def test_many_bonds(a, cells, drop):
    """Bond orders without the overcoordination corrections (ovc and 13corr 0) in compressed diamond: 14 to 23 bonds per atom above
    the three-body cutoff, so that an angle row and a torsion row fill the queue several times per slot, and the far bonds of a
    central bond exceed those kept in LDS. Bars as above, the energy bar also scaled: 1e-4 kcal/mol per atom for terms that sum to
    100 kcal/mol per atom."""
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ffield.C2013")) as fh:
        t = fh.read().split("\n")
    b = next(k for k, line in enumerate(t) if "Nr of bonds" in line) + 2
    for line, field in ((b, 7), (b + 1, 6)):
        f = t[line].split()
        f[field] = "0.0"
        t[line] = " ".join(f)
    ff = "\n".join(t)
    x, L = diamond(cells, drop, seed=9, a=a, sigma=0.05)
    n = len(x)
    types, tags, q = np.ones(n, dtype=np.int32), np.arange(1, n + 1), np.zeros(n)
    ref = Oracle(ff).compute(x, types - 1, tags, [0, 0, 0, L[0], 0, 0, 0, L[1], 0, 0, 0, L[2]], (True, True, True), q=q)
    scale = max(1.0, np.abs(ref["grad"]).max() / 100.0)
    e_scale = max(1.0, sum(abs(v) for v in ref["energy"].values()) / n / 100.0)
    for prec in ("fp64", "mixed"):
        e = new_engine(ff, ["C"], prec, extra=("checkqeq", "no"))
        e.set_box(np.zeros(3), L)
        e.set_atoms(types, tags, x)
        e.set_charges(q)
        r = e.compute(rebuild=True, census=True)
        cen = e.census()
        e.close()
        d = (r["grad"] - np.asarray(ref["grad"])) / scale
        if prec == "fp64":
            for k in TERMS:
                assert abs(r["energy"][k] - ref["energy"][k]) <= 1e-9 * max(1.0, abs(ref["energy"][k])), (n, k)
            assert np.abs(d).max() <= 1e-7, n
        else:
            assert abs(sum(r["energy"].values()) - sum(ref["energy"].values())) / n <= 1e-4 * e_scale, n
            assert np.abs(d).max() <= 4e-3 and np.sqrt((d ** 2).mean()) <= 9e-4, n
        for k, name in enumerate(("bonds", "angle_sets", "torsions")):
            assert np.array_equal(cen[k], np.asarray(ref["census"][name])), (n, prec, name)


@pytest.mark.gpu
@pytest.mark.parametrize("n,density", [(13003, 1.6), (12000, 1.3)])
def test_two_group_sizes(n, density):
    """Disordered carbon with a few atoms of 9 to 16 bonds: the launch that gives 16 lanes to their groups of 8 atoms and 8 to the rest
    against the per-atom call, which takes 64 lanes for every atom: the sums are the same, bit for bit."""
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ffield.C2013")) as fh:
        ff = fh.read()
    w = systems.random_carbon(n, density=density, seed=4)
    for prec in ("fp64", "mixed", "fp32"):
        e = new_engine(ff, ["C"], prec, extra=("checkqeq", "no"))
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        r = e.compute(rebuild=True, census=True)
        bonds = np.asarray(e.census()[0])
        ra = e.compute(peratom=True)
        e.close()
        assert 8 < bonds.max() <= 16 and 0 < 64 * (bonds > 8).sum() <= n, (bonds.max(), (bonds > 8).sum())   # the launch in question
        assert r["energy"] == ra["energy"], prec
        assert np.array_equal(r["grad"], ra["grad"]) and np.array_equal(r["virial"], ra["virial"]), prec
