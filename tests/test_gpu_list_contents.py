"""What the neighbour lists hold, entry by entry, through results that depend on each entry's partner and image (the totals of
test_gpu_neighbors do not tell a wrong image from a right one):

* the charge matrix (pairs within 10 A of the skin list) times a random vector, against the FP64 oracle: 1e-12 of the largest element, for
  every cell of test_gpu_neighbors, the tilted and the partly open ones among them;
* energies and gradient (bond candidates, H-bond candidates and their transpose) of water in tilted and partly open cells on both search
  paths, against the oracle: FP64, each term within 1e-9 of max(1, |E|), the gradient within 1e-7 kcal/mol/A of forces of the order
  of 100;
* the non-bonded pass over the matrix rows with the tables of 27 shifts, which cells of at least three list radii have, against the pass
  over the skin list, bit for bit."""
import os

import numpy as np
import pytest

from helpers import new_engine
from test_gpu_neighbors import CELLS, atoms
from reaxamd import Engine, systems
from oracle.oracle import Oracle


def box12_of(lo, hi, tilt):
    L = np.asarray(hi) - np.asarray(lo)
    return list(lo) + [L[0], 0, 0, tilt[0], L[1], 0, tilt[1], tilt[2], L[2]]


@pytest.mark.gpu
@pytest.mark.parametrize("n,box,tilt,per,faces", CELLS)
def test_matrix_of_every_cell(ffield_text, n, box, tilt, per, faces):
    lo = np.array([-1.0, 2.0, 0.5])
    hi = lo + np.array(box)
    x, _, types = atoms(n, lo, hi, tilt, n, faces)
    v = np.random.default_rng(n).normal(size=n)
    tags = np.arange(1, n + 1)
    e = new_engine(ffield_text, ["C", "H", "O"])
    e.set_box(lo, hi, tilt, per)
    e.set_atoms(types, tags, x)
    e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
    y = e.qeq_matvec(v)
    e.close()
    yo = Oracle(ffield_text).qeq_matvec(x, types - 1, tags, box12_of(lo, hi, tilt), tuple(map(bool, per)), v)
    assert np.abs(y - yo).max() <= 1e-12 * max(1.0, np.abs(yo).max())


# (bricks of water shifted against each other along the tilts: molecules stay a lattice constant apart)
WATER = [
    (4, (0, 0, 0), (1, 0, 1)),
    (4, (3.0, -4.0, 2.0), (1, 1, 1)),
    (5, (-7.0, 5.0, 6.5), (1, 1, 1)),
    (4, (3.0, 0, 0), (1, 1, 0)),
    (4, (0, 0, 0), (0, 0, 0)),
    (13, (2.0, -3.0, 1.5), (1, 1, 1)),   # cell search
]


@pytest.mark.gpu
@pytest.mark.parametrize("nside,tilt,per", WATER)
def test_water_in_tilted_and_open_cells(ffield_text, nside, tilt, per):
    w = systems.water_box(nside, seed=nside)
    q = np.where(w.types == 3, -0.7, 0.35) + np.random.default_rng(1).normal(size=w.n) * 0.02
    ref = Oracle(ffield_text).compute(w.x, w.types - 1, w.tags, box12_of(w.lo, w.hi, tilt), tuple(map(bool, per)), q=q)
    e = new_engine(ffield_text, ["C", "H", "O"])
    e.set_box(w.lo, w.hi, tilt, per)
    e.set_atoms(w.types, w.tags, w.x)
    e.set_charges(q)
    r = e.compute(rebuild=True)
    e.close()
    assert ref["energy"]["e_hb"] != 0.0 and ref["energy"]["e_ang"] != 0.0
    for k, v in r["energy"].items():
        assert abs(v - ref["energy"][k]) <= 1e-9 * max(1.0, abs(ref["energy"][k])), k
    assert np.abs(r["grad"] - np.asarray(ref["grad"])).max() <= 1e-7 * max(1.0, np.abs(ref["grad"]).max() / 100.0)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed", "fp32"])
def test_rows_with_27_shifts(ffield_text, prec):
    w = systems.water_box(12, seed=5)
    assert w.hi[0] - w.lo[0] >= 36.0
    out = []
    for rows in ("1", "0"):
        os.environ["RXA_NB_ROWS"] = rows
        try:
            e = Engine(0)
        finally:
            os.environ.pop("RXA_NB_ROWS", None)
        e.pair_style(["NULL", "precision", prec])
        e.pair_coeff(ffield_text, list(systems.ELEMENTS))
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
        q = e.qeq_charges(imax=200, tol=1e-8)[0]
        out.append((q, e.compute()))
        if prec == "fp64" and rows == "1":
            v = np.random.default_rng(2).normal(size=w.n)
            y = e.qeq_matvec(v)
            yo = Oracle(ffield_text).qeq_matvec(w.x, w.types - 1, w.tags, w.box12(), w.periodic, v)
            assert np.abs(y - yo).max() <= 1e-12 * max(1.0, np.abs(yo).max())
        e.close()
    (qa, ra), (qb, rb) = out
    assert np.array_equal(qa, qb) and ra["energy"] == rb["energy"]
    assert np.array_equal(ra["grad"], rb["grad"]) and np.array_equal(ra["virial"], rb["virial"])
