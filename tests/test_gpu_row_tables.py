"""Rows whose lookups (shift vectors, type parameters) fit in LDS and rows that read them from memory: periodic cells of molecules on
a lattice, from one with the 27 or 125 shifts of a wide cell to thin ones with more than 64, lists with fewer entries than a wave, with
several chunks, and with a last chunk partly filled.

The charge matrix against the FP64 oracle's product (the bar of test_gpu_qeq: 1e-12 of the largest element), and the non-bonded pass
over its rows against the pass over the skin list (which uses no tables), bit for bit in every precision."""
import os

import numpy as np
import pytest

from reaxamd import Engine, systems

from oracle.oracle import Oracle


def _cell(shape, seed):
    w = systems.water_box(5, seed=seed)
    a = w.hi[0] / 5.0
    mol = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), -1).reshape(-1, 3)
    take = np.repeat((mol < np.array(shape)).all(1), 3)
    x, types = w.x[take], np.asarray(w.types)[take]
    return x, types.astype(np.int32), np.arange(1, len(x) + 1), np.array(shape) * a


def _engine(ff, cell, prec, rows):
    x, types, tags, L = cell
    os.environ["RXA_NB_ROWS"] = "1" if rows else "0"
    try:
        e = Engine(0)
    finally:
        os.environ.pop("RXA_NB_ROWS", None)
    e.pair_style(["NULL", "precision", prec])
    species = e.pair_coeff(ff, list(systems.ELEMENTS))
    e.set_box(np.zeros(3), L)
    e.set_atoms(types, tags, x)
    e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
    return e, species


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(5, 5, 5), (5, 5, 2), (5, 4, 1), (3, 2, 2), (2, 2, 1)])
def test_rows_with_and_without_tables(ffield_text, shape):
    cell = _cell(shape, seed=sum(shape))
    x, types, tags, L = cell
    box12 = [0, 0, 0, L[0], 0, 0, 0, L[1], 0, 0, 0, L[2]]
    v = np.random.default_rng(3).normal(size=len(x))
    e, species = _engine(ffield_text, cell, "fp64", True)
    y = e.qeq_matvec(v)
    e.close()
    yo = Oracle(ffield_text).qeq_matvec(x, species[types - 1], tags, box12, (True, True, True), v)
    assert np.abs(y - yo).max() <= 1e-12 * max(1.0, np.abs(yo).max()), shape
    for prec in ("fp64", "mixed", "fp32"):
        out = []
        for rows in (True, False):
            e = _engine(ffield_text, cell, prec, rows)[0]
            q = e.qeq_charges(imax=200, tol=1e-8)[0]
            out.append((q, e.compute()))
            e.close()
        (qa, ra), (qb, rb) = out
        assert np.array_equal(qa, qb), (shape, prec)
        assert ra["energy"] == rb["energy"], (shape, prec)
        assert np.array_equal(ra["grad"], rb["grad"]) and np.array_equal(ra["virial"], rb["virial"]), (shape, prec)


@pytest.mark.gpu
def test_rows_from_empty_to_several_groups(ffield_text):
    """A cluster of n atoms in a wide cell, n - 1 entries per row: rows without an entry beside rows of 1, 63, 64, 65 and 129, where a
    product's groups of 64 begin, end and run past each other in one wave."""
    rng = np.random.default_rng(11)
    centres = np.array([[20.0, 20, 20], [60, 20, 20], [20, 60, 20], [60, 60, 20], [20, 20, 60], [60, 20, 60]])
    x = np.concatenate([c + rng.uniform(-2.5, 2.5, (n, 3)) for c, n in zip(centres, (1, 2, 64, 65, 66, 130))])
    order = rng.permutation(len(x))
    x = x[order]
    types, tags, L = np.full(len(x), 3, dtype=np.int32), np.arange(1, len(x) + 1), np.full(3, 80.0)
    v = rng.normal(size=len(x))
    for prec, bar in (("fp64", 1e-12), ("mixed", 1e-6)):   # mixed: FP32 values, 6e-8 each
        e, species = _engine(ffield_text, (x, types, tags, L), prec, True)
        y = e.qeq_matvec(v)
        e.close()
        yo = Oracle(ffield_text).qeq_matvec(x, species[types - 1], tags, [0, 0, 0, 80, 0, 0, 0, 80, 0, 0, 0, 80], (True, True, True), v)
        assert np.abs(y - yo).max() <= bar * max(1.0, np.abs(yo).max()), prec
