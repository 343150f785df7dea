"""The ordinary force call's angle kernels on both sides of the rule that gives 16 lanes to the aligned groups of 8 atoms that hold one of 9
to 16 bonds and 8 lanes to the others (more than 12,288 atoms, at most one such atom in 64, in FP64 below 18,000 atoms one in 256):
disordered carbon on, above and below the lines. An atom's sums are the same with any number of lanes, so the ordinary call (the kernels
of MD and of plain force calls) must equal the call with the census (its own torsion kernel) and the per-atom call (64 lanes for every
atom) bit for bit, in every precision."""
import os

import numpy as np
import pytest

from helpers import new_engine
from reaxamd import systems


@pytest.mark.gpu
@pytest.mark.parametrize("n,density,both", [(12288, 1.3, ()), (12289, 1.3, ("fp64", "mixed", "fp32")), (13003, 1.6, ("mixed", "fp32")),
                                            (18001, 1.5, ("fp64", "mixed", "fp32")), (12301, 2.2, ())])
def test_ordinary_call_equals_census_and_per_atom(n, density, both):
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ffield.C2013")) as fh:
        ff = fh.read()
    w = systems.random_carbon(n, density=density, seed=4)
    for prec in ("fp64", "mixed", "fp32"):
        e = new_engine(ff, ["C"], prec, extra=("checkqeq", "no"))
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        r = e.compute(rebuild=True)
        rc = e.compute(census=True)
        bonds = np.asarray(e.census()[0])
        ra = e.compute(peratom=True)
        r2 = e.compute()
        e.close()
        over = int((bonds > 8).sum())
        assert 8 < bonds.max() <= 16 and over > 0
        line = 256 if prec == "fp64" and n < 18000 else 64
        assert (prec in both) == (n > 12288 and line * over <= n), over   # the side in question
        for other in (rc, ra, r2):
            assert r["energy"] == other["energy"], prec
            assert np.array_equal(r["grad"], other["grad"]) and np.array_equal(r["virial"], other["virial"]), prec
