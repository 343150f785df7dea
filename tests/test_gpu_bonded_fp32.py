"""The single-precision bond-order chain and bonded kernels on dense carbon (the systems of test_gpu_bonded_edges, which runs FP64 and mixed)
against the FP64 oracle, where the kernels' work splits have their edges: several atoms per wave, numbers within bond_cut beyond 64,
queues that fill several times per slot, far bonds beyond those in LDS.

Bars as tests/test_gpu_parity.py for FP32: 1e-3 kcal/mol per atom and 5e-2 / 5e-3 kcal/mol/A (largest, RMS). They hold for terms of the
order of 100 kcal/mol per atom and forces of the order of 100 kcal/mol/A; single-precision rounding grows with the terms, so they are
scaled by the terms' sum and the largest reference gradient over 100."""
import os

import numpy as np
import pytest

from helpers import new_engine
from test_gpu_bonded_edges import diamond
from oracle.oracle import Oracle


def carbon_field(corrections=True):
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ffield.C2013")) as fh:
        t = fh.read().split("\n")
    if not corrections:   # bond orders without the overcoordination corrections
        b = next(k for k, line in enumerate(t) if "Nr of bonds" in line) + 2
        for line, field in ((b, 7), (b + 1, 6)):
            f = t[line].split()
            f[field] = "0.0"
            t[line] = " ".join(f)
    return "\n".join(t)


@pytest.mark.gpu
@pytest.mark.parametrize("corrections,a,sigma,cells,drop,seed", [
    (True, 3.567, 0.08, (2, 2, 2), 1, 6), (True, 3.567, 0.08, (2, 2, 3), 31, 7), (True, 3.567, 0.08, (9, 10, 9), 17, 28),
    (False, 3.2, 0.05, (2, 3, 3), 0, 9), (False, 3.0, 0.05, (2, 2, 3), 5, 9)])
def test_dense_carbon_fp32(corrections, a, sigma, cells, drop, seed):
    ff = carbon_field(corrections)
    x, L = diamond(cells, drop, seed, a=a, sigma=sigma)
    n = len(x)
    types, tags, q = np.ones(n, dtype=np.int32), np.arange(1, n + 1), np.zeros(n)
    ref = Oracle(ff).compute(x, types - 1, tags, [0, 0, 0, L[0], 0, 0, 0, L[1], 0, 0, 0, L[2]], (True, True, True), q=q)
    e = new_engine(ff, ["C"], "fp32", extra=("checkqeq", "no"))
    e.set_box(np.zeros(3), L)
    e.set_atoms(types, tags, x)
    e.set_charges(q)
    r = e.compute(rebuild=True)
    e.close()
    scale = max(1.0, np.abs(ref["grad"]).max() / 100.0)
    e_scale = max(1.0, sum(abs(v) for v in ref["energy"].values()) / n / 100.0)
    d = (r["grad"] - np.asarray(ref["grad"])) / scale
    de = abs(sum(r["energy"].values()) - sum(ref["energy"].values())) / n / e_scale
    print("n %d: dE %.1e, dF max %.1e rms %.1e (scaled by %.1f, %.1f)" % (n, de, np.abs(d).max(), np.sqrt((d ** 2).mean()), e_scale, scale))
    assert de <= 1e-3
    assert np.abs(d).max() <= 5e-2 and np.sqrt((d ** 2).mean()) <= 5e-3
