"""Force fields with many species take the kernels' other branches: above 8 species the bond build reads its distance bound from the
pair table instead of LDS, above 16 the matrix build and the non-bonded pass read the type parameters and shift vectors from memory.

The fields here are the C/H/O stand-in with every species copied under other names (Ca, Ha, Oa, Cb, ...) and every parameter line given to
all combinations of the copies, so a system whose atoms are spread over the copies is the same system: everything must equal the
three-species result bit for bit. (The C2 correction, which goes by the name C, is off in both.) A field whose bond orders do not all fall with the distance (an
infinite bound: every candidate is evaluated) against the oracle, at the bars of test_gpu_variants."""
import itertools

import numpy as np
import pytest

from helpers import new_engine
from reaxamd import systems
from oracle.oracle import Oracle


def copies_of(text, copies):
    """The field with each of its species copied, and the names of all species."""
    lines = text.split("\n")
    ngp = int(lines[1].split()[0])
    lines[2 + 5] = "    0.0000 !C2-correction"
    at = 2 + ngp
    out, nt = lines[:at], int(lines[at].split()[0])
    out += ["%3d ! atoms" % (nt * copies)] + lines[at + 1:at + 4]
    names = []
    for c in range(copies):
        for k in range(nt):
            block = lines[at + 4 + 4 * k:at + 8 + 4 * k]
            f = block[0].split()
            names.append(f[0] + ("abcdefghij"[c - 1] if c else ""))
            out += [" ".join([names[-1]] + f[1:])] + block[1:]
    at += 4 + 4 * nt
    # sections: species per line, header lines, lines per entry, the species pair whose swap gives the same entry
    for idx, head, per, same in ((2, 2, 2, (0, 1)), (2, 1, 1, (0, 1)), (3, 1, 1, (0, 2)), (4, 1, 1, None), (3, 1, 1, None)):
        n, rows = int(lines[at].split()[0]), []
        for k in range(n):
            block = lines[at + head + per * k:at + head + per * (k + 1)]
            f = block[0].split()
            ids = [int(v) for v in f[:idx]]
            for cs in itertools.product(range(copies), repeat=idx):
                if any(i == 0 and c for i, c in zip(ids, cs)):
                    continue   # a wildcard
                if same and ids[same[0]] == ids[same[1]] and cs[same[0]] > cs[same[1]]:
                    continue   # the same entry the other way round
                rows.append(" ".join([str(i + nt * c) for i, c in zip(ids, cs)] + f[idx:]))
                rows += block[1:]
        out += ["%d ! entries" % (len(rows) // per)] + lines[at + 1:at + head] + rows
        at += head + per * n
    return "\n".join(out) + "\n", names


def spread(types, copies, seed):
    """each atom's type among the copies of its species"""
    return (np.asarray(types) + 3 * np.random.default_rng(seed).integers(0, copies, len(types))).astype(np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [3, 6])   # 9 and 18 species
@pytest.mark.parametrize("prec", ["fp64", "mixed", "fp32"])
def test_species_copies_change_nothing(ffield_text, copies, prec):
    for w in (systems.water_box(6, seed=2), systems.ch4_o2_gas(450, density=0.3, seed=3), systems.random_carbon(700, seed=4)):
        res = []
        for c in (1, copies):
            text, names = copies_of(ffield_text, c)
            e = new_engine(text, names, prec)
            e.set_box(w.lo, w.hi)
            e.set_atoms(spread(w.types, c, 5), w.tags, w.x)
            e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
            q, it, _ = e.qeq_charges(imax=200, tol=1e-8)
            r = e.compute(census=True)
            cen = e.census()
            p = e.compute(peratom=True)
            v = systems.maxwell_boltzmann(w.masses(), 300.0, seed=6)
            m = np.array([0.0] + [systems.MASS[name[0]] for name in names])
            e.md_setup(v, m, dt=0.25, t_target=300.0, t_damp=25.0)
            th = e.md_run(10)
            res.append((q, it, r, cen, p, th["pe"]) + tuple(e.state()))
            e.close()
        a, b = res
        assert np.array_equal(a[0], b[0]) and list(a[1]) == list(b[1])
        for k in (2, 4):
            assert a[k]["energy"] == b[k]["energy"]
            for f in ("grad", "virial"):
                assert np.array_equal(a[k][f], b[k][f]), f
        assert np.array_equal(a[4]["eatom"], b[4]["eatom"]) and np.array_equal(a[4]["vatom"], b[4]["vatom"])
        assert all(np.array_equal(x, y) for x, y in zip(a[3], b[3]))
        assert a[5] == b[5]
        assert all(np.array_equal(x, y) for x, y in zip(a[6:], b[6:]))


@pytest.mark.gpu
def test_bond_order_that_does_not_fall(ffield_text):
    """The pi bond of a carbon pair with power 0 and coefficient -12: a constant 6e-6 at every distance, far below the bond cutoff."""
    lines = ffield_text.split("\n")
    k = next(i for i, line in enumerate(lines) if "Nr of bonds" in line) + 3   # the second line of the pair 1 1
    f = lines[k].split()
    f[1], f[2] = "-12.0", "0.0"
    lines[k] = " ".join(f)
    text = "\n".join(lines)
    w = systems.random_carbon(700, seed=4)
    q = np.zeros(w.n)
    ref = Oracle(text).compute(w.x, w.types - 1, w.tags, w.box12(), w.periodic, q=q)
    for prec, e_tol, f_max, f_rms in (("fp64", None, 1e-7, None), ("mixed", 1e-4, 4e-3, 9e-4), ("fp32", 1e-3, 5e-2, 5e-3)):
        e = new_engine(text, ["C", "H", "O"], prec, extra=("checkqeq", "no"))
        e.set_box(w.lo, w.hi)
        e.set_atoms(w.types, w.tags, w.x)
        e.set_charges(q)
        r = e.compute(rebuild=True)
        e.close()
        d = (r["grad"] - np.asarray(ref["grad"])) / max(1.0, np.abs(ref["grad"]).max() / 100.0)
        assert np.abs(d).max() <= f_max, prec
        if prec == "fp64":
            for t, v in r["energy"].items():
                assert abs(v - ref["energy"][t]) <= 1e-9 * max(1.0, abs(ref["energy"][t])), t
        else:
            assert abs(sum(r["energy"].values()) - sum(ref["energy"].values())) / w.n <= e_tol, prec
            assert np.sqrt((d ** 2).mean()) <= f_rms, prec
