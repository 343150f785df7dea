"""Charge solves whose matrix has empty rows beside long ones: atoms out of every other's reach and atoms of a type without an
element (NULL in the pair_coeff list) among bulk water, so that in the product, which walks four rows side by side, a row without
entries waits for rows of several groups of 64. Before each system a larger one is solved in the same context, so that the matrix
storage has held other columns.

A solve's charges q = s - mu t, mu = sum(s) / sum(t), from A s = -chi + r_s and A t = -1 + r_t, satisfy A q + chi - mu = r_s - mu r_t in
every row (A = diag(eta) + H; H q comes from qeq_matvec, whose kernel shares no code with the solve's product). Each residual is
bounded by the solve's stopping rule sqrt(r.r / eta) <= tol |b|: |r_i| <= sqrt(eta_i) tol |b|; the bar is twice that, for the difference between
the recursion's residual and the true one, plus 1e-12 of the largest product for rounding."""
import numpy as np
import pytest

from helpers import new_engine
from reaxamd import systems

TOL = 1e-9
ELEMENTS = ["C", "H", "O", "NULL"]   # the type without an element is 4


def mixed_rows(nside, gap, seed):
    """Bulk water with every fifth atom of the caller's order (and of its cell, most likely) of type 4, and in an enlarged cell
    lone atoms far from everything else, scattered over the order."""
    w = systems.water_box(nside, seed=seed)
    x, types = np.array(w.x), np.array(w.types, dtype=np.int32)
    types[::5] = 4
    L = w.hi + gap
    if gap > 0:
        far = np.stack(np.meshgrid(*[np.arange(w.hi[0] + 11.0, L[0] - 10.5, 11.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x, types = np.concatenate([x, far]), np.concatenate([types, np.full(len(far), 3, dtype=np.int32)])
    order = np.random.default_rng(seed).permutation(len(x))
    return x[order], types[order], L


def check(e, x, types, chi, eta, solve):
    q, it, rel = solve()
    assert np.isfinite(q).all()
    y = e.qeq_matvec(q)
    c, n = chi[types], eta[types]
    r = y + c
    mu = (r / n).sum() / (1.0 / n).sum()
    bar = 2.0 * TOL * np.sqrt(n) * (np.sqrt((c * c).sum()) + abs(mu) * np.sqrt(len(c))) + 1e-12 * max(1.0, np.abs(y).max())
    # mu is taken from the residuals themselves: their weighted mean moves it by no more than the largest of them
    assert (np.abs(r - mu) <= bar + bar.max()).all(), np.abs(r - mu).max()
    assert abs(q.sum()) <= 1e-10 * len(q)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,refine", [("fp64", -1), ("mixed", -1), ("mixed", 0), ("fp32", 0)])
def test_empty_rows_beside_long_ones(ffield_text, prec, refine):
    e = new_engine(ffield_text, ELEMENTS, prec)
    e.qeq_refine(refine)
    first = True
    # a smaller system after a larger one each time; narrow cells (caller's order) and wide ones (cell order), with and without lone atoms
    for nside, gap in ((12, 0.0), (6, 0.0), (5, 45.0), (4, 0.0)):
        x, types, L = mixed_rows(nside, gap, seed=nside)
        e.set_box(np.zeros(3), L)
        e.set_atoms(types, np.arange(1, len(x) + 1), x)
        if first:
            e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
            first = False
        chi, eta = np.array(e.extract("chi")), np.array(e.extract("eta"))
        chi[4], eta[4] = 0.0, 1.0
        check(e, x, types, chi, eta, lambda: e.qeq_charges(imax=1000, tol=TOL))
    e.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed", "fp32"])
def test_empty_rows_in_packed_systems(ffield_text, prec):
    class W:
        pass
    members = []
    for nside, gap in ((5, 0.0), (3, 45.0), (6, 0.0)):
        w = W()
        w.x, w.types, w.hi = mixed_rows(nside, gap, seed=10 + nside)
        w.lo, w.tags, w.periodic = np.zeros(3), np.arange(1, len(w.x) + 1), (True, True, True)
        members.append(w)
    e = new_engine(ffield_text, ELEMENTS, prec)
    e.set_systems(members)
    e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
    q = e.qeq_charges(imax=1000, tol=TOL)[0]
    e.close()
    assert np.isfinite(q).all()
    at = 0
    for w in members:   # each system as a lone one: the packed solve is the same solve
        n = len(w.x)
        s = new_engine(ffield_text, ELEMENTS, prec)
        s.set_systems([w])
        s.qeq_setup(0.0, 10.0, s.extract("chi"), s.extract("eta"), s.extract("gamma"))
        chi, eta = np.array(s.extract("chi")), np.array(s.extract("eta"))
        chi[4], eta[4] = 0.0, 1.0
        check(s, w.x, w.types, chi, eta, lambda: (q[at:at + n], None, None))
        s.close()
        at += n


@pytest.mark.gpu
def test_empty_rows_with_wide_columns(ffield_text):
    """More than 65535 atoms (32-bit columns): bulk water, lone atoms and untyped ones on a lattice of single sites."""
    w = systems.water_box(10, seed=3)
    m = 41
    site = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * 10.5 + w.hi[0] + 11.0
    x = np.concatenate([w.x, site])
    types = np.concatenate([np.array(w.types, dtype=np.int32), np.where(np.arange(len(site)) % 2, 4, 3).astype(np.int32)])
    types[:3000:7] = 4
    L = np.full(3, site.max() + 11.0)
    order = np.random.default_rng(4).permutation(len(x))
    x, types = x[order], types[order]
    assert len(x) > 65535
    for prec in ("fp64", "mixed"):
        e = new_engine(ffield_text, ELEMENTS, prec)
        e.set_box(np.zeros(3), L)
        e.set_atoms(types, np.arange(1, len(x) + 1), x)
        e.qeq_setup(0.0, 10.0, e.extract("chi"), e.extract("eta"), e.extract("gamma"))
        chi, eta = np.array(e.extract("chi")), np.array(e.extract("eta"))
        chi[4], eta[4] = 0.0, 1.0
        check(e, x, types, chi, eta, lambda: e.qeq_charges(imax=1000, tol=TOL))
        e.close()
