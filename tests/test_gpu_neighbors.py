"""Neighbour search against a direct count of all images: the entries of the skin list, of the bond candidates and of the H-bond
candidates (donor lists and their transpose) for cells on both search paths, at the sizes where they can go wrong: one atom, atom
counts around a wave, cells thinner than the list radius (many images, several per wave), tilted cells (where the distance to a
block of the cell is bounded by one face only), open directions, cells just wide enough for the cell search, atoms on the
faces, and several systems in one context. Counts are integers: equal."""
import numpy as np
import pytest

from helpers import new_engine

RS, RB, RH = 12.0, 7.0, 9.5   # nonb_cut, bond_cut and hbond_cut plus the 2 A skin


def atoms(n, lo, hi, tilt, seed, faces=False):
    rng = np.random.default_rng(seed)
    f = rng.random((n, 3))
    if faces:
        f[:: 3, 0] = 0.0
        f[1:: 3, 1] = np.nextafter(1.0, 0.0)
        f[2:: 3] += np.array([2.0, -3.0, 1.0])   # outside the cell: wrapped by the search
    v = np.array([[hi[0] - lo[0], 0, 0], [tilt[0], hi[1] - lo[1], 0], [tilt[1], tilt[2], hi[2] - lo[2]]])
    return f @ v + lo, v, rng.integers(1, 4, n).astype(np.int32)


def count(x, v, types, per):
    """(skin entries, bond candidates, H-bond candidates) over all images."""
    h = [abs(np.linalg.det(v)) / np.linalg.norm(np.cross(v[(d + 1) % 3], v[(d + 2) % 3])) for d in range(3)]
    f = x @ np.linalg.inv(v)
    x = x - np.where(per, np.floor(f), 0.0) @ v
    m = [int(np.ceil(RS / h[d])) + 1 if per[d] else 0 for d in range(3)]
    skin = bond = hb = 0
    for a in range(-m[0], m[0] + 1):
        for b in range(-m[1], m[1] + 1):
            for c in range(-m[2], m[2] + 1):
                d = x[None] + np.array([a, b, c]) @ v - x[:, None]
                r = np.sqrt((d * d).sum(-1))
                if (a, b, c) == (0, 0, 0):
                    np.fill_diagonal(r, np.inf)
                skin += int((r <= RS).sum())
                bond += int((r <= RB).sum())
                hb += 2 * int(((r <= RH) & (types[:, None] == 2) & (types[None] == 3)).sum())   # donor slots and their transpose
    return skin, bond, hb


CELLS = [
    (1, (4.0, 5.0, 6.0), (0, 0, 0), (1, 1, 1), False),
    (2, (5.0, 5.0, 30.0), (1.5, -2.0, 3.0), (1, 1, 1), False),
    (24, (6.2, 6.2, 6.2), (0, 0, 0), (1, 1, 1), True),
    (63, (9.0, 14.0, 11.0), (3.0, -4.0, 2.0), (1, 1, 1), True),
    (64, (14.0, 14.0, 14.0), (0, 0, 0), (1, 0, 1), False),
    (65, (14.0, 20.0, 9.0), (6.0, 3.0, -8.0), (1, 1, 1), False),
    (130, (20.0, 20.0, 20.0), (0, 0, 0), (0, 0, 0), False),
    (501, (31.0, 31.0, 31.0), (0, 0, 0), (1, 1, 1), True),
    (700, (36.01, 37.0, 40.0), (0, 0, 0), (1, 1, 1), True),       # 3 x 3 x 3 search cells
    (900, (44.0, 50.0, 60.0), (12.0, -9.0, 15.0), (1, 1, 1), True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("n,box,tilt,per,faces", CELLS)
def test_lists_hold_every_image(ffield_text, n, box, tilt, per, faces):
    lo = np.array([-1.0, 2.0, 0.5])
    hi = lo + np.array(box)
    x, v, types = atoms(n, lo, hi, tilt, n, faces)
    e = new_engine(ffield_text, ["C", "H", "O"])
    e.set_box(lo, hi, tilt, per)
    e.set_atoms(types, np.arange(1, n + 1), x)
    e.compute(rebuild=True)
    st = e.stats()
    e.close()
    assert (st["skin_entries"], st["bond_candidates"], st["hb_candidates"]) == count(x - lo, v, types, np.array(per, bool))


@pytest.mark.gpu
def test_lists_of_packed_systems(ffield_text):
    class W:
        pass
    systems, want = [], np.zeros(3, dtype=int)
    for k, (n, L) in enumerate(((1, 5.0), (24, 6.2), (65, 13.0), (300, 26.0))):
        w = W()
        w.lo, w.hi = np.zeros(3), np.full(3, L)
        w.x, v, w.types = atoms(n, w.lo, w.hi, (0, 0, 0), 50 + k, faces=True)
        w.tags, w.periodic = np.arange(1, n + 1), (True, True, True)
        systems.append(w)
        want += count(w.x, v, w.types, np.ones(3, bool))
    e = new_engine(ffield_text, ["C", "H", "O"])
    e.set_systems(systems)
    e.compute(rebuild=True)
    st = e.stats()
    e.close()
    assert (st["skin_entries"], st["bond_candidates"], st["hb_candidates"]) == tuple(want)
