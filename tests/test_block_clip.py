"""The block form of the batched FP64 deposit: shares of a tet in the cells of a small block, as
differences of cumulative shares between the block's face planes, and the positive recompute of a
single cell.

Tolerances: every share carries a few roundings of the whole tet, so 2e-14 of the tet absolute (a
tet with a 1e-6 of its size in thickness included: no determinant is taken); the recompute of one
cell, whose terms are all positive, to 1e-6 of the share or 1e-15 of the tet.
"""

from fractions import Fraction as F

import numpy as np
import pytest

import adeco_amd as A
from tests import _oracle as O
from tests.rational_clip import tet_box_volume

SHAPES = [(1, 1, 1), (1, 1, 16), (1, 16, 1), (2, 2, 4), (1, 3, 5), (4, 2, 2), (3, 5, 1), (2, 1, 8)]


def block_shares(t, cells):
    c = np.array(cells, np.int32)
    shares, alone = np.zeros(16), np.zeros(16)
    t = np.ascontiguousarray(t, np.float64)
    n = A.load().adeco_selftest_block_f64(A.ptr(t), A.ptr(c), A.ptr(shares), A.ptr(alone))
    assert n == int(np.prod(cells))
    return shares[:n], alone[:n]


def exact_shares(t, cells):
    v = [tuple(F(float(x)) for x in p) for p in t]
    a, b, c = ([v[i][k] - v[3][k] for k in range(3)] for i in range(3))
    vol = abs(a[0] * (b[1] * c[2] - b[2] * c[1]) + b[0] * (c[1] * a[2] - c[2] * a[1]) + c[0] * (a[1] * b[2] - a[2] * b[1])) / 6
    out = []
    for i in range(cells[0]):
        for j in range(cells[1]):
            for k in range(cells[2]):
                out.append(float(tet_box_volume(v, (i, j, k), (i + 1, j + 1, k + 1)) / vol))
    return np.array(out)


@pytest.mark.parametrize("cells", SHAPES)
def test_shares_match_the_rational_clip(cells):
    """Tets inside the block, across its faces and much larger than it, thin ones, and vertices on
    cell faces."""
    rng = np.random.default_rng(7)
    for it in range(6):
        size = [0.3, 0.8, 3.0][it % 3]
        d = rng.standard_normal((4, 3)) * size
        if it >= 3:
            d[:, rng.integers(3)] *= 1e-6
            q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
            d = d @ q
        t = rng.uniform(0.1, 0.9, 3) * np.array(cells) + d
        if it == 1:
            t = np.round(2 * t) / 2 + np.array([[0, 0, 0], [0, 0, 1], [0, 1, 0], [1, 0, 0]]) * 0.5
        want = exact_shares(t, cells)
        shares, alone = block_shares(t, cells)
        assert np.abs(shares - want).max() <= 2e-14, (cells, it)
        assert (np.abs(alone - want) <= np.maximum(1e-15, 1e-6 * want)).all(), (cells, it)


def test_shares_are_a_partition():
    """A tet inside the block: its shares sum to 1, whatever the block, its axis order and the cells the
    vertices lie in."""
    rng = np.random.default_rng(8)
    for it in range(3000):
        cells = SHAPES[it % len(SHAPES)]
        t = rng.uniform(0.0, 1.0, (4, 3)) * np.array(cells)
        if it % 5 == 0:
            t = np.round(t)  # vertices on the faces (possibly a flat tet)
        shares, alone = block_shares(t, cells)
        vol = np.linalg.det(t[1:] - t[0])
        if abs(vol) < 1e-9:
            continue
        assert abs(shares.sum() - 1.0) <= 2e-14
        assert abs(alone.sum() - 1.0) <= 2e-14
        assert np.abs(shares - alone).max() <= 2e-14


def soup_of_extents(rng, extents, per):
    """Tets whose bounding boxes cover the given numbers of unit cells of a [0, 32]^3 grid, in every
    axis order, at random places (some across the grid's faces)."""
    out = []
    for e in extents:
        for _ in range(per):
            e3 = np.array(e)[rng.permutation(3)]
            lo = rng.integers(-1, 32 - e3 + 2)
            t = np.empty((4, 3))
            for a in range(3):
                t[:, a] = lo[a] + rng.uniform(0.2, 0.8, 4) * e3[a]
                i, j = rng.permutation(4)[:2]
                t[i, a], t[j, a] = lo[a] + rng.uniform(0.02, 0.6), lo[a] + e3[a] - rng.uniform(0.02, 0.6)
            out.append(t)
    return np.array(out, np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("extents", [
    [(1, 1, 1), (1, 1, 2), (1, 2, 2), (2, 2, 2)],       # small tets: one block each
    [(1, 1, 16), (1, 4, 4), (2, 2, 4), (2, 4, 2)],      # blocks of 16 cells
    [(1, 1, 17), (2, 2, 5), (3, 3, 2), (3, 3, 3)],      # just over: several blocks
    [(5, 9, 13), (16, 16, 16), (2, 30, 30)],            # many blocks, empty and filled ones among them
])
def test_batched_soup_over_block_shapes(extents):
    rng = np.random.default_rng(17)
    per = 40 if max(max(e) for e in extents) > 17 or len(extents) == 3 else 300
    tets = soup_of_extents(rng, extents, per)
    box = np.array([0, 32, 0, 32, 0, 32], np.float32)
    print(f"[blocks] {extents} x {per}", flush=True)
    got = A.deposit_soup(tets, box, 32, 1.0, mode=A.MODE_BATCHED, precision=A.PREC_FP64)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_soup_ld(tets, box, 32, 1.0)
    assert O.max_rel_err(got, want, tet_mass=1.0) <= 1e-6
    assert abs(got.sum() - want.sum()) <= 1e-9 * want.sum()
