"""The block form of the FP64 deposit on the host: whole soups, from the covers of their tets to the cells' sums,
against the extended-precision oracle and the one-tet-per-thread form."""

from fractions import Fraction as F

import numpy as np
import pytest

import adeco_amd as A
from tests import _oracle as O
from tests.rational_clip import tet_box_volume
from tests.test_block_clip import soup_of_extents

KUHN = [(0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)]


def blocks(tets, box, dims):
    """The block form: the grid and the number of cells recomputed alone."""
    grid, n = np.zeros(dims ** 3), np.zeros(1, np.int64)
    tets, box = np.ascontiguousarray(tets, np.float32), np.ascontiguousarray(box, np.float32)
    assert A.load().adeco_selftest_deposit_blocks_f64(A.ptr(tets), len(tets), A.ptr(box), dims, 1.0, A.ptr(grid), A.ptr(n)) == A.ADECO_OK
    return grid, int(n[0])


def one_per_thread(tets, box, dims):
    grid = np.zeros(dims ** 3)
    tets, box = np.ascontiguousarray(tets, np.float32), np.ascontiguousarray(box, np.float32)
    assert A.load().adeco_selftest_deposit_soup_f64(A.ptr(tets), len(tets), A.ptr(box), dims, 1.0, A.ptr(grid), None) == A.ADECO_OK
    return grid


def oracle(tets, box, dims):
    with O.cell_scaling(O.EXACT):
        return O.deposit_soup_ld(np.ascontiguousarray(tets, np.float32), np.ascontiguousarray(box, np.float32), dims, 1.0)


def unit_box(dims):
    return np.array([0, dims] * 3, np.float32)


@pytest.mark.parametrize("extents", [
    [(1, 1, 1), (1, 2, 2), (2, 2, 2), (1, 1, 16)],
    [(2, 2, 6), (1, 4, 6), (1, 1, 24), (2, 3, 4), (1, 3, 8), (1, 2, 12)],  # one block of 24 cells
    [(1, 1, 25), (1, 2, 13), (2, 2, 7), (3, 3, 3), (1, 5, 5)],             # just over
    [(5, 9, 13), (16, 16, 16), (2, 30, 30)],                               # many blocks, empty and filled ones among them
])
def test_soups_of_all_block_shapes(extents):
    """Every share within a few roundings of its tet (2e-14), so a cell within that for each tet."""
    tets = soup_of_extents(np.random.default_rng(21), extents, 30)
    got, _ = blocks(tets, unit_box(32), 32)
    assert np.abs(got - oracle(tets, unit_box(32), 32)).max() <= 2e-14 * len(tets)


def wide_tets(width, seed):
    """Kuhn tets of 2^3 displaced cubes, each cube `width` cells wide, around the middle of a 32^3 grid."""
    rng = np.random.default_rng(seed)
    v = np.stack(np.meshgrid(*[np.arange(3.0)] * 3, indexing="ij"), -1)
    v = (v + rng.normal(0, 0.2, v.shape) - 1.0) * width + 16.0
    out = []
    for p in KUHN:
        o, vs = np.zeros(3, int), []
        for s in range(4):
            vs.append(v[o[0]:o[0] + 2, o[1]:o[1] + 2, o[2]:o[2] + 2].reshape(-1, 3))
            if s < 3:
                o[p[s]] += 1
        out.append(np.stack(vs, 1))
    return np.concatenate(out).astype(np.float32)


def wedges(rng, n, length):
    """Tets `length` cells long and about a cell thick: faces at small angles across the grid."""
    t = rng.normal(0, length, (n, 4, 3))
    axis = rng.integers(0, 3, n)
    t[np.arange(n), :, axis] = rng.uniform(-1.5, 1.5, (n, 4))
    return (t + 16.0).astype(np.float32)


def rms(a, want):
    return float(np.sqrt(((a - want) ** 2).sum() / (want ** 2).sum()))


WIDE = [("cubes", 27), ("cubes", 80), ("cubes", 120), ("cubes", 400), ("cubes", 1000), ("wedges", 40), ("wedges", 600)]


def wide(kind, width):
    if kind == "cubes":
        return wide_tets(width, 7)
    return np.concatenate([wedges(np.random.default_rng(8), 30, width), wide_tets(width, 9)])


@pytest.mark.parametrize("kind,width", WIDE)
def test_large_tets_are_as_exact_as_cell_by_cell(kind, width):
    """Tets of 1e3 to 1e8 cells: no further off than one tet per thread, which clips each cell on its own."""
    tets = wide(kind, width)
    want = oracle(tets, unit_box(32), 32)
    got, _ = blocks(tets, unit_box(32), 32)
    assert rms(got, want) <= rms(one_per_thread(tets, unit_box(32), 32), want)


def test_cells_inside_a_large_tet_are_full():
    """Their mass is cell volume / tet volume, to the rounding of that quotient, whatever block they are in."""
    t = np.array([[[-20, -21, -19], [70, -18, -15], [-17, 66, -22], [-14, -16, 75]]], np.float32)
    v = t[0].astype(np.float64)
    full = 6.0 / abs(np.linalg.det(v[1:] - v[0]))
    got, _ = blocks(t, unit_box(32), 32)
    # barycentric coordinates of the cells' corners
    g = np.stack(np.meshgrid(*[np.arange(33.0)] * 3, indexing="ij"), -1).transpose(2, 1, 0, 3).reshape(-1, 3)
    l = np.linalg.solve((v[1:] - v[0]).T, (g - v[0]).T).T
    corner = (np.column_stack([l, 1.0 - l.sum(1)]) > 1e-9).all(1).reshape(33, 33, 33)
    inner = np.all([corner[i:32 + i, j:32 + j, k:32 + k] for i in (0, 1) for j in (0, 1) for k in (0, 1)], axis=0).reshape(-1)
    assert inner.sum() > 1000 and (got > 0).sum() > inner.sum()
    assert np.abs(got[inner] - full).max() <= 4 * np.finfo(float).eps * full


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [A.MODE_PLAIN, A.MODE_BATCHED])
@pytest.mark.parametrize("kind,width", WIDE)
def test_large_tets_on_the_gpu(mode, kind, width):
    tets = wide(kind, width)
    want = oracle(tets, unit_box(32), 32)
    print(f"[block deposit] {kind} {width} mode {mode}", flush=True)
    got = A.deposit_soup(tets, unit_box(32), 32, 1.0, mode=mode)
    cells, _ = A.deposit_soup(tets, unit_box(32), 32, 1.0, stats=True)  # one tet per thread
    assert rms(got, want) <= rms(cells, want)


def kuhn_lattice(n, noise, scale, offset, seed):
    """The Kuhn tets of n^3 displaced cubes."""
    rng = np.random.default_rng(seed)
    v = np.stack(np.meshgrid(*[np.arange(n + 1.0)] * 3, indexing="ij"), -1)
    v = (v + rng.normal(0, noise, v.shape)) * scale + offset
    out = []
    for p in KUHN:
        o, vs = np.zeros(3, int), []
        for s in range(4):
            vs.append(v[o[0]:o[0] + n, o[1]:o[1] + n, o[2]:o[2] + n].reshape(-1, 3))
            if s < 3:
                o[p[s]] += 1
        out.append(np.stack(vs, 1))
    return np.concatenate(out).astype(np.float32)


def cells_in_extended_precision(tets, box, dims):
    """Every cell of every tet on its own, its faces and coordinates in extended precision (the oracle's faces are
    doubles): the grid."""
    clip = O.load().oracle_clip_unit_cube_ld
    box = box.astype(np.longdouble)
    c = (tets.astype(np.longdouble) - box[0::2]) * dims / (box[1::2] - box[0::2])
    grid = np.zeros((dims, dims, dims), np.longdouble)
    for t in c:
        a, b, d = (t[i] - t[3] for i in range(3))
        vol = a @ np.array([b[1] * d[2] - b[2] * d[1], b[2] * d[0] - b[0] * d[2], b[0] * d[1] - b[1] * d[0]]) / 6
        if vol < 0:  # the clip takes positively oriented tets
            t, vol = t[[3, 1, 2, 0]], -vol
        lo, hi = np.maximum(np.floor(t.min(0)), 0).astype(int), np.minimum(np.floor(t.max(0)), dims - 1).astype(int)
        for i in range(lo[0], hi[0] + 1):
            for j in range(lo[1], hi[1] + 1):
                for k in range(lo[2], hi[2] + 1):
                    local = np.ascontiguousarray((t - np.array([i, j, k])).astype(np.float64))
                    grid[k, j, i] += np.longdouble(clip(A.ptr(local))) / vol
    return grid.reshape(-1)


def rounded_box():
    """Tets of about a cell, 50 cells from the grid's corner, in a box whose cells are no binary fractions."""
    tets = kuhn_lattice(5, 0.25, 2 * 0.37, 31.3 + 47 * 0.37, 12)
    return tets, np.array([31.3, 31.3 + 60 * 0.37] * 3, np.float32), 60


# A vertex is rounded at up to 8 cells from its cover's corner (4.4e-16, and as much in its block), which moves faces whose
# area is about 6 times the tet's volume: 5e-15 at worst, and less than half of it rms.  Rounded at 50 cells: 7e-15.
NEAR = 2e-15


def test_cell_coordinates_are_rounded_near_the_tet():
    tets, box, dims = rounded_box()
    got, _ = blocks(tets, box, dims)
    assert rms(got, cells_in_extended_precision(tets, box, dims)) <= NEAR


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [A.MODE_PLAIN, A.MODE_BATCHED])
def test_cell_coordinates_on_the_gpu(mode):
    tets, box, dims = rounded_box()
    want = cells_in_extended_precision(tets, box, dims)
    print(f"[block deposit] rounded box, mode {mode}", flush=True)
    assert rms(A.deposit_soup(tets, box, dims, 1.0, mode=mode), want) <= NEAR


# Flat tets with a share of 1e-8 to 1e-7 that the differences get wrong by 3e-6 to 1.5e-5 of itself (7 of 40 000 drawn as
# below).
FLAT = [
    [[5.124186038970947, 2.7174665927886963, 2.9999868869781494], [7.428884983062744, 3.4607295989990234, 3.00002121925354],
     [4.628147602081299, 2.9347012042999268, 3.000011444091797], [4.359897136688232, 3.0584897994995117, 3.0000274181365967]],
    [[3.814727544784546, 5.635190963745117, 5.000024795532227], [3.1704132556915283, 5.788705348968506, 5.0000081062316895],
     [4.357591152191162, 4.377269744873047, 4.999981880187988], [3.50095272064209, 4.846557140350342, 4.999975204467773]],
    [[4.999984264373779, 5.610897541046143, 4.5403618812561035], [5.000033378601074, 7.301886081695557, 3.4920175075531006],
     [5.000016689300537, 4.822857856750488, 3.4201204776763916], [5.000036239624023, 4.0167341232299805, 3.6561317443847656]],
    [[1.9999812841415405, 7.243916034698486, 2.5601866245269775], [2.0001235008239746, 4.069445610046387, 3.419501543045044],
     [2.0000534057617188, 3.630175828933716, 2.6255669593811035], [1.9998281002044678, 6.657833576202393, 3.228499174118042]],
]


def flat_tets(n):
    rng = np.random.default_rng(2)
    out = [np.array(FLAT)]
    for i in range(n):
        t = rng.uniform(2, 4, 3) + rng.uniform(0, 1, (4, 3)) * np.array([1.5, 2.5, 4.0])[rng.permutation(3)]
        t[:, rng.integers(3)] = rng.integers(2, 6) + rng.uniform(-0.5, 0.5, 4) * [1e-3, 1e-4][i % 2]
        out.append(t[None])
    return np.concatenate(out).astype(np.float32)


def volume(v):
    a, b, c = ([v[i][k] - v[3][k] for k in range(3)] for i in range(3))
    return abs(a[0] * (b[1] * c[2] - b[2] * c[1]) + b[0] * (c[1] * a[2] - c[2] * a[1]) + c[0] * (a[1] * b[2] - a[2] * b[1])) / 6


def test_flat_tets_cut_along():
    """Tets that are thin along an axis and lie across a cell face there.  A cut point is rounded to about 1e-15 cells,
    1e-15 / thickness of a share; shares below 1e-9 / thickness are recomputed, to 1e-15 of the tet: so to that or 1e-6
    of the share.  Small shares against rationals."""
    checked = 0
    for t in flat_tets(1000):
        got, _ = blocks(t[None], unit_box(8), 8)
        v = [tuple(F(float(x)) for x in p) for p in t]
        for c in np.nonzero((got >= 1e-12) & (got < 1e-6))[0]:
            lo = (int(c) % 8, int(c) // 8 % 8, int(c) // 64)
            want = float(tet_box_volume(v, lo, tuple(i + 1 for i in lo)) / volume(v))
            assert abs(got[c] - want) <= max(1e-15, 1e-6 * want)
            checked += 1
        assert abs(got.sum() - 1.0) <= 1e-9
    assert checked > 80


@pytest.mark.parametrize("depth", [1e-7, 1e-9, 1e-12])
def test_a_vertex_just_beyond_a_face(depth):
    """What is cut off is a share of 1e-19 to 1e-36, a negative term far below the unit of the sums."""
    rng = np.random.default_rng(6)
    for i in range(300):
        t = rng.uniform(0.2, 2.0, (4, 3))
        t[i % 4, (i // 4) % 3] = -depth
        t = t[None].astype(np.float32)
        got, _ = blocks(t, unit_box(8), 8)
        assert np.abs(got - oracle(t, unit_box(8), 8)).max() <= 2e-14


@pytest.mark.parametrize("cells", [(2, 2, 6), (1, 4, 6), (2, 3, 4), (1, 1, 24), (2, 2, 5)])
def test_blocks_of_up_to_24_cells_match_the_rational_clip(cells):
    """The clip of one block against rationals: 2e-14 of the tet, and where it is thin along an axis a few roundings of
    its coordinates there (up to 24 cells: 1e-14 with those of the cut points) over the thickness."""
    rng = np.random.default_rng(cells[2])
    for i in range(6):
        thickness = [0.0, 0.0, 0.0, 1e-1, 1e-2, 1e-3][i]
        t = rng.uniform(0.2, 0.8, 3) * np.array(cells) + rng.standard_normal((4, 3)) * [0.4, 1.0, 3.0][i % 3]
        if thickness:
            axis = int(np.argmax(np.array(cells) > 1)) if i % 2 else 2
            t[:, axis] = rng.integers(1, max(cells[axis], 2)) + rng.uniform(-0.5, 0.5, 4) * thickness
        t = np.ascontiguousarray(t)
        shares, alone, c = np.zeros(24), np.zeros(24), np.array(cells, np.int32)
        assert A.load().adeco_selftest_block_f64(A.ptr(t), A.ptr(c), A.ptr(shares), A.ptr(alone)) == int(np.prod(cells))
        v = [tuple(F(float(x)) for x in p) for p in t]
        tol = 2e-14 + (1e-14 / thickness if thickness else 0.0)
        for n, (a, b, k) in enumerate(np.ndindex(*cells)):
            want = float(tet_box_volume(v, (a, b, k), (a + 1, b + 1, k + 1)) / volume(v))
            assert abs(shares[n] - want) <= tol
            assert abs(alone[n] - want) <= max(1e-15, 1e-6 * want)
