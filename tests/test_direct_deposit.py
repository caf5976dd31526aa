"""Plain FP64 deposits, whose tets are shared by the lanes of each wave (unit scaled cells, no work
statistics), against the extended-precision oracle and against the one-tet-per-thread form.

Tolerances: a cell's mass is a sum of shares that each carry a few roundings of a tet (2e-14); the
one-tet-per-thread form stays within 1e-6 of a share, or 1e-12 of a tet where shares are tiny.
"""

import numpy as np
import pytest

import adeco_amd as A
from tests import _oracle as O
from tests.test_block_clip import soup_of_extents
from tests.test_gpu_leaves import make_lattice

pytestmark = pytest.mark.gpu
BOX = np.array([0, 32, 0, 32, 0, 32], np.float32)


@pytest.mark.parametrize("extents", [
    [(1, 1, 24), (2, 2, 6), (1, 4, 6), (2, 3, 4)],   # one block of 24 cells
    [(1, 1, 25), (1, 2, 13), (2, 2, 7), (3, 3, 3)],  # just over
])
@pytest.mark.parametrize("mode", [A.MODE_PLAIN, A.MODE_BATCHED])
def test_soup_around_the_largest_block(extents, mode):
    tets = soup_of_extents(np.random.default_rng(11), extents, 80)
    print(f"[direct] {extents} mode {mode}", flush=True)
    got = A.deposit_soup(tets, BOX, 32, 1.0, mode=mode, precision=A.PREC_FP64)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_soup_ld(tets, BOX, 32, 1.0)
    assert O.max_rel_err(got, want, tet_mass=1.0) <= 1e-6
    assert abs(got.sum() - want.sum()) <= 1e-9 * want.sum()


@pytest.mark.parametrize("n", [1, 63, 65, 700])
@pytest.mark.parametrize("extents", [
    [(1, 1, 1), (1, 2, 2)],                          # one block each: taken without a second walk
    [(1, 1, 1), (2, 2, 5), (3, 3, 3)],               # some tets of several blocks
    [(1, 1, 1), (16, 16, 16), (2, 30, 30)],          # tets of very unequal size
])
def test_soup(n, extents):
    rng = np.random.default_rng(n)
    tets = soup_of_extents(rng, extents, (n + len(extents) - 1) // len(extents))
    tets = tets[rng.permutation(len(tets))][:n]
    tets[n // 2, 3] = tets[n // 2, 2]                # a tet without volume
    tets[n // 3] += 40.0                             # and one beyond the grid
    print(f"[direct] {n} of {extents}", flush=True)
    got = A.deposit_soup(tets, BOX, 32, 1.0)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_soup_ld(tets, BOX, 32, 1.0)
    assert O.max_rel_err(got, want, tet_mass=1.0) <= 1e-6
    assert abs(got.sum() - want.sum()) <= 1e-9 * max(want.sum(), 1.0)


@pytest.mark.parametrize("dims", [1, 4, 5, 16])
def test_batched_soup_on_either_side_of_four_tets_per_cell(dims):
    tets = soup_of_extents(np.random.default_rng(dims), [(1, 2, 2), (3, 3, 3), (9, 12, 14)], 100)  # 300 >= 4 * 4^3
    print(f"[direct] batched soup {dims}", flush=True)
    got = A.deposit_soup(tets, BOX, dims, 1.0, mode=A.MODE_BATCHED)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_soup_ld(tets, BOX, dims, 1.0)
    assert O.max_rel_err(got, want, tet_mass=1.0) <= 1e-6
    assert abs(got.sum() - want.sum()) <= 1e-9 * want.sum()


@pytest.mark.parametrize("dims", [1, 2, 17, 64])
def test_lattice_tets_all_and_listed(dims):
    rng = np.random.default_rng(dims)
    pos = [np.ascontiguousarray(c, np.float32) for c in (np.stack(np.meshgrid(*[np.arange(9.0)] * 3, indexing="ij"), -1)
                                                         + rng.normal(0, 0.4, (9, 9, 9, 3))).transpose(3, 2, 1, 0)]
    lat = A.ResidentLattice(*[p.reshape(-1) for p in pos], (9, 9, 9))
    box = A.cubic_root_box(lat.bbox())
    n = lat.num_tets
    for ids in (None, rng.permutation(n)[: n // 3].astype(np.int32), np.array([n - 1], np.int32)):
        print(f"[direct] lattice {dims} {0 if ids is None else ids.size}", flush=True)
        got = lat.deposit_grid(box, dims, tet_ids=ids)
        want, _ = lat.deposit_grid(box, dims, tet_ids=ids, stats=True)  # one tet per thread
        assert np.abs(got - want).max() <= 1e-6 * want.max()
        assert abs(got.sum() - want.sum()) <= 1e-9 * want.sum()


def test_reference_scaling_keeps_its_own_cells():
    """Cells that are no unit cells are not cut in blocks: the result is the one-tet-per-thread form's."""
    tets = soup_of_extents(np.random.default_rng(3), [(1, 1, 1), (3, 3, 3)], 40)
    box = np.array([0, 32, 0, 31, 0, 30], np.float32)
    A.set_cell_scaling(A.SCALING_REFERENCE)
    try:
        got = A.deposit_soup(tets, box, 32, 1.0)
        want, _ = A.deposit_soup(tets, box, 32, 1.0, stats=True)
    finally:
        A.set_cell_scaling(A.SCALING_EXACT)
    assert np.abs(got - want).max() <= 1e-12


def test_cells_with_a_sentinel_vertex_deposit_nothing():
    rng = np.random.default_rng(5)
    ax = np.arange(8.0)
    base = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).transpose(2, 1, 0, 3)
    pat = (base[None] + rng.normal(0, 0.2, (3, 8, 8, 8, 3))).astype(np.float32)
    pat[1, 4:] = 666.0                               # cells k' >= 3 have no tets
    pat[2, 0, 0, 0] = 666.0                          # one cell
    box = np.array([-1, 9, -1, 9, -1, 9], np.float32)
    data = np.zeros(16 ** 3, np.float32)
    A.DepositWrapper.deposit_tets(True, 0, 0, 3, np.ascontiguousarray(pat).reshape(-1), pat.size, 7, box, 16, data)
    cells = 343 + 3 * 49 + 342
    assert abs(data.astype(np.float64).sum() - 6 * cells) <= 1e-5 * 6 * cells


@pytest.mark.parametrize("dims", [2, 5, 10, 24])
def test_leaves_from_pairs_or_pair_lines(dims):
    """Batched leaves on either side of 4 pairs per cell, and plain ones, against the captured deposit, which
    always goes through pair lines."""
    lat = make_lattice(24, 3.0, seed=9)
    print(f"[direct] leaves {dims}", flush=True)
    with A.ResidentLattice.from_lattice(lat) as rl, A.Octree(rl, 1500, 3) as tree:
        pairs = int(tree.bin(A.DECOMP_KUHN).sum())
        assert (pairs >= 4 * tree.num_leaves * dims ** 3) == (dims <= 5)
        with A.DepositGraph(tree, dims, A.DECOMP_KUHN, 0.5, A.PREC_FP64) as g:
            g.launch()
            want = g.leaf_grids()
        for mode in (A.MODE_BATCHED, A.MODE_PLAIN):
            tree.deposit(dims, A.DECOMP_KUHN, 0.5, mode)
            got = tree.leaf_grids()
            assert got.shape == want.shape
            assert np.abs(got - want).max() <= 1e-12 * want.max()


@pytest.mark.parametrize("dims", [101, 102, 131])
def test_results_around_the_split_download(dims):
    """Grids just below and above 8 MiB (one copy, four side by side, no whole number of pages each)."""
    rng = np.random.default_rng(dims)
    tets = (soup_of_extents(rng, [(1, 2, 2), (3, 3, 2)], 60).astype(np.float64) * (dims / 32.0)).astype(np.float32)
    box = np.array([0, dims] * 3, np.float32)
    print(f"[direct] download {dims}", flush=True)
    got = A.deposit_soup(tets, box, dims, 1.0)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_soup_ld(tets, box, dims, 1.0)
    assert all(part.sum() > 0 for part in np.array_split(want, 4))
    assert O.max_rel_err(got, want, tet_mass=1.0) <= 1e-6
