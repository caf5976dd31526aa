"""The block form of the FP64 deposit on the host: whole soups, from the covers of their tets to the cells' sums,
against the extended-precision oracle and the one-tet-per-thread form."""

import numpy as np
import pytest

import adeco_amd as A
from tests import _oracle as O
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
