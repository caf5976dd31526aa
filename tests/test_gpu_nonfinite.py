"""Tets with a vertex that is not finite deposit nothing, in every FP64 form: each result equals that of the same
input without them (to the rounding of sums of a few hundred terms in another order, 1e-12 of the largest cell)."""

import numpy as np
import pytest

import adeco_amd as A
from tests import _oracle as O

BAD = [np.nan, np.inf, -np.inf]


def small_tets(rng, n, dims, size):
    """n tets of about `size` cells across: in one cell, or over a few."""
    return (rng.uniform(1.0, dims - 1.0, (n, 1, 3)) + rng.uniform(-0.5, 0.5, (n, 4, 3)) * size).astype(np.float32)


def broken(tets):
    """Copies of the tets, each with one coordinate (of every vertex and axis in turn) not finite."""
    out = tets.copy()
    for i in range(len(out)):
        out[i, i % 4, (i // 4) % 3] = BAD[(i // 12) % 3]
    return out


def test_one_tet_per_thread_drops_them():
    """The routine that the other forms are compared with, on the host."""
    rng = np.random.default_rng(2)
    box = np.array([0, 8, 0, 8, 0, 8], np.float32)
    t = broken(small_tets(rng, 72, 8, 0.3))
    grid = np.zeros(512)
    assert A.load().adeco_selftest_deposit_soup_f64(A.ptr(t), len(t), A.ptr(box), 8, 1.0, A.ptr(grid), None) == A.ADECO_OK
    assert not grid.any()


@pytest.mark.gpu
@pytest.mark.parametrize("size", [0.3, 2.5, 7.0])  # tets of one cell, of a block and of several
@pytest.mark.parametrize("mode", [A.MODE_PLAIN, A.MODE_BATCHED])
def test_soup(mode, size):
    rng = np.random.default_rng(3)
    dims = 16
    box = np.array([0, dims] * 3, np.float32)
    good = small_tets(rng, 108, dims, size)
    mixed = np.stack([good, broken(good)], axis=1).reshape(-1, 4, 3)
    print(f"[nonfinite] soup mode {mode} size {size}", flush=True)
    got = A.deposit_soup(np.ascontiguousarray(mixed), box, dims, 1.0, mode=mode)
    want = A.deposit_soup(good, box, dims, 1.0, mode=mode)
    assert want.sum() > 50
    assert np.abs(got - want).max() <= 1e-12 * want.max()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [4, 24])  # batched: straight from the patches, and from a soup of their tets
@pytest.mark.parametrize("mode", [A.MODE_PLAIN, A.MODE_BATCHED])
def test_patches(mode, dims):
    """A vertex that is not finite takes the tets around it away, as the one-tet-per-thread oracle does."""
    rng = np.random.default_rng(4)
    ax = np.arange(8.0)
    base = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).transpose(2, 1, 0, 3)
    pat = (base[None] + rng.normal(0, 0.2, (2, 8, 8, 8, 3))).astype(np.float32)
    for n, value in enumerate(BAD):
        pat[n % 2, 2 + n, 3, 1 + n, n] = value
    box = np.array([-2, 9, -2, 9, -2, 9], np.float32)
    flat = np.ascontiguousarray(pat).reshape(-1)
    assert (2 * 2058 >= 4 * dims ** 3) == (dims == 4)
    print(f"[nonfinite] patches mode {mode} dims {dims}", flush=True)
    prev = A.set_boundary_form(mode=mode)
    try:
        data = np.zeros(dims ** 3, np.float32)
        A.DepositWrapper.deposit_tets(True, 0, 0, 2, flat, flat.size, 7, box, dims, data)
    finally:
        A.set_boundary_form(**prev)
    with O.cell_scaling(O.EXACT):
        want = O.deposit_patches_f64(flat, box, dims)
    assert np.isfinite(want).all() and want.sum() > 4000 - 100
    assert np.abs(data - want).max() <= 1e-6 * want.max()
