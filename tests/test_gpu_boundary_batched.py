"""The batched boundary call, which deposits a pass of 4 or more tets per cell straight from its patches and any other
from a soup of their tets: on either side of that rule, and in passes of both kinds.

Tolerance: FP32 results against the extended-precision oracle, 1e-6; counts of a pass are those of the same patches
deposited alone.
"""

import numpy as np
import pytest

import adeco_amd as A
from adeco_amd.lattice import make_lattice, meta_patches
from tests import _oracle as O

pytestmark = pytest.mark.gpu
PER_PATCH = 6 * 7 ** 3


@pytest.fixture
def batched():
    prev = A.set_boundary_form(mode=A.MODE_BATCHED)
    yield
    A.set_memory_budget(0)
    A.set_boundary_form(**prev)


def patches(n):
    lat = make_lattice(14, 2.0, seed=11)
    p = meta_patches(lat).reshape(-1, 1536)[:n]
    assert len(p) == n
    return np.ascontiguousarray(p).reshape(-1), A.cubic_root_box(lat.bbox())


def deposit(pat, box, dims):
    out = np.zeros(dims ** 3, np.float32)
    A.DepositWrapper.deposit_tets(True, 0, 0, pat.size // 1536, pat, pat.size, 7, box, dims, out)
    t = A.Octree.last_timings()
    return out, (t["candidates"], t["partials"], t["fallbacks"])


def check(got, pat, box, dims):
    with O.cell_scaling(O.EXACT):
        want = O.deposit_patches_ld(pat, box, dims)
    assert O.max_rel_err(got, want) <= 1e-6


@pytest.mark.parametrize("dims", [1, 8, 9, 12, 16, 17])  # 2 patches: straight from them up to 10^3 cells
def test_either_side_of_four_tets_per_cell(batched, dims):
    pat, box = patches(2 if dims < 16 else 8)  # 8 patches: up to 16^3
    print(f"[boundary] dims {dims}", flush=True)
    got, (candidates, partials, _) = deposit(pat, box, dims)
    check(got, pat, box, dims)
    assert candidates >= pat.size // 1536 * PER_PATCH and int(dims > 1) <= partials <= candidates


@pytest.mark.parametrize("n", [2, 3, 4, 5])
def test_passes_of_both_kinds(batched, n):
    """Two patches a pass on 10^3 cells: straight from them; a last one of a single patch from its soup."""
    pat, box = patches(n)
    dims = 10
    assert 2 * PER_PATCH >= 4 * dims ** 3 > PER_PATCH
    last = pat[-1536 * (2 - n % 2):]
    _, alone = deposit(np.ascontiguousarray(last), box, dims)
    # a patch, its soup, ids and candidate space take 410 kB (6144 bytes, and 48 + 4 + 144 per tet)
    A.set_memory_budget(dims ** 3 * 8 + 1_200_000)
    print(f"[boundary] {n} patches in passes", flush=True)
    got, counts = deposit(pat, box, dims)
    check(got, pat, box, dims)
    assert counts[0] == alone[0] and counts[1] == alone[1]
