"""Captured leaf deposits after their octree is gone: a graph owns what it reads and writes, and only the
lattice has to outlive it."""

import numpy as np
import pytest

import adeco_amd as A
from adeco_amd.lattice import make_lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [8, 40])  # leaf grids below and above the size that is downloaded in parts
@pytest.mark.parametrize("step", [False, True])
def test_graph_outlives_its_octree(dims, step):
    lat = make_lattice(16, 2.0, seed=3)
    print(f"[graph] dims {dims} step {step}", flush=True)
    with A.ResidentLattice.from_lattice(lat) as rl:
        with A.Octree(rl, 1000, 2) as tree:
            leaves = tree.num_leaves
            tree.deposit(dims, A.DECOMP_KUHN, 0.5, A.MODE_BATCHED)
            want = tree.leaf_grids()
            graph = A.DepositGraph(tree, dims, A.DECOMP_KUHN, 0.5, A.PREC_FP64, step=step)
        with graph as g:
            assert (leaves * dims ** 3 * 8 >= 8 << 20) == (dims == 40)
            for _ in range(2):
                g.launch()
                got = g.leaf_grids(0, leaves)
                assert np.abs(got - want).max() <= 1e-12 * want.max()
