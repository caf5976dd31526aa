"""Per-leaf binning whose workgroups count the leaves of many tets in LDS: lattices whose workgroups meet more
leaves than the table holds, tets of several leaves each (more entries than the list holds), and tets too large
for the leaf map, against a test of every tet with every leaf.

A leaf's list holds each tet once, every tet whose box strictly overlaps the leaf's, and none whose box misses
the leaf's by more than 1e-5 of the root.
"""

import numpy as np
import pytest

import adeco_amd as A
from adeco_amd.lattice import make_lattice
from tests import _oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rms,split,depth", [
    (0.2, 1, 4),    # small tets, a leaf or two each, hundreds of leaves to a workgroup
    (1.0, 1, 4),    # several leaves each
    (6.0, 1, 3),    # many leaves each, some left to the descent of the tree
    (2.0, 100000, 3),  # one leaf
])
def test_lists_hold_the_overlapping_tets(rms, split, depth):
    lat = make_lattice(16, rms, seed=21)
    tets = O.lattice_tets(lat, A.DECOMP_KUHN)
    lo, hi = tets.min(axis=1).astype(np.float64), tets.max(axis=1).astype(np.float64)
    print(f"[bin] rms {rms} split {split} depth {depth}", flush=True)
    with A.ResidentLattice.from_lattice(lat) as rl, A.Octree(rl, split, depth) as tree:
        counts = tree.bin(A.DECOMP_KUHN)
        boxes = tree.leaf_boxes_f64()
        margin = 1e-5 * (boxes[:, 1::2].max() - boxes[:, ::2].min())
        total = 0
        for l in range(tree.num_leaves):
            ids = tree.leaf_tets(l)
            assert ids.size == counts[l] == np.unique(ids).size
            b0, b1 = boxes[l, ::2], boxes[l, 1::2]
            strict = ((lo < b1) & (b0 < hi)).all(axis=1)
            near = ((lo < b1 + margin) & (b0 - margin < hi)).all(axis=1)
            member = np.zeros(len(tets), bool)
            member[ids] = True
            assert not (strict & ~member).any() and not (member & ~near).any()
            total += ids.size
        assert total >= len(tets) * 0.9
        print(f"[bin] {tree.num_leaves} leaves, {total / len(tets):.2f} pairs per tet", flush=True)
