"""Leaves of very different numbers of targets in the FP64 leaf kernel (GPU):
its work items name a leaf's blocks of 32 targets, so a launch holds the blocks
that exist, and a leaf may have more of them than a second grid dimension
(65,535).  Bounds as in test_gpu_direct64."""
import numpy as np
import pytest

from test_gpu_direct64 import EPS, _direct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("big", [31, 32, 33, 64, 65, 3000])
def test_one_large_leaf_among_small_ones(nnk, big):
    rng = np.random.default_rng(big)
    corners = np.array([[0, 0, 0], [1, 1, 1.0]])
    tgt = np.concatenate([0.5 * rng.random((big, 3)), 0.5 + 0.5 * rng.random((3, 3)),
                          [0.5, 0, 0] + 0.5 * rng.random((1, 3))])
    src = np.concatenate([corners, rng.random((40, 3))])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 4000)
    assert tree.nodeCount <= 9
    q = rng.standard_normal(src.shape)
    f = nnk.KIFMM(tree, [1e-2, 1.0])
    s, t = tree.getPotentialPoints(), tree.getTargetPoints()
    ref, mod = _direct(s, q, t, 1e-2)
    assert (np.abs(f.computeVel(q) - ref) <= (len(s) + 40) * EPS * mod).all()
    # the leaf's own sources
    low_s, low_t = (s < 0.5).all(1), (t < 0.5).all(1)
    ref, mod = _direct(s[low_s], q[low_s], t[low_t], 1e-2)
    assert (np.abs(f.reducedComputeVel(q)[low_t] - ref) <= (len(s) + 40) * EPS * mod).all()


def test_more_blocks_than_a_grid_dimension(nnk):
    rng = np.random.default_rng(0)
    n = 32 * 65536 + 5
    tgt = 0.5 * rng.random((n, 3))
    src = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], rng.random((6, 3))])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 1 << 22)
    assert tree.nodeCount <= 9
    q = rng.standard_normal(src.shape)
    u = nnk.KIFMM(tree, [1e-2, 1.0]).computeVel(q)
    t = tree.getTargetPoints()
    some = np.r_[0:40, n - 100:n, rng.integers(0, n, 2000)]
    ref, mod = _direct(tree.getPotentialPoints(), q, t[some], 1e-2)
    assert (np.abs(u[some] - ref) <= 60 * EPS * mod).all()
    assert np.isfinite(u).all() and (np.abs(u).max(1) > 0).all()
