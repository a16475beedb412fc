"""Direct sums at an eps whose inverse cube overflows (GPU): with sources and
targets apart the velocities are finite, as the kernel is then the unregularized
one.  Targets on grids of spacing one, so that a made-up source one unit beside
a target would meet another of its block."""
import numpy as np
import pytest

from test_gpu_direct64 import EPS, _direct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [1e-150, 1e-110, 1e-3])
@pytest.mark.parametrize("ns", [1, 63, 70, 300])
def test_leaf_targets_one_unit_apart(nnk, eps, ns):
    rng = np.random.default_rng(ns)
    # four targets at each x: a block of eight holds two neighbouring x
    tgt = np.stack(np.meshgrid(np.arange(16.0), np.arange(2.0), np.arange(2.0), indexing="ij"), -1).reshape(-1, 3)
    src = np.concatenate([[[-20, -20, -20], [60, 60, 60.0]], 17 + 3 * rng.random((ns, 3))])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 1024)
    assert tree.nodeCount <= 9
    q = rng.standard_normal(src.shape)
    u = nnk.KIFMM(tree, [eps, 1.0]).computeVel(q)
    ref, mod = _direct(tree.getPotentialPoints(), q, tree.getTargetPoints(), eps)
    assert (np.abs(u - ref) <= (len(src) + 40) * EPS * mod).all()


def test_surface_points_one_unit_apart(oracle, nnk):
    """A leaf of width 10 in the X lists of boxes of width 5: at six points an
    edge their surface points lie one unit apart."""
    rng = np.random.default_rng(2)
    wide, near = lambda n: 10 * rng.random((n, 3)), lambda n: 10 * rng.random((n, 3)) + [10, 0, 0]  # noqa: E731
    src = np.concatenate([[[0, 0, 0], [20, 20, 20.0]], wide(90), near(150)])
    tgt = np.concatenate([wide(5), near(150)])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 100)
    owners = [n for n in range(1, tree.nodeCount + 1) if len(tree.interactions.get(n, 4))]
    assert len(owners) >= 4 and (np.ptp(tree.nodeCorners[np.array(owners) - 1][:, [0, 3]], axis=1) == 5).all()
    q = rng.standard_normal(src.shape)
    u = nnk.KIFMM(tree, [1e-120, 1.0]).computeVel(q)
    uo = oracle.Tree(src, tgt, nodeCapacity=100).matvec(q, 1e-120, 1.0, 6, 1)
    assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)
