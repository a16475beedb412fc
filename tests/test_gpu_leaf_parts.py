"""Leaves shared by several workgroups (GPU): a large leaf whose face touches
a sheet of small ones has a source list many times the others'.  Few and many
targets in it (one workgroup block of 32, several, more than one pass of the
FP32-math kernel), U lists below and above 512 leaves, against the oracle at
each form's bound, and the same product twice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-10), ("mixed", 1e-4)])
@pytest.mark.parametrize("big,sheet,cap", [(3, 9000, 6), (40, 9000, 50), (33, 12000, 40), (600, 12000, 620)])
def test_shared_leaf(oracle, nnk, big, sheet, cap, precision, bound):
    rng = np.random.default_rng(big + sheet)
    thin = np.stack([0.5 + 0.004 * rng.random(sheet), rng.random(sheet), rng.random(sheet)], 1)
    own = 0.1 + 0.3 * rng.random((big, 3))
    p = np.concatenate([thin, [[0, 0, 0], [1, 1, 1.0]], own])
    tree = nnk.OcTree(p, p, "nodeCapacity", cap)
    q = rng.standard_normal(p.shape)
    fmm = nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4, "precision", precision)
    u = fmm.computeVel(q)
    uo = oracle.Tree(p, p, nodeCapacity=cap).matvec(q, 1e-2, 1.0, 4, 1)
    mine = slice(len(p) - big, len(p))
    assert np.linalg.norm(u - uo) <= bound * np.linalg.norm(uo)
    assert np.linalg.norm(u[mine] - uo[mine]) <= bound * np.linalg.norm(uo[mine])
    assert np.array_equal(u, fmm.computeVel(q))


@pytest.mark.parametrize("shells", [1, 2])
def test_shared_p2l(oracle, nnk, shells):
    """Three nodes with X lists of 4,282 to 7,941 sources: P2L's own sharing,
    added onto the check potentials of the frequency-space M2L (one shell) and
    through the separate buffer beside the dense one (two)."""
    rng = np.random.default_rng(3)
    big = 0.02 + 0.47 * rng.random((6000, 3))
    spot = np.stack([0.5 + 0.12 * rng.random(26000), 0.3 * rng.random(26000), 0.3 * rng.random(26000)], 1)
    p = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], big, spot])
    tree = nnk.OcTree(p, p, "nodeCapacity", 6100)
    owners = [n for n in range(1, tree.nodeCount + 1) if len(tree.interactions.get(n, 4))]
    assert len(owners) >= 3
    q = rng.standard_normal(p.shape)
    u = nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4, "coronaShells", shells).computeVel(q)
    uo = oracle.Tree(p, p, nodeCapacity=6100).matvec(q, 1e-2, 1.0, 4, shells)
    assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)
