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
