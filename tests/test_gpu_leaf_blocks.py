"""The leaf-block preconditioner at the sizes where its panels, tiles and
launch shapes end (GPU): blocks of 3 rows to past the 1,024 a panel holds in
registers, against a dense solve at the preconditioner's 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dense(p, eps):
    r = p[:, None, :] - p[None, :, :]
    r2 = (r * r).sum(2)
    s = (r2 + eps * eps) ** -1.5 / (8 * np.pi)
    A = np.einsum("ij,ijp,ijq->ipjq", s, r, r) + np.einsum("ij,pq->ipjq", (r2 + 2 * eps * eps) * s, np.eye(3))
    return A.reshape(3 * len(p), 3 * len(p))


@pytest.mark.parametrize("nt", [2, 5, 6, 10, 11, 21, 22, 43, 64, 85, 86, 171, 200, 341, 342, 400])
def test_block_sizes(nnk, nt):
    rng = np.random.default_rng(nt)
    own = np.concatenate([[[0, 0, 0]], 0.5 * rng.random((nt - 1, 3))])   # one leaf, larger than the others
    other = np.concatenate([[[1, 1, 1.0]], 0.5 + 0.5 * rng.random((min(nt - 1, 40), 3))])
    p = np.concatenate([own, other])
    tree = nnk.OcTree(p, p, "nodeCapacity", nt)
    assert tree.nodeCount == 9
    p = tree.getPotentialPoints()
    v = rng.standard_normal(p.shape)
    f = np.asarray(nnk.KIFMM(tree, [0.05, 1.0]).reducedSolve(v)).reshape(-1, 3)
    low = (p < 0.5).all(1)
    for sel in (low, ~low):
        x = np.linalg.solve(_dense(p[sel], 0.05), v[sel].ravel())
        assert np.linalg.norm(f[sel].ravel() - x) <= 1e-10 * np.linalg.norm(x)
