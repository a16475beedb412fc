"""Leaf blocks of growing condition number (GPU).  With X the computed inverse,
v - A X v is bounded by |I - A X| |v|, and for an inverse from LU factors
|I - A X| is at most about rows eps cond(A) (Higham, Accuracy and Stability of
Numerical Algorithms, section 14.3, growth of the factors aside)."""
import numpy as np
import pytest

from test_gpu_leaf_blocks import _dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,eps", [(30, 0.02), (30, 0.1), (30, 0.25), (30, 0.4), (30, 0.7), (300, 0.02), (300, 0.1),
                                   (300, 0.25), (300, 0.4)])
def test_residual_follows_the_condition(nnk, n, eps):
    rng = np.random.default_rng(n)
    p = np.concatenate([[[0, 0, 0]], 0.5 * rng.random((n - 1, 3)), [[1, 1, 1.0]]])
    tree = nnk.OcTree(p, p, "nodeCapacity", n + 1)
    v = rng.standard_normal(p.shape)
    f = np.asarray(nnk.KIFMM(tree, [eps, 1.0], "coronaRes", 3).reducedSolve(v)).reshape(-1, 3)
    p = tree.getPotentialPoints()
    low = (p < 0.5).all(1)
    A, b = _dense(p[low], eps), v[low].ravel()
    cond = np.linalg.cond(A)
    r = np.linalg.norm(A @ f[low].ravel() - b) / np.linalg.norm(b)
    print(f"[conditioning] rows {len(b)} eps {eps}: cond {cond:.1e}, residual {r:.1e}", flush=True)
    assert r <= len(b) * np.finfo(float).eps * cond
