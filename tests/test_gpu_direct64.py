"""The FP64 direct-sum kernels of the matvec at the sizes where their blocks
and batches end (GPU).

Leaf kernel: 1, 2 or 4 blocks of at most 8 targets and 32 targets per
workgroup; sources in batches of 256 and chunks of 64, U lists in parts of
512 leaves.  A root-and-8-leaves tree has no far field, so the matvec is the
direct sum; the bound is a priori: (sources + 40) eps times the sum of the
terms' moduli.  P2L and S2M: surfaces whose point count is no multiple of a
block or a wavefront, against the oracle at the FP64 form's 1e-10."""
import numpy as np
import pytest

from geometry import blobs

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _direct(src, q, tgt, eps):
    """Velocities and, per component, the sum of the terms' moduli."""
    r = tgt[:, None, :] - src[None, :, :]
    r2 = (r * r).sum(2)
    s = (r2 + eps * eps) ** -1.5 / (8 * np.pi)
    a = ((r2 + 2 * eps * eps) * s)[:, :, None] * q
    b = ((r * q).sum(2) * s)[:, :, None] * r
    mod = ((r2 + 2 * eps * eps) * s)[:, :, None] * np.abs(q) + (np.abs(r * q).sum(2) * s)[:, :, None] * np.abs(r)
    return (a + b).sum(1), mod.sum(1)


@pytest.mark.parametrize("nt,ns", [(1, 1), (2, 63), (5, 64), (6, 65), (7, 255), (8, 256), (14, 257), (15, 300),
                                   (29, 511), (32, 512), (33, 513), (64, 100), (65, 700), (100, 64)])
def test_leaf_block_edges(nnk, nt, ns):
    rng = np.random.default_rng(1000 * nt + ns)
    corners = np.array([[0, 0, 0], [1, 1, 1.0]])
    src = np.concatenate([corners, 0.5 + 0.5 * rng.random((ns, 3))])[:max(ns, 2)]
    tgt = np.concatenate([0.5 * rng.random((nt, 3))])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 1024)
    assert tree.nodeCount <= 9
    q = rng.standard_normal(src.shape)
    u = nnk.KIFMM(tree, [1e-2, 1.0]).computeVel(q)
    ref, mod = _direct(tree.getPotentialPoints(), q, tree.getTargetPoints(), 1e-2)
    assert (np.abs(u - ref) <= (len(src) + 40) * EPS * mod).all()


def test_reduced_product_and_empty_leaves(nnk):
    """reducedComputeVel takes the leaf's own sources only; leaves with
    targets and no sources get zero."""
    rng = np.random.default_rng(4)
    src = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], 0.1 * rng.random((70, 3))])
    tgt = np.concatenate([0.1 * rng.random((40, 3)), 0.6 + 0.1 * rng.random((9, 3))])
    tree = nnk.OcTree(src, tgt, "nodeCapacity", 1024)
    q = rng.standard_normal(src.shape)
    u = nnk.KIFMM(tree, [1e-2, 1.0]).reducedComputeVel(q)
    t = tree.getTargetPoints()
    low = (t < 0.5).all(1)
    own = (src < 0.5).all(1)
    ref, mod = _direct(src[own], q[own], t[low], 1e-2)
    assert (np.abs(u[low] - ref) <= 120 * EPS * mod).all()
    far, fmod = _direct(src[1:2], q[1:2], t[~low], 1e-2)   # the corner (1, 1, 1) is those targets' own leaf
    assert (np.abs(u[~low] - far) <= 50 * EPS * fmod).all()


def test_more_than_512_u_leaves(oracle, nnk):
    """A large leaf whose face touches a sheet of small ones."""
    rng = np.random.default_rng(8)
    sheet = np.stack([0.5 + 0.004 * rng.random(6000), rng.random(6000), rng.random(6000)], 1)
    far = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], [0.1, 0.1, 0.1] + 0.3 * rng.random((5, 3))])
    p = np.concatenate([sheet, far])
    tree = nnk.OcTree(p, p, "nodeCapacity", 6)
    u_len = [len(tree.interactions.get(n, 1)) for n in range(1, tree.nodeCount + 1)]
    assert max(u_len) > 512, max(u_len)
    q = rng.standard_normal(p.shape)
    u = nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4).computeVel(q)
    uo = oracle.Tree(p, p, nodeCapacity=6).matvec(q, 1e-2, 1.0, 4, 1)
    assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)


@pytest.mark.parametrize("res", [3, 5])
def test_surface_point_counts(oracle, nnk, res):
    """26 and 98 surface points: partial blocks of P2L and wavefronts of S2M."""
    p = blobs(np.random.default_rng(21))
    tree = nnk.OcTree(p, p, "nodeCapacity", 16)
    assert any(len(tree.interactions.get(n, 4)) for n in range(1, tree.nodeCount + 1))
    q = np.random.default_rng(22).standard_normal(p.shape)
    u = nnk.KIFMM(tree, [1e-3, 1.0], "coronaRes", res).computeVel(q)
    uo = oracle.Tree(p, p, nodeCapacity=16).matvec(q, 1e-3, 1.0, res, 1)
    assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)


@pytest.mark.parametrize("cap,n", [(100, 4500), (180, 9000), (400, 20000)])
def test_s2m_of_large_leaves(oracle, nnk, cap, n):
    """Leaves of 64 sources and more on average take their sources on lanes:
    chunks of 64 and batches of 256, with remainders."""
    rng = np.random.default_rng(n + cap)
    p = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], rng.random((n, 3))])
    tree = nnk.OcTree(p, p, "nodeCapacity", cap)
    assert tree.nodeCount == 73   # 64 leaves
    q = rng.standard_normal(p.shape)
    u = nnk.KIFMM(tree, [1e-3, 1.0], "coronaRes", 4).computeVel(q)
    uo = oracle.Tree(p, p, nodeCapacity=cap).matvec(q, 1e-3, 1.0, 4, 1)
    assert np.linalg.norm(u - uo) <= 1e-10 * np.linalg.norm(uo)
