"""That the lists of the sharing tests are shared, and lists just below the
line are not (GPU)."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shared(nnk, fmm):
    st = ctypes.CDLL(os.path.join(os.path.dirname(nnk.library_path()), "libnnk_selftest.so"))
    a, b = ctypes.c_int(), ctypes.c_int()
    st.nnk_selftest_shared(fmm._handle().h, ctypes.byref(a), ctypes.byref(b))
    return a.value, b.value


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("big,sheet,cap", [(3, 9000, 6), (40, 9000, 50), (33, 12000, 40), (600, 12000, 620)])
def test_leaf_cases_share(nnk, big, sheet, cap, precision):
    """The trees of test_gpu_leaf_parts.test_shared_leaf."""
    rng = np.random.default_rng(big + sheet)
    thin = np.stack([0.5 + 0.004 * rng.random(sheet), rng.random(sheet), rng.random(sheet)], 1)
    own = 0.1 + 0.3 * rng.random((big, 3))
    p = np.concatenate([thin, [[0, 0, 0], [1, 1, 1.0]], own])
    tree = nnk.OcTree(p, p, "nodeCapacity", cap)
    leaves, _ = _shared(nnk, nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4, "precision", precision))
    assert leaves > 0


@pytest.mark.parametrize("shells", [1, 2])
@pytest.mark.parametrize("spot,shares", [(26000, True), (13000, False)])
def test_p2l_cases_share(nnk, spot, shares, shells):
    """The tree of test_gpu_leaf_parts.test_shared_p2l, and one whose X lists
    stay below 4,096 sources."""
    rng = np.random.default_rng(3)
    big = 0.02 + 0.47 * rng.random((6000 if shares else 3000, 3))
    dust = np.stack([0.5 + 0.12 * rng.random(spot), 0.3 * rng.random(spot), 0.3 * rng.random(spot)], 1)
    p = np.concatenate([[[0, 0, 0], [1, 1, 1.0]], big, dust])
    tree = nnk.OcTree(p, p, "nodeCapacity", 6100 if shares else 3100)
    cnt = np.bincount(tree.pointIndex, minlength=tree.nodeCount + 1)
    longest = max(sum(cnt[m] for m in tree.interactions.get(n, 4)) for n in range(1, tree.nodeCount + 1))
    print(f"[shared] longest X list {longest}", flush=True)
    assert longest > 4096 if shares else 0 < longest <= 4096
    _, x = _shared(nnk, nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4, "coronaShells", shells))
    assert (x > 0) == shares


def test_even_leaves_do_not_share(nnk):
    p = np.random.default_rng(1).random((20000, 3))
    tree = nnk.OcTree(p, p, "nodeCapacity", 64)
    assert _shared(nnk, nnk.KIFMM(tree, [1e-2, 1.0], "coronaRes", 4)) == (0, 0)
