"""The leaf-block solve in each of its launch shapes (GPU): a leaf per
workgroup at 128 to 512 threads (leaves of different sizes, up to the last row
of each shape), eight wavefronts per 64 rows, and a thread per row (many leaves,
or inverses of gigabytes), against dense solves of some leaves at the
preconditioner's 1e-10."""
import numpy as np
import pytest

from test_gpu_leaf_blocks import _dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,sizes,eps", [
    (16, [21, 5, 6, 10], 0.01),                   # 4,096 leaves of at most 63 rows
    (16, [42, 8, 22, 11], 0.01), (8, [85, 43, 64, 70], 0.015),
    (8, [106, 30, 86, 40], 0.01),                 # 512 threads: one to five share a row
    (8, [170, 60, 107, 90], 0.008),               # a thread per row: 510 rows
    (8, [21, 5, 6, 10], 0.02), (4, [86, 30], 0.03), (4, [341, 100], 0.02),   # few: eight wavefronts
    (4, [700], 0.02)])                            # 2.3 GB
def test_shapes(nnk, cells, sizes, eps):
    rng = np.random.default_rng(cells + sizes[0])
    grid = np.stack(np.meshgrid(*[np.arange(cells)] * 3, indexing="ij"), -1).reshape(-1, 3)
    count = rng.choice(sizes[1:] or sizes, len(grid))
    count[::17] = sizes[0]
    count[3] = 1 if cells >= 8 else sizes[0]      # a parent's points are still more than the largest leaf's
    p = (np.repeat(grid, count, axis=0) + rng.random((count.sum(), 3))) / cells
    tree = nnk.OcTree(p, p, "nodeCapacity", max(sizes), "rootCube", [0.0, 1.0])
    assert tree.nodeCount == (8 * cells ** 3 - 1) // 7
    v = rng.standard_normal(p.shape)
    f = np.asarray(nnk.KIFMM(tree, [eps, 1.0], "coronaRes", 3).reducedSolve(v)).reshape(-1, 3)
    p = tree.getPotentialPoints()
    cell = np.floor(p * cells).astype(int) @ [cells * cells, cells, 1]
    for c in [0, 1, 2, 3, 17] + list(rng.choice(len(grid), 4, replace=False)):
        sel = cell == c
        assert sel.sum() == count[c]
        x = np.linalg.solve(_dense(p[sel], eps), v[sel].ravel())
        assert np.linalg.norm(f[sel].ravel() - x) <= 1e-10 * np.linalg.norm(x)
