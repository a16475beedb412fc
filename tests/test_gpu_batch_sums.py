"""The batched pair sums at the sizes where their tiles, runs and parts end
(GPU): 64-target tiles, four interleaved source runs read three records at a
time (FP64), contiguous source parts of at least 512 sources and groups of
four (FP32 math).  Force-point rows against the sums in numpy, per component
within (sources + 40) eps of the sum of the terms' moduli (FP64) or 1e-6 of
it (FP32 math: about ten roundings of 2^-24 a term); the transpose by
<y, A x> = <A^T y, x>."""
import importlib

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps

SIZES = [(1, 1), (2, 3), (5, 7), (63, 12), (64, 13), (65, 130), (130, 511), (7, 512), (9, 513), (64, 1030),
         (200, 2050), (70, 4099)]


def _system(nnk, rng, n, q):
    pts, fine = rng.standard_normal((n, 3)), rng.standard_normal((q, 3))
    NN = sp.csr_matrix((rng.random(q), (np.arange(q), rng.integers(0, n, q))), shape=(q, n))
    sw = nnk.Swimmers()
    frame, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    sw.addSwimmer(pts, fine, NN, rng.standard_normal(3), np.concatenate([frame[:, 0], frame[:, 1]]),
                  np.zeros_like(pts), np.zeros(3), np.zeros(3))
    return sw


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes", [SIZES, SIZES[5:6], SIZES[-1:], SIZES[:3]])
def test_pair_sums(nnk, precision, sizes):
    rng = np.random.default_rng(len(sizes))
    systems = [_system(nnk, rng, n, q) for n, q in sizes]
    eps = rng.uniform(0.01, 0.1, len(sizes))
    bm = nnk.BatchedMobility(systems, eps, precision=precision, hipGraph=False)
    x, z = rng.standard_normal(bm.n), rng.standard_normal(bm.n)
    y, t = bm.apply(x), bm.apply(z, transpose=True)
    np.testing.assert_array_equal(bm.apply(x), y)
    for sw, e, xp, yp in zip(systems, eps, bm.split(x), bm.split(y)):
        pts, fine, NN, rot, _ = sw.getSwimmers()
        n = len(pts)
        f = np.asarray(NN @ xp[:3 * n].reshape(3, n).T)
        r = pts[:, None, :] - fine[None, :, :]
        r2 = (r * r).sum(2)
        s = (r2 + e * e) ** -1.5 / (8 * np.pi)
        iso = ((r2 + 2 * e * e) * s)[:, :, None]
        u = (iso * f + ((r * f).sum(2) * s)[:, :, None] * r).sum(1)
        mod = (iso * np.abs(f) + (np.abs(r * f).sum(2) * s)[:, :, None] * np.abs(r)).sum(1)
        U, W = xp[3 * n:3 * n + 3], xp[3 * n + 3:]
        rigid = U + np.cross(W, rot)
        mod = mod + np.abs(U) + np.abs(W).sum() * np.abs(rot).sum(1, keepdims=True)
        tol = (len(fine) + 40) * EPS if precision == "fp64" else 1e-6
        assert (np.abs(yp[:3 * n].reshape(3, n).T - (u - rigid)) <= tol * mod).all(), (n, len(fine))
    scale = np.linalg.norm(z) * np.linalg.norm(y)
    assert abs(z @ y - t @ x) <= (1e-13 if precision == "fp64" else 1e-6) * scale
