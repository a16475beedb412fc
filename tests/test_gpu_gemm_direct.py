"""The direct FP64 gather GEMM against the host product, in each of its three
launch shapes (GPU): remainders of the 16-row tiles, the 16-deep chunks and
the column tiles, ranks below one load, absent sources, jobs of different
widths.  The bound is a priori: (nb K + 8) eps times the sum of the terms'
moduli.  Columns that no job reads, and what lies past a column's K values,
are NaN: nothing of them may arrive."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def selftest(nnk):
    nnk.lib()
    return ctypes.CDLL(os.path.join(os.path.dirname(nnk.library_path()), "libnnk_selftest.so"))


@pytest.mark.parametrize("M,K,nb,widths,beta", [
    (24, 24, 8, (1,), 0), (2, 3, 1, (5,), 0), (3, 2, 8, (17, 3), 1), (33, 4, 2, (16,), 0), (168, 168, 8, (37,), 0),
    (456, 456, 1, (64, 9, 0, 31), 1), (456, 30, 3, (101,), 1), (17, 1158, 1, (2,), 0),        # 32 x 16, eight wavefronts
    (168, 168, 8, (2050,), 0), (456, 60, 1, (200, 1030, 7), 1), (456, 456, 2, (831,), 1),     # 48 x 32, four wavefronts
    (24, 24, 8, (65500,), 0), (456, 168, 2, (6530,), 1), (100, 2, 1, (22000,), 0),            # 48 x 128, one
])
def test_direct_gemm(selftest, M, K, nb, widths, beta):
    c, ref, mod = _run(selftest, M, K, nb, widths, beta, 0)
    assert (np.abs(c - ref) <= (nb * K + 8) * EPS * mod).all()


@pytest.mark.parametrize("M,K,nb,widths,beta", [
    (24, 24, 8, (1,), 0), (2, 3, 1, (5,), 0), (3, 2, 8, (17, 3), 1), (33, 4, 2, (16,), 0), (168, 168, 8, (65,), 0),
    (457, 457, 1, (64, 9, 0, 200), 1), (456, 30, 3, (101,), 1), (17, 1158, 1, (130,), 0)])
def test_ordered_gemm(selftest, M, K, nb, widths, beta):
    """The ordered launch has the bits of the kernel whose order it keeps."""
    c, ref, mod = _run(selftest, M, K, nb, widths, beta, 1)
    assert (np.abs(c - ref) <= (nb * K + 8) * EPS * mod).all()
    assert np.array_equal(c, _run(selftest, M, K, nb, widths, beta, 2)[0])


def _run(selftest, M, K, nb, widths, beta, ordered):
    rng = np.random.default_rng(M * K + nb)
    Mpad, Kpad, ldx, ldc = -(-M // 160) * 160, -(-K // 16) * 16, max(K, 32) + 2, M + 3
    nx, nc = 60, sum(widths) + 4
    at = np.zeros((nb, Kpad, Mpad))
    at[:, :K, :M] = rng.standard_normal((nb, K, M))
    x = np.full((nx, ldx), np.nan)
    x[1:, :K] = rng.standard_normal((nx - 1, K))
    g = [rng.integers(1, nx, (nb, n)) * (rng.random((nb, n)) < 0.7) for n in widths]
    g = [np.where(t == 0, -1, t).astype(np.int32) for t in g]
    slots = rng.permutation(nc)[:sum(widths)].astype(np.int32)
    c0 = rng.standard_normal((nc, ldc))
    ref, mod = c0.copy(), np.abs(c0)
    xs = np.vstack([x[1:, :K], np.zeros((1, K))])   # row -1: no source
    gall = np.concatenate([np.where(t < 0, 0, t) - 1 for t in g], axis=1)
    acc = sum(xs[gall[b]] @ at[b, :K, :M] for b in range(nb))
    absum = sum(np.abs(xs[gall[b]]) @ np.abs(at[b, :K, :M]) for b in range(nb))
    ref[slots, :M] = acc + beta * c0[slots, :M]
    mod[slots, :M] = absum + beta * np.abs(c0[slots, :M])
    c = c0.copy()
    d, ip = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
    gf = np.concatenate([t.ravel() for t in g])
    w = np.array(widths, np.int32)
    assert selftest.nnk_selftest_gemm_direct(
        M, K, Mpad, Kpad, at.ctypes.data_as(d), nb, x.ctypes.data_as(d), nx, ldx, gf.ctypes.data_as(ip),
        slots.ctypes.data_as(ip), w.ctypes.data_as(ip), len(widths), c.ctypes.data_as(d), nc, ldc, beta, ordered) == 0
    return c, ref, mod
