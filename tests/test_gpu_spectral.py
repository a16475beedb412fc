"""The frequency-space M2L against explicit kernel sums (GPU).

chk[t] = sum over the V list of t of T u, with T the regularized Stokeslet
between the two up surfaces, on random parent neighbourhoods: every compiled
surface resolution, few and many parents (the wavefronts of a tile split the
directions or take parents each), two levels in one launch, absent parents,
children without sources or targets, and kx planes done in several launches.

Tolerance, a priori: per axis the transforms sum 2 res - 1 terms and the
products 26 x 48, so the 2-norm of a target's error is at most about
(6 (2 res - 1) + 1248) eps sum ||T||_F ||u||; 2000 eps of that sum covers
res <= 10."""
import ctypes

import numpy as np
import pytest

from spectral_cases import arg, library, make, tables

pytestmark = pytest.mark.gpu


def _codes(res):
    return [(ix, iy, iz) for iz in range(res) for ix in range(res) for iy in range(res)
            if not all(0 < v < res - 1 for v in (ix, iy, iz))]


def _kernel(r, eps, mu):
    r2 = (r * r).sum(-1)
    s = (r2 + eps * eps) ** -1.5 / (8 * np.pi * mu)
    T = r[..., :, None] * r[..., None, :] + (r2 + 2 * eps * eps)[..., None, None] * np.eye(3)
    T *= s[..., None, None]
    return T.transpose(0, 2, 1, 3).reshape(3 * r.shape[0], 3 * r.shape[1])


@pytest.mark.parametrize("res,shape,pp,levels,buf", [
    (3, (4, 4, 4), 0.8, 2, 4 << 30), (4, (7, 7, 6), 1.0, 1, 4 << 30), (4, (7, 7, 6), 0.9, 2, 1 << 20),
    (5, (3, 3, 3), 0.9, 1, 1), (6, (3, 3, 3), 1.0, 1, 4 << 30), (6, (7, 7, 7), 0.9, 1, 80 << 20),
    (7, (2, 2, 3), 1.0, 1, 4 << 30), (8, (2, 2, 2), 1.0, 2, 4 << 30), (9, (2, 2, 2), 1.0, 1, 4 << 30),
    (10, (2, 2, 2), 1.0, 1, 1)])
def test_matches_kernel_sums(nnk, res, shape, pp, levels, buf):
    st = library(nnk)
    rng = np.random.default_rng(100 * res + levels)
    c = make(rng, shape, pp, 0.85, 0.85)
    codes = _codes(res)
    K = 3 * len(codes)
    w, eps, mu = 0.37, 0.01, 1.3
    packed = np.array([x | y << 8 | z << 16 for x, y, z in codes], np.int32)
    up = rng.standard_normal((levels * c["count"], K))
    chk = np.full((levels * c["count"], K), 7.0)
    head, tail = tables(c)
    st.nnk_selftest_spectral_run.restype = ctypes.c_int
    print(f"[spectral] res {res} parents {c['n']} pairs {len(c['pairs'])}", flush=True)
    for _ in range(2):   # the second call on the same inputs gives the same bits
        out = chk.copy()
        assert st.nnk_selftest_spectral_run(
            *[arg(a) for a in head], ctypes.c_int32(c["count"]), *[arg(a) for a in tail], ctypes.c_int(res),
            arg(packed), ctypes.c_int(len(codes)), ctypes.c_double(w), ctypes.c_double(eps), ctypes.c_double(mu),
            ctypes.c_int(levels), ctypes.c_int64(buf), arg(up), arg(out)) == 0
        if _ == 0:
            first = out
    np.testing.assert_array_equal(out, first)
    per = {}
    for t, s, o in c["pairs"]:
        per.setdefault(t, []).append((s, o))
    targets = [t for t in range(8 * c["n"]) if c["tgt"][t]]
    rows = np.zeros(levels * c["count"], bool)
    for l in range(levels):
        rows[np.array(targets) + l * c["count"]] = True
    np.testing.assert_array_equal(out[~rows], 7.0)   # other nodes' rows untouched
    grid = np.array(codes, float)
    worst = 0.0
    for l in range(levels):
        wl = (l + 1) * w
        h = wl / (res - 1)
        for t in rng.choice(targets, 4 if res < 7 else 2, replace=False):
            ref, scale = np.zeros(K), 0.0
            for s, o in per.get(t, []):
                T = _kernel((grid[:, None, :] - grid[None, :, :]) * h - np.array(o) * wl, eps, mu)
                u = up[l * c["count"] + s]
                ref += T @ u
                scale += np.linalg.norm(T) * np.linalg.norm(u)
            err = np.linalg.norm(out[l * c["count"] + t] - ref)
            worst = max(worst, err / max(scale, 1e-300))
            assert err <= 2000 * np.finfo(float).eps * scale, (t, err, scale)
    print(f"[spectral] worst error / scale {worst:.2e}", flush=True)


@pytest.mark.parametrize("res", [4, 6])
def test_matvec_matches_dense_translations(nnk, res):
    """Whole matvecs with targets other than the sources on an adaptive tree:
    every level's M2L in frequency space against the dense class tiles.  The
    check-to-equivalent inverses amplify rounding by a factor of the tree, so
    the bound is the dense sums' own: four times what their summation order
    (split-K factors 1, 2, 4) moves the same result by."""
    rng = np.random.default_rng(3)
    p = np.concatenate([rng.normal(0.3, 0.02, (1500, 3)), rng.random((1500, 3))])
    t = np.concatenate([rng.random((2000, 3)), p[:300], rng.normal(0.6, 0.03, (700, 3))])
    tree = nnk.OcTree(p, t, "nodeCapacity", 20)
    q = rng.standard_normal((int(tree.potentials.sum()), 3))
    f = nnk.KIFMM(tree, [2e-3, 1.0], "coronaRes", res)
    lib, h = nnk.lib(), f._handle().h
    i32 = ctypes.POINTER(ctypes.c_int32)

    def config():
        s, d = np.zeros(16, np.int32), np.zeros(16, np.int32)
        assert lib.nnk_fmm_launch_config(h, s.ctypes.data_as(i32), d.ctypes.data_as(i32), 16) == 0
        return s, d

    def setcfg(s, d):
        return lib.nnk_fmm_set_launch_config(h, s.ctypes.data_as(i32), d.ctypes.data_as(i32), 16)

    s, d = config()
    on = (s > 0).astype(np.int32)
    u1 = f.computeVel(q)
    dense = []
    for split in (1, 2, 4):
        if setcfg(split * on, 0 * on) == 0:
            assert (config()[1][s > 0] == 0).all()
            dense.append(f.computeVel(q))
    assert len(dense) >= 2
    noise = max(np.linalg.norm(u - dense[0]) for u in dense[1:])
    off = np.linalg.norm(u1 - dense[0])
    print(f"[spectral] res {res}: off {off:.2e}, summation order {noise:.2e}", flush=True)
    assert 0 < noise and off <= 4 * noise
    assert setcfg(s, d) == 0      # the reported configuration brings the first launch back
    np.testing.assert_array_equal(f.computeVel(q), u1)
