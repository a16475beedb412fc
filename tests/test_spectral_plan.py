"""Host planner of the frequency-space M2L (CPU: no GPU call).

The V lists regrouped by parent must name the same (target, source, offset)
pairs as the lists they came from, for any subset of parents, sources and
targets; lists that are not their parents' product sets are left to the
dense translations."""
import ctypes

import numpy as np
import pytest

from spectral_cases import arg, bits, library, make, tables


def _plan(st, c):
    head, tail = tables(c)
    n = c["n"]
    sizes, pairs = np.zeros(3, np.int32), np.zeros(2, np.int64)
    out = [np.zeros(max(n, 1), np.int32) for _ in range(4)] + [np.zeros(26 * max(n, 1), np.int32)]
    st.nnk_selftest_spectral_plan.restype = ctypes.c_int
    assert st.nnk_selftest_spectral_plan(*[arg(a) for a in head], ctypes.c_int32(c["count"]),
                                         *[arg(a) for a in tail], arg(sizes), arg(pairs), *[arg(a) for a in out]) == 0
    return sizes, pairs, out


@pytest.mark.parametrize("shape,pp,ps,pt", [((4, 4, 4), 1.0, 1.0, 1.0), ((5, 3, 4), 0.6, 0.7, 0.5),
                                            ((6, 6, 6), 0.3, 0.9, 0.9), ((2, 2, 2), 1.0, 0.5, 1.0),
                                            ((9, 1, 1), 1.0, 1.0, 0.1), ((3, 3, 3), 1.0, 0.0, 1.0),
                                            ((3, 3, 3), 1.0, 1.0, 0.0)])
def test_plan_covers_the_lists(nnk, shape, pp, ps, pt):
    st = library(nnk)
    c = make(np.random.default_rng(5), shape, pp, ps, pt)
    sizes, pairs, (tgt0, tmask, src0, smask, nb) = _plan(st, c)
    if not c["tgt"].any():
        assert not sizes[0]      # no targets: nothing to plan
        return
    assert sizes[0] and pairs[0] == len(c["pairs"])
    nt, ns = sizes[1], sizes[2]
    dirs = [(x, y, z) for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1) if (x, y, z) != (0, 0, 0)]
    got = []
    for d, dv in enumerate(dirs):
        for t in range(nt):
            s = nb[d * nt + t]
            assert -1 <= s < ns
            if s < 0:
                continue
            for a in range(8):
                for b in range(8):
                    o = tuple(2 * np.array(dv) + bits(b) - bits(a))
                    if (tmask[t] >> a) & 1 and (smask[s] >> b) & 1 and max(map(abs, o)) >= 2:
                        got.append((tgt0[t] + a, src0[s] + b, o))
    assert sorted(got) == sorted(c["pairs"])
    assert pairs[1] >= sum(1 for d in range(26) if (nb[d * nt:(d + 1) * nt] >= 0).any())


@pytest.mark.parametrize("what", ["missing", "foreign", "wrong child"])
def test_other_lists_stay_dense(nnk, what):
    st = library(nnk)
    c = make(np.random.default_rng(6), (3, 3, 3), 1.0, 1.0, 1.0)
    g = c["gv"][3]
    b, j = np.argwhere(g >= 0)[17]
    if what == "missing":
        g[b, j] = -1                        # one pair short of the product set
    elif what == "foreign":
        g[b, j] = (g[b, j] + 8) % (8 * c["n"])   # the right child of another parent
    else:
        g[b, j] ^= 1                        # another child of the right parent
    sizes, _, _ = _plan(st, c)
    assert not sizes[0]
