"""Launch configurations changed under captured HIP graphs (GPU).

Switching a level from the frequency-space M2L to the dense one forms
operators and may move the split-K and pair buffers.  Graphs captured before
(the matvec's own, and the mobility solve's, which holds the kernels of two
operators) must not replay with the old launches or addresses, also when the
configuration is refused.  Each replay is compared bit for bit with an eager
operator of the same configuration, several times, with eager work between."""
import ctypes
from importlib import import_module

import numpy as np
import pytest

from geometry import blobs
from test_gpu_mobility import _system

pytestmark = pytest.mark.gpu
I32 = ctypes.POINTER(ctypes.c_int32)


def _config(nnk, h):
    s, d = np.zeros(16, np.int32), np.zeros(16, np.int32)
    assert nnk.lib().nnk_fmm_launch_config(h, s.ctypes.data_as(I32), d.ctypes.data_as(I32), 16) == 0
    return s, d


def _set(nnk, h, levels, split, depth):
    s, d = np.zeros(16, np.int32), np.zeros(16, np.int32)
    s[levels], d[levels] = split, depth
    return nnk.lib().nnk_fmm_set_launch_config(h, s.ctypes.data_as(I32), d.ctypes.data_as(I32), 16)


@pytest.mark.parametrize("kind", ["blobs", "uniform"])
def test_matvec_graph_follows_the_configuration(nnk, kind):
    rng = np.random.default_rng(21)
    p = blobs(rng) if kind == "blobs" else rng.random((20000, 3))
    t = nnk.OcTree(p, p, "nodeCapacity", 24)
    eager = nnk.KIFMM(t, [2e-3, 1.0], "coronaRes", 4)
    graph = nnk.KIFMM(t, [2e-3, 1.0], "coronaRes", 4, "hipGraph", 1)
    handles = [f._handle().h for f in (eager, graph)]
    levels = np.flatnonzero(_config(nnk, handles[0])[0])
    assert len(levels) >= 3

    def same():
        for _ in range(3):
            q = rng.standard_normal(p.shape)
            np.testing.assert_array_equal(graph.computeVel(q), eager.computeVel(q))

    def both(lv, split, depth):
        return [_set(nnk, h, lv, split, depth) for h in handles]

    same()
    # the smallest level first, split over K: its graph names the part buffer
    assert both(levels[:1], 2, 0) == [0, 0]
    same()
    assert all(r != 0 for r in both(levels[-1:], 65, 0))     # refused: beyond any split
    same()
    for lv in levels[1:]:     # refused, after planning, where it is past the part buffer
        r = both([lv], 64, 0)
        print(f"[config] level {lv} split 64: {r}", flush=True)
        assert r[0] == r[1]
        assert kind != "uniform" or lv != levels[-1] or r[0] != 0
        same()
    for lv in levels[::-1]:
        assert both([lv], 1, 0) == [0, 0]
        same()
    assert both(levels, 1, 1) == [0, 0]
    same()


def test_mobility_graph_follows_the_configuration(oracle, nnk):
    mob = import_module("stokes-nnkifmm_amd.mobility")
    systems = []
    for graph in (0, 1):
        sw, B, BT, A1, A2, _ = _system(nnk, oracle, True)
        sw.FMM.arguments["hipGraph"] = graph
        systems.append((sw, B, BT, A1, A2, mob._rhs(sw, lambda t, x: np.zeros_like(x), 0.0)))

    def same():
        x = [mob.mobility_gmres(*s, 1e-8, 300, True) for s in systems]
        np.testing.assert_array_equal(x[1], x[0])

    same()
    same()
    for split in (2, 1):
        for s in systems:
            fmm = s[0].FMM
            for h in (fmm._handle().h, fmm._handle(res=4).h):
                levels = np.flatnonzero(_config(nnk, h)[0])
                assert _set(nnk, h, levels[:1], split, 0) == 0
                if split == 1:
                    assert _set(nnk, h, levels, 1, 0) == 0
        same()
        same()


def test_depths_name_one_launch(oracle, nnk):
    """On a level in frequency space depth 1 is that, 2 its pair jobs, 0 class
    tiles; what is reported brings the same bits back.  Where there is no
    frequency-space M2L, 1 is the pair jobs and 2 is refused."""
    rng = np.random.default_rng(5)
    p = blobs(rng)
    t = nnk.OcTree(p, p, "nodeCapacity", 24)
    q = rng.standard_normal(p.shape)
    f = nnk.KIFMM(t, [2e-3, 1.0], "coronaRes", 6)
    h = f._handle().h
    s0, d0 = _config(nnk, h)
    levels = np.flatnonzero(s0)
    assert (s0[levels] == 1).all() and (d0[levels] == 1).all()
    u = f.computeVel(q)
    assert _set(nnk, h, levels, 1, 0) == 0
    tiles = f.computeVel(q)
    sparse = [lv for lv in levels if _set(nnk, h, [lv], 1, 2) == 0]
    print(f"[config] pair jobs on levels {sparse} of {levels.tolist()}", flush=True)
    assert sparse and all(_set(nnk, h, [lv], 2, 2) != 0 for lv in levels)
    s, d = _config(nnk, h)
    assert (s[sparse] == 1).all() and (d[sparse] == 2).all()
    pairs = f.computeVel(q)
    assert _set(nnk, h, levels, 1, 1) == 0
    np.testing.assert_array_equal(f.computeVel(q), u)
    assert _set(nnk, h, levels, s[levels], d[levels]) == 0     # as reported
    np.testing.assert_array_equal(f.computeVel(q), pairs)
    uo = oracle.Tree(p, p, nodeCapacity=24).matvec(q, 2e-3, 1.0, 6, 1)
    for v in (u, tiles, pairs):
        assert np.linalg.norm(v - uo) <= 1e-10 * np.linalg.norm(uo)

    # an autotuned mix of tiles and pair jobs replays from its report
    f = nnk.KIFMM(t, [2e-3, 1.0], "coronaRes", 6, "autotune", 1)
    h = f._handle().h
    assert _set(nnk, h, levels, 1, 0) == 0
    u = f.computeVel(q)
    s, d = _config(nnk, h)
    assert (d != 1).all()
    assert _set(nnk, h, levels, 1, 1) == 0
    assert _set(nnk, h, levels, s[levels], d[levels]) == 0
    np.testing.assert_array_equal(f.computeVel(q), u)

    f = nnk.KIFMM(t, [2e-3, 1.0], "coronaRes", 6, "coronaShells", 2)
    h = f._handle().h
    levels = np.flatnonzero(_config(nnk, h)[0])
    assert all(_set(nnk, h, [lv], 1, 2) != 0 for lv in levels)
    assert any(_set(nnk, h, [lv], 1, 1) == 0 for lv in levels)
