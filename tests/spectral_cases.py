"""Random parent neighbourhoods for the tests of the frequency-space M2L."""
import ctypes
import os

import numpy as np

P = ctypes.POINTER


def slot_order():
    """The V-list offsets in the M2L's visiting order (parity classes, each
    along a boustrophedon path)."""
    out = []
    for p in range(8):
        vals = [[v for v in range(-3, 4) if (v & 1) == ((p >> s) & 1)] for s in (2, 1, 0)]
        row = 0
        for i, x in enumerate(vals[0]):
            ys = vals[1][::-1] if i & 1 else vals[1]
            for y in ys:
                zs = vals[2][::-1] if row & 1 else vals[2]
                row += 1
                out += [(x, y, z) for z in zs if max(abs(x), abs(y), abs(z)) >= 2]
    return out


def bits(c):
    return np.array([c >> 2, (c >> 1) & 1, c & 1])


def make(rng, shape, p_parent, p_src, p_tgt):
    """A level whose parents are a random subset of a grid: slots 8 i + c are
    the children of parent i, parents follow as slots; returns the tables
    the planner takes and the brute-force list of (target, source, offset)."""
    cells = np.stack(np.meshgrid(*map(np.arange, shape), indexing="ij"), -1).reshape(-1, 3)
    cells = cells[rng.random(len(cells)) < p_parent]
    n = len(cells)
    index = {tuple(c): i for i, c in enumerate(cells)}
    count = 9 * n
    parent = np.zeros(count, np.int32)
    child0 = np.full(count, -1, np.int32)
    for i in range(n):
        parent[8 * i:8 * i + 8] = 8 * n + i + 1   # 1-based ids
        child0[8 * n + i] = 8 * i
    has = np.zeros(count + 1, np.uint8)
    has[1:8 * n + 1] = rng.random(8 * n) < p_src
    tgt = rng.random(8 * n) < p_tgt
    order = slot_order()
    cls, gv, pairs = [], [], []
    for a in range(8):
        nodes = [8 * i + a for i in range(n) if tgt[8 * i + a]]
        offs = [o for o in order if all(-2 - g <= v <= 3 - g for v, g in zip(o, bits(a)))]
        assert len(offs) == 189
        g = np.full((189, len(nodes)), -1, np.int32)
        for j, t in enumerate(nodes):
            for b, o in enumerate(offs):
                pos = 2 * cells[t // 8] + bits(a) + o
                s = index.get(tuple(pos // 2))
                if s is None:
                    continue
                src = 8 * s + int(4 * (pos[0] & 1) + 2 * (pos[1] & 1) + (pos[2] & 1))
                if has[src + 1]:
                    g[b, j] = src
                    pairs.append((t, src, o))
        cls.append(np.array(nodes, np.int32))
        gv.append(g)
    return {"cells": cells, "n": n, "count": count, "parent": parent, "child0": child0, "has": has, "tgt": tgt,
            "cls": cls, "gv": gv, "pairs": pairs, "ncls": np.array([len(c) for c in cls], np.int32)}


def library(nnk):
    nnk.lib()
    return ctypes.CDLL(os.path.join(os.path.dirname(nnk.library_path()), "libnnk_selftest.so"))


def arg(a):
    return ctypes.c_void_p(a.ctypes.data)


def tables(c):
    """The planner's array arguments (kept alive by the caller)."""
    return [c["ncls"], np.concatenate(c["cls"]).astype(np.int32),
            np.concatenate([g.ravel() for g in c["gv"]]).astype(np.int32)], [c["parent"], c["child0"], c["has"]]
