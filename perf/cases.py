"""The work that users of this framework run, as measurable cases.

Every case goes through the public Python API (OcTree, KIFMM, Swimmers,
mobility_gmres, mobilityProblem, BatchedMobility) with the options a program
sets.  listed() spans the range from launch-bound matvecs to 2^20 points,
uniform, clustered and surface point sets, plain and nearest-quadrature
sources, FP64 and the mixed forms, single matvecs and whole solves, forward
and adjoint.  draw() gives more cases of the same kinds and ranges.

Kinds:
  uniform      matvec of points uniform in the unit cube, sources = targets
               (the FMM-matvec configuration)
  clustered    matvec of two Gaussian clusters over a uniform background
               (adaptive tree with W and X lists)
  flow_field   velocities of forces on spheroid surfaces at the points of a
               grid around them: sources and targets disjoint
               (Data Generation/FlowField.m)
  suspension   matvec of spheroids above a wall with nearest quadrature, on
               the solver's vector layout: one GMRES iteration's main cost
  mobility     the preconditioned mobility solve of such a suspension
  time_step    one right-hand side of the squirmer suspension in a closed
               box (Data Generation/Squiremers.m): tree, operators and solve
  batch        independent single-body problems solved at once
  adjoint      squirmer pair: forward solve, transpose solve, gradients with
               respect to node positions and eps
"""
import ctypes
import importlib

import numpy as np
import torch

nnk = importlib.import_module("stokes-nnkifmm_amd")
geo = importlib.import_module("stokes-nnkifmm_amd.geometries")
mob = importlib.import_module("stokes-nnkifmm_amd.mobility")

# direct sums above this many pairs take too long in plain torch
MAX_EXACT_PAIRS = 4.0e10
PAIR_FLOPS = 33.0


def listed():
    return [
        # smallest: a few thousand points, a handful of launches; what a user
        # tries first and what a small body costs per GMRES iteration
        {"name": "uniform_3k_fp64", "kind": "uniform", "n": 3000, "capacity": 32, "res": 6, "precision": "fp64"},
        # ordinary: an odd count with the default node capacity
        {"name": "uniform_65k_fp64", "kind": "uniform", "n": 65537, "capacity": 200, "res": 6, "precision": "fp64"},
        # the FMM-matvec configuration at its stated size, the reference's numbers
        {"name": "uniform_1m_fp64", "kind": "uniform", "n": 1 << 20, "capacity": 64, "res": 6, "precision": "fp64"},
        # the same in the fastest form below 1e-6 (what the benchmark quotes), tuned as a long run would
        {"name": "uniform_1m_mixedh", "kind": "uniform", "n": 1 << 20, "capacity": 64, "res": 9,
         "precision": "mixedh", "svd_tol": 3e-7, "autotune": 1},
        # adaptive cloud in the three-part form (the other form below 1e-6)
        {"name": "clustered_100k_mixed3", "kind": "clustered", "n": 100003, "capacity": 40, "res": 8,
         "precision": "mixed3", "svd_tol": 1e-8},
        # post-processing: velocities on a grid around swimmers
        {"name": "flow_field_fp64", "kind": "flow_field", "bodies": 10, "side": 9, "grid": 41, "capacity": 64,
         "res": 6, "precision": "fp64"},
        # one GMRES iteration's matvec of the 64-spheroid suspension (126k force / 2M quadrature points)
        {"name": "suspension_64_fp64", "kind": "suspension", "bodies": 64, "side": 18, "box": 20.0, "wall": 40,
         "res": 6, "precision": "fp64"},
        # the inner iteration of its flexible-GMRES solve, at a third of the bodies
        {"name": "suspension_20_mixed", "kind": "suspension", "bodies": 20, "side": 18, "box": 14.0, "wall": 28,
         "res": 6, "precision": "mixed", "svd_tol": 1e-8},
        # a whole preconditioned solve
        {"name": "mobility_8_fp64", "kind": "mobility", "bodies": 8, "side": 12, "box": 9.0, "wall": 20,
         "res": 6, "tol": 1e-6},
        # what ode45 calls at every stage
        {"name": "time_step_10", "kind": "time_step", "bodies": 10, "wall_h": 0.3, "capacity": 500, "maxit": 50},
        # many small problems at once
        {"name": "batch_24_fp64", "kind": "batch", "problems": 24, "nmin": 200, "nmax": 5000, "tol": 1e-6,
         "precision": "fp64"},
        # gradients for design and control, in the FP32-math form
        {"name": "adjoint_pair_mixed", "kind": "adjoint", "side": 12, "gap": 0.5, "tol": 1e-6,
         "precision": "mixed"},
    ]


def _loguniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "clustered", "flow_field", "suspension", "suspension", "mobility",
                       "time_step", "batch", "adjoint"])
    prec = rng.choice(["fp64", "fp64", "fp64", "fp64t", "mixed", "mixed3", "mixedh"])
    form = {"precision": prec, "res": 6 if prec in ("fp64", "mixed") else rng.choice([8, 9])}
    if prec != "fp64":
        form["svd_tol"] = 3e-7 if form["res"] == 9 else 1e-8
    if kind == "uniform":
        return {"kind": kind, "n": int(_loguniform(rng, 1000, 300000)), "capacity": rng.choice([32, 40, 64, 100, 200]),
                **form}
    if kind == "clustered":
        return {"kind": kind, "n": int(_loguniform(rng, 2000, 200000)), "capacity": rng.choice([24, 40, 64, 200]),
                **form}
    if kind == "flow_field":
        return {"kind": kind, "bodies": rng.randint(1, 20), "side": rng.randint(6, 14), "grid": rng.randint(13, 47),
                "capacity": rng.choice([64, 100, 200]), **form}
    if kind == "suspension":
        return {"kind": kind, "bodies": rng.randint(2, 40), "side": rng.randint(8, 18), "box": 16.0 + rng.randint(0, 4),
                "wall": rng.randint(12, 40), **form}
    if kind == "mobility":
        return {"kind": kind, "bodies": rng.randint(1, 8), "side": rng.randint(5, 12), "box": 8.0 + rng.randint(0, 3),
                "wall": rng.randint(6, 20), "res": rng.choice([4, 6]), "tol": 1e-6}
    if kind == "time_step":
        return {"kind": kind, "bodies": rng.randint(2, 12), "wall_h": round(rng.uniform(0.3, 0.6), 3),
                "capacity": rng.choice([200, 350, 500]), "maxit": 50}
    if kind == "batch":
        return {"kind": kind, "problems": rng.randint(2, 24), "nmin": 200, "nmax": rng.randint(500, 5000),
                "tol": 1e-6, "precision": rng.choice(["fp64", "mixed"])}
    return {"kind": "adjoint", "side": rng.randint(5, 12), "gap": round(rng.uniform(0.3, 1.0), 3), "tol": 1e-6,
            "precision": rng.choice(["fp64", "mixed"])}


# -- inputs ------------------------------------------------------------------

def _generator(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _points(case, rng):
    """(sources, targets) of the plain matvec kinds."""
    if case["kind"] == "uniform":
        p = rng.random((case["n"], 3))
        return p, p
    if case["kind"] == "clustered":
        n = case["n"]
        na, nb = int(0.4 * n), int(0.3 * n)
        p = np.concatenate([0.3 + 0.02 * rng.standard_normal((na, 3)), 0.7 + 0.05 * rng.standard_normal((nb, 3)),
                            rng.random((n - na - nb, 3))])
        return p, p
    body = geo.prolate_spheroid(case["side"], 0.5, 1.0)
    centres, b1, b2 = geo.random_frames(case["bodies"], 12.0, 2.1, -5.0, int(rng.integers(1 << 30)))
    frames = np.stack([b1, b2, np.cross(b1, b2)], 2)
    src = np.concatenate([body @ f.T + c for f, c in zip(frames, centres)])
    g = np.linspace(-6.5, 12.5, case["grid"])
    X, Y, Z = np.meshgrid(g - 3.0, g - 3.0, g, indexing="ij")
    return src, np.stack([X.ravel(), Y.ravel(), Z.ravel()], 1)


def _forces(case, rng, n):
    if case["kind"] != "flow_field":
        return rng.standard_normal((n, 3))
    # a body's traction varies little over its surface
    body = rng.standard_normal((case["bodies"], 3)).repeat(n // case["bodies"], axis=0)
    return body * (1.0 + 0.1 * rng.standard_normal((n, 1)))


def _bodies(case, rng):
    """Bodies of fixed sizes and shapes; frames, loads and eps from rng."""
    bodies, _ = geo.batch_bodies(nprob=case["problems"], nmin=case["nmin"], nmax=case["nmax"])
    for sw in bodies:
        frame, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        load = rng.standard_normal((2, 3))
        load /= np.linalg.norm(load, axis=1, keepdims=True)
        sw.updateSwimmmer(1, rng.uniform(-5, 5, 3), np.concatenate([frame[:, 0], frame[:, 1]]))
        sw.F[0], sw.Moment[0] = load[0], 0.1 * load[1]
    return bodies, rng.uniform(0.002, 0.02, len(bodies))


def _spheroids(case, seed):
    force = _generator(seed + 1).standard_normal(3)
    return geo.spheroid_suspension(nbody=case["bodies"], n=case["side"], box=case["box"], wall_n=case["wall"],
                                   seed=seed, force=tuple(force / np.linalg.norm(force)))


def _kifmm_options(case):
    opt = {"coronaRes": case["res"], "precision": case["precision"]}
    if "svd_tol" in case:
        opt["svdTol"] = case["svd_tol"]
    if case.get("autotune"):
        opt["autotune"] = 1
    return opt


EPS = {"uniform": 1e-3, "clustered": 1e-3, "flow_field": 0.01, "suspension": 0.005, "mobility": 0.005,
       "time_step": 0.1, "adjoint": 0.01}


def prepare(case, seed):
    kind = case["kind"]
    rng = _generator(seed)
    if kind in ("uniform", "clustered", "flow_field"):
        src, tgt = _points(case, rng)
        q = torch.from_numpy(_forces(case, rng, len(src))).cuda()
        tree = nnk.OcTree(src, tgt, "nodeCapacity", case["capacity"])
        fmm = nnk.KIFMM(tree, [EPS[kind], 1.0], **_kifmm_options(case))
        fmm.computeVel(torch.ones_like(q))   # builds (and tunes) the operator, which the program keeps
        return {"kind": kind, "fmm": fmm, "q": q}
    if kind in ("suspension", "mobility"):
        sw = _spheroids(case, seed)
        sw.genTree("nodeCapacity", 64, "nearest", 1)
        form = _kifmm_options(case) if kind == "suspension" else {"coronaRes": case["res"]}
        sw.genKIFMM([EPS[kind], 1.0], "GMRES", 1, "format", 2, *[v for kv in form.items() for v in kv])
        if kind == "suspension":
            q = torch.from_numpy(rng.standard_normal(3 * len(sw.Tree.points))).cuda()
            sw.FMM.computeVel(torch.ones_like(q))
            return {"kind": kind, "sw": sw, "fmm": sw.FMM, "q": q}
        B, BT, A1, A2 = nnk.genMatrixComponets(sw)
        b = mob._rhs(sw, lambda t, x: np.zeros_like(x), 0.0)
        return {"kind": kind, "sw": sw, "sys": (B, BT, A1, A2), "b": b, "tol": case["tol"]}
    if kind == "time_step":
        nnk.operatorCache(8 << 30)   # as a time-stepping program does: the walls fix the root box
        sw, y0 = geo.squirmer_box(nsw=case["bodies"], seed=seed, wall_h=case["wall_h"])
        return {"kind": kind, "sw": sw, "y0": y0, "tree": ["nodeCapacity", case["capacity"], "nearest", 1],
                "maxit": case["maxit"]}
    if kind == "batch":
        bodies, eps = _bodies(case, rng)
        bm = nnk.BatchedMobility(bodies, eps, precision=case["precision"], hipGraph=True)
        return {"kind": kind, "bm": bm, "b": bm.rhs(), "tol": case["tol"], "bodies": bodies, "eps": eps}
    B1, B2 = rng.uniform(0.5, 2.0), rng.uniform(-5.0, 5.0)
    sw = geo.squirmer_pair(n=case["side"], refine=4, gap=case["gap"], B1=B1, B2=B2, tilt=rng.uniform(0.2, 0.8))
    bm = nnk.BatchedMobility([sw], [EPS[kind]], precision=case["precision"])
    e = np.zeros(bm.n)
    e[bm.n - 12:] = rng.standard_normal(12)   # a functional of the swimming velocities
    return {"kind": kind, "bm": bm, "b": bm.rhs(), "e": e, "tol": case["tol"], "bodies": [sw],
            "eps": np.array([EPS[kind]])}


def _no_flow(t, x):
    return np.zeros_like(x)


def run(state):
    kind = state["kind"]
    if kind in ("uniform", "clustered", "flow_field", "suspension"):
        return state["fmm"].computeVel(state["q"])
    if kind == "mobility":
        return nnk.mobility_gmres(state["sw"], *state["sys"], state["b"], state["tol"], 400, True)
    if kind == "time_step":
        return nnk.mobilityProblem(state["sw"], _no_flow, 0.0, state["y0"], [0.1, 1.0], state["tree"], 20, 0, 1,
                                   1e-4, state["maxit"], [1e-5, 100])
    bm = state["bm"]
    if kind == "batch":
        return bm.solve(state["b"], state["tol"], 300)
    z = bm.solve(state["b"], state["tol"], 400)
    lam = bm.solve(state["e"], state["tol"], 400, transpose=True)
    gx, gy, ge = bm.gradient(z, lam)
    return {"z": z, "lambda": lam, "gx": gx[0], "gy": gy[0], "geps": ge}


# -- what a pass cannot do without ------------------------------------------

def _matvec_work(handle, tree, nsrc):
    """Direct-sum pairs at 33 flop; a translation at the cost of its diagonal
    (frequency) form, nine complex products per unique frequency of the
    (2 res - 1)^3 grid; dense products for M2M, L2L and the solves."""
    st = np.zeros(14, np.int64)
    nnk.lib().nnk_fmm_stats(handle.h, st.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), 14)
    K, R = int(st[12]), int(st[13]) or int(st[12])
    res = round((K / 18.0 - 1.0 / 3.0) ** 0.5 + 1)   # K = 3 (6 (res - 1)^2 + 2)
    flops = PAIR_FLOPS * float(st[1:6].sum()) + 36.0 * (2 * res - 1) ** 3 * float(st[0])
    flops += 2.0 * R * R * float(8 * st[8] + st[9]) + 2.0 * R * K * float(st[6] + st[7])
    npts = len(tree.points)
    return {"bytes": 24.0 * (3 * npts + nsrc), "flops": flops}


def work(case):
    kind = case["kind"]
    s = prepare(case, 0)
    if kind in ("uniform", "clustered", "flow_field", "suspension"):
        tree = s["fmm"].tree
        nsrc = len(tree.points) if tree.finePoints is None else len(tree.finePoints)
        return _matvec_work(s["fmm"]._handle(), tree, nsrc)
    if kind in ("mobility", "time_step"):   # iterations x one matvec
        x = run(s)
        fmm = s["sw"].FMM
        w = _matvec_work(fmm._handle(), fmm.tree, len(fmm.tree.finePoints))
        it = mob.last_solve["iter"]
        return {"bytes": w["bytes"] + x.nbytes, "flops": w["flops"] * it}
    run(s)
    bm = s["bm"]
    pairs = (bm.npts.astype(float) * bm.nfine).ravel()
    passes = float((pairs * bm.last_solve["iter"]).sum()) * (2.0 if kind == "adjoint" else 1.0)
    return {"bytes": 16.0 * bm.n + 24.0 * float(bm.nfine.sum()), "flops": PAIR_FLOPS * passes}


# -- 64-bit values in plain torch --------------------------------------------

def _direct(src, q, tgt, eps):
    """sum_s S(t - s) q_s / (8 pi), regularized Stokeslet of Cortez et al."""
    out = torch.empty_like(tgt)
    step = max(1, int(1.0e8 // len(src)))
    for a in range(0, len(tgt), step):
        t = tgt[a:a + step]
        r = [t[:, d, None] - src[None, :, d] for d in range(3)]
        r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2]
        dot = r[0] * q[:, 0] + r[1] * q[:, 1] + r[2] * q[:, 2]
        inv = (r2 + eps * eps).rsqrt_()
        inv3 = inv * inv * inv
        dot.mul_(inv3)
        iso = inv3.mul_(r2.add_(2.0 * eps * eps))
        out[a:a + step] = iso @ q + torch.stack([(dot * r[d]).sum(1) for d in range(3)], 1)
    return out / (8.0 * np.pi)


def _dense_stokeslet(src, tgt, eps):
    """(3 nt) x (3 ns), rows and columns all x, all y, all z."""
    r = tgt[:, None, :] - src[None, :, :]
    r2 = (r * r).sum(2)
    inv3 = (r2 + eps * eps) ** -1.5
    nt, ns = r2.shape
    S = torch.empty((3, nt, 3, ns), dtype=torch.float64, device=src.device)
    for a in range(3):
        for b in range(3):
            S[a, :, b] = r[:, :, a] * r[:, :, b] * inv3
        S[a, :, a] += (r2 + 2.0 * eps * eps) * inv3
    return S.reshape(3 * nt, 3 * ns) / (8.0 * np.pi)


def _nearest_columns(S, nn, n):
    """S (3 nt x 3 Q) times the nearest map NN (Q x n) per component."""
    Q = S.shape[1] // 3
    idx = torch.from_numpy(np.repeat(np.arange(Q), np.diff(nn.indptr))).cuda()
    col = torch.from_numpy(nn.indices.astype(np.int64)).cuda()
    val = torch.from_numpy(nn.data).cuda()
    out = torch.zeros((S.shape[0], 3, n), dtype=torch.float64, device=S.device)
    T = S.reshape(S.shape[0], 3, Q)
    out.index_add_(2, col, T[:, :, idx] * val)
    return out.reshape(S.shape[0], 3 * n)


def _system_matrix(sw, eps, fine_leaf=None, points_leaf=None):
    """The dense saddle-point matrix [S BT; B 0] of a Swimmers system from
    its definitions; the leaves stand in for the points where gradients are
    wanted."""
    pts, fine, NN = sw.getSwimmerBnd()
    nn = NN.tocsr()
    _, _, _, prot, frot = sw.getSwimmers()
    sizes, _ = sw.getSwimmerSizes()
    n, nsw, nb = len(pts), sw.swimmerNo(), len(prot)
    body = np.repeat(np.arange(nsw), sizes)
    A = torch.zeros((3 * n + 6 * nsw, 3 * n + 6 * nsw), dtype=torch.float64, device="cuda")
    tp, tf = torch.from_numpy(pts).cuda(), torch.from_numpy(fine).cuda()
    step = max(1, int(1.5e8 // (9 * len(fine))))
    for a in range(0, n, step):
        blk = _nearest_columns(_dense_stokeslet(tf, tp[a:a + step], eps), nn, n)
        m = blk.shape[0] // 3
        for d in range(3):
            A[d * n + a:d * n + a + m, :3 * n] = blk[d * m:(d + 1) * m]
    w = np.asarray(nn.sum(axis=0)).ravel()
    ff = np.zeros((len(fine), 3))
    ff[:len(frot)] = frot
    arm = np.asarray(nn.T @ ff)
    C = np.zeros((6 * nsw, 3 * n))   # B: forces, then moments (arm x f)
    D = np.zeros((3 * n, 6 * nsw))   # BT: -(U + Omega x r)
    i = np.arange(nb)
    for d in range(3):
        e, f = (d + 1) % 3, (d + 2) % 3
        C[d * nsw + body, d * n + i] = w[:nb]
        C[3 * nsw + d * nsw + body, f * n + i] = arm[:nb, e]
        C[3 * nsw + d * nsw + body, e * n + i] = -arm[:nb, f]
        D[d * n + i, d * nsw + body] = -1.0
        D[d * n + i, 3 * nsw + e * nsw + body] = -prot[:, f]
        D[d * n + i, 3 * nsw + f * nsw + body] = prot[:, e]
    A[3 * n:, :3 * n] = torch.from_numpy(C).cuda()
    A[:3 * n, 3 * n:] = torch.from_numpy(D).cuda()
    return A


def _pair_gradient(sw, eps, z, lam):
    """-d(lam^T S z)/d(points, quadrature points, eps) by automatic
    differentiation, in target chunks (sources that are body points through
    the nearest map)."""
    pts, fine, NN = sw.getSwimmerBnd()
    n = len(pts)
    f = torch.from_numpy(np.asarray(NN.tocsr() @ z[:3 * n].cpu().numpy().reshape(3, n).T)).cuda()
    l = lam[:3 * n].reshape(3, n).T
    x = torch.from_numpy(pts).cuda().requires_grad_()
    y = torch.from_numpy(fine).cuda().requires_grad_()
    e = torch.tensor(float(eps), dtype=torch.float64, device="cuda", requires_grad=True)
    for a in range(0, n, 256):
        r = x[a:a + 256, None, :] - y[None, :, :]
        r2 = (r * r).sum(2)
        inv3 = (r2 + e * e) ** -1.5
        lf, lr, rf = l[a:a + 256] @ f.T, (l[a:a + 256, None, :] * r).sum(2), (r * f).sum(2)
        (-(((r2 + 2 * e * e) * lf + lr * rf) * inv3).sum() / (8.0 * np.pi)).backward()
    # the bodies' arms move with the nodes too: forces and moments by the
    # quadrature points (B), the rigid velocity by the force points (BT)
    nsw = sw.swimmerNo()
    sizes, fsizes = sw.getSwimmerSizes()
    body = torch.from_numpy(np.repeat(np.arange(nsw), sizes)).cuda()
    fbody = torch.from_numpy(np.repeat(np.arange(nsw), fsizes)).cuda()
    om = z[3 * n + 3 * nsw:].reshape(3, nsw).T[body]
    lm = lam[3 * n + 3 * nsw:].reshape(3, nsw).T[fbody]
    gx = x.grad + torch.linalg.cross(l[:len(body)], om)
    gy = y.grad - torch.linalg.cross(f[:len(fbody)], lm)
    return gx, gy, e.grad.reshape(1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("uniform", "clustered", "flow_field"):
        rng = _generator(seed)
        src, tgt = _points(case, rng)
        if float(len(src)) * len(tgt) > MAX_EXACT_PAIRS:
            return None
        q = torch.from_numpy(_forces(case, rng, len(src))).cuda()
        return _direct(torch.from_numpy(src).cuda(), q, torch.from_numpy(tgt).cuda(), EPS[kind])
    if kind == "suspension":
        sw = _spheroids(case, seed)
        pts, fine, NN = sw.getSwimmerBnd()
        if float(len(pts)) * len(fine) > MAX_EXACT_PAIRS:
            return None
        q = _generator(seed).standard_normal(3 * len(pts))
        f = torch.from_numpy(np.asarray(NN.tocsr() @ q.reshape(3, -1).T)).cuda()
        u = _direct(torch.from_numpy(fine).cuda(), f, torch.from_numpy(pts).cuda(), EPS[kind])
        return u.T.reshape(-1).contiguous()
    if kind == "time_step":
        return None   # a capped iteration: its iterate has no closed value
    if kind == "mobility":
        return None   # first-kind system: the force density is fixed by the iteration's tolerance only
    s = prepare(case, seed)
    if kind == "batch":
        out, at = [], 0
        for sw, eps in zip(s["bodies"], s["eps"]):
            A = _system_matrix(sw, float(eps))
            b = torch.from_numpy(s["b"][at:at + len(A)]).cuda()
            at += len(A)
            out.append(torch.linalg.solve(A, b))
            del A
        return torch.cat(out)
    A = _system_matrix(s["bodies"][0], EPS[kind])
    z = torch.linalg.solve(A, torch.from_numpy(s["b"]).cuda())
    lam = torch.linalg.solve(A.T, torch.from_numpy(s["e"]).cuda())
    gx, gy, ge = _pair_gradient(s["bodies"][0], EPS[kind], z, lam)
    return {"z": z, "lambda": lam, "gx": gx, "gy": gy, "geps": ge}
