"""The work that the speed of this framework is judged by, through its public
entry points (vvflow_amd.Context and the C ABI beneath it).

What users run is the reference's time loop (vvflow_amd/simulate.py,
bench.py): tree, epsilon with merging, convective (plain or learned far
field), diffusive; with a body also the boundary system, shedding, forces and
flow-move; many small simulations in one context; probes and velocity maps
after the run; and the training of the learned far field.

  wake        one step over a Karman-street wake without a body: restore the
              list, tree, epsilon, convective, diffusive, list back on the host
  cylinder    a restart of a cylinder run (bodies uploaded, list restored) and
              two whole steps of the loop, list and bodies back; optionally
              with heat and streak lists, or with many simulations in a batch
  probes      velocity at probe points and velocity maps over a finished wake
  train       Adam steps of the far-field network on pairs held on the device
"""
import math
import os

import numpy as np
import torch

import vvflow_amd as V

INF = (1.0, 0.0)
RE = 600.0
DT = 0.005
MODEL = os.path.join(os.path.dirname(os.path.abspath(V.__file__)), "farfield_mlp.npy")
DBL_MAX = float(np.finfo(np.float64).max)


def listed():
    return [
        # an early wake, a few launches deep: the first hundreds of steps of every run are of this size
        dict(name="wake_2k", kind="wake", n=2003, far=8, learned=False, kahan=True),
        # an ordinary small wake at a high far criterion, as accuracy checks use it (near field heavy)
        dict(name="wake_20k_far64", kind="wake", n=20011, far=64, learned=False, kahan=True),
        # an ordinary wake with plain FP32 sums, the fast option of the near field
        dict(name="wake_200k_fp32", kind="wake", n=200003, far=8, learned=False, kahan=False),
        # an ordinary wake on the learned path
        dict(name="wake_100k_learned", kind="wake", n=100003, far=8, learned=True, kahan=True),
        # the benchmark's workload: 1M vortices, learned far field
        dict(name="wake_1m_learned", kind="wake", n=1000000, far=8, learned=True, kahan=True),
        # the largest: the 4M wake of the precision sweep, plain path, compensated sums
        dict(name="wake_4m", kind="wake", n=4000000, far=8, learned=False, kahan=True),
        # the README's example run: a 350-segment cylinder early in its wake
        dict(name="cylinder_3k", kind="cylinder", n=3001, nseg=350, sims=1, learned=False, heat=0, streak=0),
        # a developed cylinder wake, the size the batched benchmark's median simulation has
        dict(name="cylinder_100k", kind="cylinder", n=100003, nseg=500, sims=1, learned=False, heat=0, streak=0),
        # a heated cylinder with dye lines
        dict(name="cylinder_heat_5k", kind="cylinder", n=5003, nseg=500, sims=1, learned=False, heat=4001, streak=1500),
        # independent cylinders advanced together (a Reynolds sweep)
        dict(name="cylinder_batch_16", kind="cylinder", n=1000000, nseg=500, sims=16, learned=False, heat=0, streak=0),
        # post-processing: probes and velocity maps over a finished wake
        dict(name="probes_200k", kind="probes", n=200003, far=8, points=20011, grid=200),
        # retraining the far-field network: Adam steps at the training batch
        dict(name="train_8192", kind="train", pairs=262144, batch=8192, steps=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.5:
        learned = rng.random() < 0.4
        far = 8 if learned else rng.choice([8, 8, 10, 16, 64])
        top = (2000000 if learned else 3900000) / (far / 8.0) ** 0.9
        return dict(kind="wake", n=_log(rng, 1500, top) | 1, far=far, learned=learned, kahan=rng.random() < 0.7)
    if u < 0.78:
        heat = _log(rng, 300, 3500) if rng.random() < 0.3 else 0
        streak = _log(rng, 100, 5000) if heat or rng.random() < 0.2 else 0
        top = 8000 if heat or streak else 250000
        return dict(kind="cylinder", n=_log(rng, 2000, top) | 1, nseg=rng.randrange(120, 501), sims=1,
                    learned=rng.random() < 0.25, heat=heat, streak=streak)
    if u < 0.86:
        return dict(kind="cylinder", n=_log(rng, 60000, 1000000) | 1, nseg=rng.randrange(200, 501),
                    sims=rng.randrange(3, 17), learned=False, heat=0, streak=0)
    if u < 0.94:
        return dict(kind="probes", n=_log(rng, 3000, 400000) | 1, far=rng.choice([8, 8, 16]),
                    points=_log(rng, 50, 40000), grid=rng.randrange(40, 321))
    return dict(kind="train", pairs=_log(rng, 20000, 400000), batch=32 * rng.randrange(32, 513), steps=rng.randrange(4, 25))


# ------------------------------------------------------------------ inputs --

def _wake(n, seed):
    """Karman street: 400 Gaussian clusters (sigma 0.05) in two staggered rows
    at y = +-0.2, cluster by cluster, as vvhd_gen_wake lays it out."""
    r = np.random.default_rng(seed)
    k = np.minimum(np.arange(n) * 400 // max(n, 1), 399)
    top = k < 200
    o = np.zeros((n, 6))
    o[:, 0] = 0.3 * (k % 200) + np.where(top, 0.0, 0.15) + 0.05 * r.standard_normal(n)
    o[:, 1] = np.where(top, 0.2, -0.2) + 0.05 * r.standard_normal(n)
    o[:, 2] = np.where(top, -1.0, 1.0) * r.uniform(0.5, 1.5, n) * 1e-3
    return o


def _cylinder_wake(n, seed):
    """A cylinder run's list near the balance that merging keeps: jittered
    lattices of spacing 0.006 sqrt(1 + distance), rings round the body (R =
    0.5) and columns behind it; few merges per step."""
    r = np.random.default_rng(seed)
    c, jit = 0.006, 0.2
    pts, nb, rad, cnt = [], int(0.1 * n), 0.502, 0
    while cnt < nb:
        h = c * math.sqrt(1.0 + (rad - 0.5))
        m = int(2 * math.pi * rad / h)
        th = (np.arange(m) + r.uniform(-jit, jit, m)) * (2 * math.pi / m)
        rr = rad + r.uniform(-jit, jit, m) * h
        pts.append(np.stack([rr * np.cos(th), rr * np.sin(th)], 1))
        cnt += m
        rad += h
    layer = np.concatenate(pts)[:nb] if pts else np.zeros((0, 2))
    w = max(1.0, n / 1e5)
    pts, x, cnt = [], max(1.0, rad + 0.1), 0
    while cnt < n - nb:
        h = c * math.sqrt(1.0 + x)
        m = int(2 * w / h)
        y = -w + (np.arange(m) + 0.5 + r.uniform(-jit, jit, m)) * (2 * w / m)
        pts.append(np.stack([x + r.uniform(-jit, jit, m) * h, y], 1))
        cnt += m
        x += h
    o = np.zeros((n, 6))
    o[:, :2] = np.concatenate([layer, np.concatenate(pts)[:n - nb]])
    o[:, 2] = np.where(o[:, 1] > 0, -1.0, 1.0) * r.uniform(0.5, 1.5, n) * 1e-3
    return o


def _heat(n, seed):
    """Warm fluid carried off the body into the near wake."""
    r = np.random.default_rng(seed)
    o = np.zeros((n, 6))
    far = r.random(n) < 0.7
    th, rad = r.uniform(0, 2 * math.pi, n), 0.51 + 0.2 * r.random(n) ** 2
    o[:, 0] = np.where(far, r.uniform(0.8, 4.0, n), rad * np.cos(th))
    o[:, 1] = np.where(far, r.uniform(-0.7, 0.7, n), rad * np.sin(th))
    o[:, 2] = r.uniform(0.5, 1.5, n) * 1e-4
    return o


def _streak(n, seed):
    """Dye lines from sources on x = -1, carried past the body."""
    r = np.random.default_rng(seed)
    o = np.zeros((n, 6))
    o[:, 0] = r.uniform(-1.0, 4.0, n)
    o[:, 1] = np.round(r.uniform(-8, 8, n)) / 8.0 + 0.01 * r.standard_normal(n)
    inside = o[:, 0] ** 2 + o[:, 1] ** 2 < 0.3
    o[inside, 1] += 1.2
    return o


def _train_data(case, seed):
    """Pairs as far_sample gives them: raw features, smooth labels, S^2 weights."""
    r = np.random.default_rng(seed)
    n = case["pairs"]
    mu = r.uniform(-0.3, 0.5, 12).astype(np.float32)
    sd = r.uniform(0.05, 0.6, 12).astype(np.float32)
    Z = r.standard_normal((n, 12)).astype(np.float32)
    A = r.standard_normal((12, 2)).astype(np.float32) * 0.4
    Y = (np.tanh(Z @ A) + 0.2 * (Z[:, 6:8] + Z[:, 2:4] * Z[:, 4:6])).astype(np.float32)
    W = np.exp(r.standard_normal(n)).astype(np.float32)
    W /= W.mean()
    P = np.concatenate([
        r.standard_normal(64 * 12) / math.sqrt(12), 0.1 * r.standard_normal(64),
        r.standard_normal(64 * 64) / 8, 0.1 * r.standard_normal(64), r.standard_normal(128) / 8, np.zeros(2),
        mu, sd, np.full(2, 0.9)]).astype(np.float32)
    lr = np.linspace(2e-3, 1e-3, case["steps"]).astype(np.float32)
    return P, np.ascontiguousarray(Z * sd + mu), Y, W, lr


def _sizes(case):
    """Vortices of each simulation of a batch, spread over a factor of ten."""
    k = case["sims"]
    w = 10.0 ** (np.arange(k) / max(k - 1, 1))
    n = np.maximum(2000, (w / w.sum() * case["n"]).astype(np.int64))
    return n


def _points(case, seed):
    r = np.random.default_rng(seed + 77)
    return np.stack([r.uniform(-2.0, 62.0, case["points"]), r.uniform(-1.0, 1.0, case["points"])], 1)


def _grid(case):
    """A map of grid x grid/2 nodes over part of the street."""
    w = case["grid"]
    return dict(xmin=10.0, ymin=-1.0, dxdy=4.0 / w, xres=w, yres=max(1, w // 2))


# ------------------------------------------------------------------ states --

def prepare(case, seed):
    kind = case["kind"]
    c = V.Context(0)
    s = dict(case=case, ctx=c, kind=kind)
    if kind == "train":
        P, X, Y, W, lr = _train_data(case, seed)
        c.far_train_data(X, Y, W)
        s.update(P=P, lr=lr)
        return s
    if kind in ("wake", "probes"):
        o = _wake(case["n"], seed)
        c.set_params(re=RE, dt=DT)
        c.upload(o)
        if kind == "wake":
            if case["learned"]:
                c.far_model_set(np.load(MODEL, allow_pickle=False))
            c.snapshot()
            s["out"] = torch.empty((case["n"], 6), dtype=torch.float64, pin_memory=True)
        else:   # a finished run: its list with a tree and epsilons, ready to be asked
            c.tree_build(case["far"], 0.0, 0.1)
            c.epsilon(False)
            s.update(pts=_points(case, seed), grid=_grid(case))
        return s
    # cylinder runs
    k, nseg = case["sims"], case["nseg"]
    ns = _sizes(case) if k > 1 else np.array([case["n"]])
    one = np.ascontiguousarray(V.segments_from_corners(V.gen_cylinder(0.5, nseg)), dtype=V.SEG_DTYPE)
    segs = np.concatenate([one] * k)
    bodies = np.zeros(k, dtype=V.BODY_DTYPE)
    bodies["nseg"] = nseg
    bodies["first_seg"] = np.arange(k) * nseg
    o = np.concatenate([_cylinder_wake(int(m), seed * 31 + q) for q, m in enumerate(ns)])
    c.set_params(re=RE, dt=DT)
    c.upload_bodies(segs, bodies)
    dl = c.download_bodies()[1][0]["slen"] / (nseg - 1)
    c.upload(o)
    c.snapshot()
    if case["learned"]:
        c.far_model_set(np.load(MODEL, allow_pickle=False))
    s.update(segs=segs, bodies=bodies, tree=(8, 5 * dl, 100 * dl),
             off=np.concatenate([[0], np.cumsum(ns)]).astype(np.int64), boff=np.arange(k + 1, dtype=np.int32),
             re=np.geomspace(100.0, 3000.0, k) if k > 1 else np.array([RE]),
             out=torch.empty((int(ns.sum()) + 4 * len(segs) + 16, 6), dtype=torch.float64, pin_memory=True))
    if case["heat"]:
        s["heat"] = _heat(case["heat"], seed * 31 + 17)
    if case["streak"]:
        s["streak"] = _streak(case["streak"], seed * 31 + 23)
        src = np.zeros((17, 6))
        src[:, 0], src[:, 1] = -1.0, np.linspace(-1.0, 1.0, 17)
        s["sources"] = src
    return s


def _read(ctx, out):
    """The vortex list into the caller's pinned records (zeros behind it)."""
    n = ctx.n
    ctx._check(ctx.L.vvhd_download_vortices(ctx.h, out.data_ptr(), n))
    out[n:].zero_()
    return out


def _padded(a, rows):
    out = np.zeros((rows, 6))
    out[:len(a)] = a
    return out


def run(s):
    c, case, kind = s["ctx"], s["case"], s["kind"]
    if kind == "wake":
        c.restore()
        c.tree_build(case["far"])
        c.epsilon(True)
        if case["learned"]:
            c.convective_learned(INF, kahan=case["kahan"])
        else:
            c.convective(INF, kahan=case["kahan"])
        c.diffusive()
        o = _read(c, s["out"])
        return dict(xyg=o[:, 0:3], v=o[:, 3:5], ie=o[:, 5])
    if kind == "probes":
        g = s["grid"]
        return dict(points=c.velocity(s["pts"], INF), vx=c.field(V.FIELD_VX, inf=INF, **g),
                    vy=c.field(V.FIELD_VY, inf=INF, **g))
    if kind == "train":
        c.far_model_set(s["P"])
        loss = c.far_train(s["lr"], batch=case["batch"], seed=11)
        return dict(loss=loss, params=c.far_model_get())
    # a restart and two steps of the time loop (simulate.CylinderRun.step)
    t0 = 2.0
    c.set_params(re=RE, dt=DT, time=t0)
    c.upload_bodies(s["segs"], s["bodies"])
    if "heat" in s:
        c.set_heat([V.HC_CONST_T], np.full(len(s["segs"]), 1.0, np.float32))
        c.set_pr(0.7)
    if "heat" in s or "streak" in s:
        c.upload_list(V.LIST_HEAT, s.get("heat", np.zeros((0, 6))))
        c.upload_list(V.LIST_STREAK, s.get("streak", np.zeros((0, 6))))
        c.upload_list(V.LIST_STREAK_SOURCE, s.get("sources", np.zeros((0, 6))))
    c.restore()
    if case["sims"] > 1:
        c.set_batch(s["off"], s["boff"], s["re"])
    forces = []
    for k in range(2):
        c.set_params(re=RE, dt=DT, time=t0 + k * DT)
        c.tree_build(*s["tree"])
        c.calc_circulation(INF)
        c.tree_destroy()
        if "heat" in s:
            c.heat_shed()
        c.vortex_shed()
        if "streak" in s and k == 0:
            c.streak_shed()
        c.calc_forces()
        b = c.download_bodies()[1]
        forces.append(np.concatenate([b["force_hydro"], b["friction"]], 1))
        c.zero_forces()
        c.tree_build(*s["tree"])
        c.epsilon(True)
        if case["learned"]:
            c.convective_learned(INF)
        else:
            c.convective(INF)
        c.diffusive()
        if "heat" in s:
            c.diffusive_heat()
        c.tree_destroy()
        c.move_and_clean(True)
        if "heat" in s:
            c.heat_crop(16.0)
    out = dict(vort=_read(c, s["out"]), forces=np.stack(forces), count=c.n)
    segs = c.download_bodies()[0]
    out["segs"] = np.ascontiguousarray(segs).view(np.float64).reshape(len(segs), -1)[:, :11]
    if "heat" in s:
        out["heat"] = _padded(c.download_list(V.LIST_HEAT), case["heat"] + 3 * case["nseg"])
    if "streak" in s:
        out["streak"] = _padded(c.download_list(V.LIST_STREAK), case["streak"] + 64)
    return out


# -------------------------------------------------------- work, tolerances --

def _near(n, far):
    """Near sources per vortex of these wakes (2636 at 1M and criterion 8, 15k
    at 4M and 64), at most the list."""
    return min(0.7 * n, 2600.0 * (far / 8.0) ** 0.7 * max(0.2, (n / 1e6) ** 0.2))


def work(case):
    kind = case["kind"]
    if kind == "train":
        fl = 2.0 * (12 * 64 + 64 * 64 + 64 * 2) * 3
        rows = case["batch"] * case["steps"]
        return {"bytes": 60.0 * rows + 5148 * 4 * 6.0 * case["steps"], "flops": fl * rows}
    n = case["n"]
    if kind == "probes":
        q = case["points"] + 2 * case["grid"] * max(1, case["grid"] // 2)
        return {"bytes": 48.0 * n + 32.0 * q, "flops": q * (11.0 * _near(n, case["far"]) + 24 * 340)}
    far = case.get("far", 8)
    # near pairs: convective 11 flops, epsilon 5 over the touching leaves, diffusive 16 over the cutoff
    fl = n * (11.0 * _near(n, far) + 5 * 100 + 16 * 300 + 40 * 34.2 * min(1.0, math.log2(n) / 20))
    if case.get("learned"):
        fl += n * 34.2 * min(1.0, (n / 1e6) ** 0.1) * 3 * 9984.0
    by = 48.0 * 2 * n
    if kind == "wake":
        return {"bytes": by, "flops": fl}
    m = case["nseg"] + 9
    # two steps; the boundary system's cells, and a solve with kept factors
    solve = case["sims"] * (m * m * 8.0 * 2)
    return {"bytes": 2 * (by + solve), "flops": 2 * (fl + case["sims"] * (m * m * 30.0 + 2.0 * m * m))}


def tolerance(case):
    kind = case["kind"]
    if kind == "wake":
        if case["learned"]:
            return {"rel": 4e-6}    # the network's gradient left out moves it by as much
        # FP32 pair sums: 1.2e-8 to 5e-8 from 64 bits compensated, 2e-7 plain;
        # the diffusive sums 3.5e-7 of their own size
        return {"rel": 5e-7} if case["kahan"] else {"rel": 2e-6}
    if kind == "probes":
        return {"rel": 2e-7}    # FP64 sums, float maps
    if kind == "train":
        return {"rel": 4e-3}    # bf16 network, Adam steps (9e-4 from 64 bits)
    return {"rel": 1e-7}        # two steps: FP32 sums in another form move the list by 2e-8


# ------------------------------------------------- the same in 64 bits --

def _tree(x, y, g, min_node, max_node):
    """Adaptive binary tree by levels; the vortices in its order (perm) and
    the nodes as arrays.  A node splits at the centre of its bounding box
    across the longer side; the k-th element left of the split that belongs
    right trades places with the k-th from the end that belongs left."""
    dev, n = x.device, x.numel()
    perm = torch.arange(n, device=dev)
    v0, v1 = torch.zeros(1, dtype=torch.long, device=dev), torch.full((1,), n, dtype=torch.long, device=dev)
    node = torch.zeros(n, dtype=torch.long, device=dev)     # node of every position, within the level
    open_ = torch.ones(n, dtype=torch.bool, device=dev)     # position in a node of this level
    levels = []
    while v0.numel():
        m = v0.numel()
        px, py = x[perm], y[perm]
        nd, p = node[open_], torch.nonzero(open_).flatten()
        box = []
        for a in (px, py):
            for how, start in (("amin", DBL_MAX), ("amax", -DBL_MAX)):
                box.append(torch.full((m,), start, dtype=torch.float64, device=dev).scatter_reduce(0, nd, a[p], how))
        cx, cy, h, w = (box[0] + box[1]) * 0.5, (box[2] + box[3]) * 0.5, box[3] - box[2], box[1] - box[0]
        mx, mn = torch.maximum(h, w), torch.minimum(h, w)
        leaf = (mx < max_node) & ((mn <= min_node) | (v1 - v0 < 16))
        left = torch.zeros(n, dtype=torch.bool, device=dev)
        byx = (h < w)[nd]
        left[p] = torch.where(byx, px[p] < cx[nd], py[p] < cy[nd]) & ~leaf[nd]
        c = torch.cat([torch.zeros(1, dtype=torch.long, device=dev), left.long().cumsum(0)])
        L = v0 + c[v1] - c[v0]
        go = ~leaf[nd]
        q, qn = p[go], nd[go]
        mis_r = (q < L[qn]) & ~left[q]                      # in the left part, belongs right
        mis_l = (q >= L[qn]) & left[q]
        a, an = q[mis_r], qn[mis_r]
        b, bn = q[mis_l], qn[mis_l]
        # per node: the k-th of a with the k-th of b counted from the end
        order = torch.argsort(bn * (n + 1) + (n - b))
        b = b[order]
        pa, pb = perm[a].clone(), perm[b].clone()
        perm[a], perm[b] = pb, pa
        kid = torch.full((m,), -1, dtype=torch.long, device=dev)
        sp = torch.nonzero(~leaf).flatten()
        kid[sp] = 2 * torch.arange(sp.numel(), device=dev)
        levels.append(dict(x=cx, y=cy, h=h, w=w, v0=v0, v1=v1, kid=kid))
        node = torch.where(open_, node, torch.zeros_like(node))
        nxt = torch.zeros_like(node)
        keep = torch.zeros_like(open_)
        nxt[q] = kid[qn] + (q >= L[qn]).long()
        keep[q] = True
        node, open_ = nxt, keep
        v0, v1 = torch.stack([v0[sp], L[sp]], 1).flatten(), torch.stack([L[sp], v1[sp]], 1).flatten()
    # one table, level after level
    base, T = 0, {k: [] for k in ("x", "y", "h", "w", "v0", "v1", "kid")}
    for d in levels:
        m = d["x"].numel()
        d["kid"] = torch.where(d["kid"] >= 0, d["kid"] + base + m, d["kid"])
        d["base"], base = base, base + m
        for k in T:
            T[k].append(d[k])
    T = {k: torch.cat(v) for k, v in T.items()}
    T["levels"] = [(d["base"], d["x"].numel()) for d in levels]
    # per-sign circulation and its centre, from the vortices up
    gs, xs, ys = g[perm], x[perm], y[perm]
    for sgn, part in (("p", gs > 0), ("m", ~(gs > 0))):
        gg = torch.where(part, gs, torch.zeros_like(gs))
        G, X, Y = (torch.zeros_like(T["x"]) for _ in range(3))
        leaf = torch.nonzero(T["kid"] < 0).flatten()
        own = torch.repeat_interleave(leaf, T["v1"][leaf] - T["v0"][leaf])
        pos = _ranges(T["v0"][leaf], T["v1"][leaf] - T["v0"][leaf])
        G.index_add_(0, own, gg[pos])
        X.index_add_(0, own, gg[pos] * xs[pos])
        Y.index_add_(0, own, gg[pos] * ys[pos])
        for b, m in reversed(T["levels"]):
            k = T["kid"][b:b + m]
            q = torch.nonzero(k >= 0).flatten()
            for A in (G, X, Y):
                A[b + q] = A[k[q]] + A[k[q] + 1]
        nz = G != 0
        T["g" + sgn], T["x" + sgn], T["y" + sgn] = G, torch.where(nz, X / G, T["x"]), torch.where(nz, Y / G, T["y"])
    leaf = torch.nonzero(T["kid"] < 0).flatten()
    T["leaf"] = leaf[torch.argsort(T["v0"][leaf] * (base + 1) + leaf)]
    return perm, T


def _ranges(start, count):
    """start[0], start[0]+1, ... for every (start, count), one after another."""
    end = count.cumsum(0)
    total = int(end[-1]) if count.numel() else 0
    r = torch.arange(total, device=start.device)
    return r - torch.repeat_interleave(end - count - start, count)


def _lists(T, far):
    """(leaf slot, node) of all near leaves and of all far nodes."""
    lf = T["leaf"]
    a = torch.arange(lf.numel(), device=lf.device)
    nd = torch.zeros_like(a)
    near, fars = [], []
    while a.numel():
        L = lf[a]
        dx, dy = T["x"][nd] - T["x"][L], T["y"][nd] - T["y"][L]
        hp = (T["h"][nd] + T["w"][nd]) + T["h"][L] + T["w"][L]
        isfar = dx * dx + dy * dy > float(far) * hp * hp
        isleaf = ~isfar & (T["kid"][nd] < 0)
        fars.append((a[isfar], nd[isfar]))
        near.append((a[isleaf], nd[isleaf]))
        rest = ~isfar & ~isleaf
        a, k = a[rest], T["kid"][nd[rest]]
        a, nd = torch.cat([a, a]), torch.cat([k, k + 1])
    near = [torch.cat(v) for v in zip(*near)]
    fars = [torch.cat(v) for v in zip(*fars)]
    o = torch.argsort(near[0], stable=True)
    return (near[0][o], near[1][o]), fars


def _pairs(T, near, slots, budget=40_000_000):
    """Chunks of (target position, source position) over the near lists of the leaf slots."""
    lf = T["leaf"]
    cnt = T["v1"] - T["v0"]
    nl = lf.numel()
    off = torch.searchsorted(near[0], torch.arange(nl + 1, device=lf.device))
    per = torch.zeros(nl, dtype=torch.long, device=lf.device).index_add_(0, near[0], cnt[near[1]])
    cost = (per * cnt[lf])[slots].cumsum(0)
    i = 0
    while i < slots.numel():
        base = int(cost[i - 1]) if i else 0
        j = max(i + 1, int(torch.searchsorted(cost, torch.tensor(base + budget, device=lf.device))))
        s = slots[i:j]
        e = _ranges(off[s], off[s + 1] - off[s])
        es, em = near[0][e], near[1][e]
        src = _ranges(T["v0"][em], cnt[em])                     # sources of the entries
        ss = torch.repeat_interleave(es, cnt[em])
        k = cnt[lf[ss]]
        tgt = _ranges(T["v0"][lf[ss]], k)
        yield tgt, torch.repeat_interleave(src, k)
        i = j


def _top2(T, near, slots, x, y, g, n):
    """Squared distances and positions of the two nearest vortices of every target of the slots."""
    dev = x.device
    d1 = torch.full((n,), math.inf, dtype=torch.float64, device=dev)
    d2, i1, i2 = d1.clone(), torch.full((n,), n, dtype=torch.long, device=dev), torch.full((n,), n, dtype=torch.long, device=dev)
    for t, s in _pairs(T, near, slots):
        ok = (g[s] != 0) & (g[t] != 0) & (s != t)
        t, s = t[ok], s[ok]
        dx, dy = x[t] - x[s], y[t] - y[s]
        d = dx * dx + dy * dy
        for D, I in ((d1, i1), (d2, i2)):
            D.scatter_reduce_(0, t, d, "amin")
            hit = d == D[t]
            I.scatter_reduce_(0, t[hit], s[hit], "amin")
            ok = s != I[t]
            t, s, d = t[ok], s[ok], d[ok]
    return d1, d2, i1, i2


def _epsilon(T, near, x, y, g, merge):
    """1/eps of every vortex with circulation, merging in list order."""
    n, dev = x.numel(), x.device
    slots = torch.arange(T["leaf"].numel(), device=dev)
    cnt = (T["v1"] - T["v0"])[T["leaf"]]
    slot_of = torch.repeat_interleave(slots, cnt)
    slot_node = torch.full((T["x"].numel(),), -1, dtype=torch.long, device=dev)
    slot_node[T["leaf"]] = slots
    st = _top2(T, near, slots, x, y, g, n)
    alive = torch.ones(n, dtype=torch.bool, device=dev)          # may still merge
    searched = g != 0                                            # a partner not yet reached is passed over

    def flags():
        ok = (g != 0) & alive & (st[3] < n)
        s1, s2 = torch.sign(g[st[2].clamp(max=n - 1)]), torch.sign(g[st[3].clamp(max=n - 1)])
        return ok & (s1 == s2) & (s1 != torch.sign(g))

    if merge:
        f = flags()
        cur = 0
        while True:
            q = torch.nonzero(f[cur:]).flatten()
            if not q.numel():
                break
            q = cur + int(q[0])
            p = int(st[2][q])
            gq, gp = float(g[q]), float(g[p])
            if (gq > 0) == (gp > 0):
                x[q], y[q] = (x[q] * gq + x[p] * gp) / (gq + gp), (y[q] * gq + y[p] * gp) / (gq + gp)
            elif abs(gq) < abs(gp):
                x[q], y[q] = x[p], y[p]
            g[q], g[p] = gq + gp, 0.0
            if p > q:
                searched[p] = False
            hit = torch.isin(slot_node[near[1]], slot_of[torch.tensor([q, p], device=dev)])
            again = torch.unique(near[0][hit])
            new = _top2(T, near, again, x, y, g, n)
            later = torch.isin(slot_of, again) & (torch.arange(n, device=dev) >= q)
            for old, nw in zip(st, new):
                old[later] = nw[later]
            alive[q] = False
            f = flags()
            cur = q + 1
    ie = torch.zeros(n, dtype=torch.float64, device=dev)
    e = torch.where(st[3] < n, st[1].sqrt(), torch.where(st[2] < n, st[0].sqrt(), torch.full_like(ie, 2.2250738585072014e-308)))
    return torch.where(searched, 1.0 / e, ie)


def _exact_wake(case, seed):
    n = case["n"]
    if n > (200000 if case["learned"] else 1200000) or n * _near(n, case["far"]) > 6e9:
        return None   # over 20 seconds
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    o = torch.from_numpy(_wake(n, seed)).to(dev)
    perm, T = _tree(o[:, 0].contiguous(), o[:, 1].contiguous(), o[:, 2].contiguous(), 0.0, DBL_MAX)
    x, y, g = (o[perm, k].contiguous() for k in range(3))
    near, far = _lists(T, case["far"])
    ie = _epsilon(T, near, x, y, g, True)
    e2 = torch.where(g != 0, 1.0 / (ie * ie), torch.ones_like(ie))
    u = torch.zeros((n, 2), dtype=torch.float64, device=dev)
    S2, S1 = torch.zeros_like(u), torch.zeros_like(x)
    for t, s in _pairs(T, near, torch.arange(T["leaf"].numel(), device=dev)):
        dx, dy = x[t] - x[s], y[t] - y[s]
        r2 = dx * dx + dy * dy
        if not case["learned"]:
            f = g[s] / (r2 + e2[s])
            u[:, 0].index_add_(0, t, -dy * f)
            u[:, 1].index_add_(0, t, dx * f)
        r = r2.sqrt()
        ea = -r * ie[t]
        ok = (g[t] * g[s] > 0) & (dx.abs() + dy.abs() >= 1e-10) & (ea >= -8.0)
        t, s, dx, dy, r = t[ok], s[ok], dx[ok], dy[ok], r[ok]
        i1 = g[s] * torch.exp(ea[ok])
        S1.index_add_(0, t, i1)
        S2[:, 0].index_add_(0, t, dx / r * i1)
        S2[:, 1].index_add_(0, t, dy / r * i1)
    if case["learned"]:   # the far field the network stands for: the sum over all vortices
        rows = max(1, 20_000_000 // n)
        for b in range(0, n, rows):
            dx, dy = x[b:b + rows, None] - x, y[b:b + rows, None] - y
            f = g / (dx * dx + dy * dy + e2)
            u[b:b + rows, 0] = -(dy * f).sum(1)
            u[b:b + rows, 1] = (dx * f).sum(1)
    u /= 2 * math.pi
    lf = T["leaf"]
    if not case["learned"]:   # first-order expansion of the far circulation about the leaf's centre
        a = torch.zeros((lf.numel(), 4), dtype=torch.float64, device=dev)
        for sg in "pm":
            dx, dy = T["x"][lf[far[0]]] - T["x" + sg][far[1]], T["y"][lf[far[0]]] - T["y" + sg][far[1]]
            G, r2 = T["g" + sg][far[1]], dx * dx + dy * dy
            for k, q in enumerate((-dy / r2, dx / r2, 2 * dx * dy / r2 ** 2, (dy * dy - dx * dx) / r2 ** 2)):
                a[:, k].index_add_(0, far[0], torch.where(G != 0, G * q, torch.zeros_like(q)))
        a /= 2 * math.pi
        slot = torch.repeat_interleave(torch.arange(lf.numel(), device=dev), (T["v1"] - T["v0"])[lf])
        ox, oy = x - T["x"][lf[slot]], y - T["y"][lf[slot]]
        A = a[slot]
        u[:, 0] += A[:, 0] + A[:, 2] * ox + A[:, 3] * oy
        u[:, 1] += A[:, 1] + A[:, 3] * ox - A[:, 2] * oy
    low = (torch.sign(S1) != torch.sign(g)) | (S1.abs() < 0.1 * g.abs())
    S1 = torch.where(low, 0.1 * g, S1)
    v = u + torch.tensor(INF, dtype=torch.float64, device=dev) + S2 * (ie / (RE * S1))[:, None]
    v = torch.where((g != 0)[:, None], v, torch.zeros_like(v))
    return dict(xyg=torch.stack([x, y, g], 1).cpu(), v=v.cpu(), ie=ie.cpu())


def _exact_probes(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    o = torch.from_numpy(_wake(case["n"], seed)).to(dev)
    perm, T = _tree(o[:, 0].contiguous(), o[:, 1].contiguous(), o[:, 2].contiguous(), 0.0, 0.1)
    x, y, g = (o[perm, k].contiguous() for k in range(3))
    near, far = _lists(T, case["far"])
    ie = _epsilon(T, near, x, y, g, False)
    e2 = torch.where(g != 0, 1.0 / (ie * ie), torch.ones_like(ie))
    lf = T["leaf"]
    slot = torch.full((T["x"].numel(),), -1, dtype=torch.long, device=dev)
    slot[lf] = torch.arange(lf.numel(), device=dev)
    noff = torch.searchsorted(near[0], torch.arange(lf.numel() + 1, device=dev))
    fo = torch.argsort(far[0], stable=True)
    far = (far[0][fo], far[1][fo])
    foff = torch.searchsorted(far[0], torch.arange(lf.numel() + 1, device=dev))

    def velocity(p):
        nd = torch.zeros(p.shape[0], dtype=torch.long, device=dev)
        while True:
            k = T["kid"][nd]
            if not bool((k >= 0).any()):
                break
            left = torch.where(T["h"][nd] < T["w"][nd], p[:, 0] < T["x"][nd], p[:, 1] < T["y"][nd])
            nd = torch.where(k >= 0, k + (~left).long(), nd)
        u = torch.zeros_like(p)
        for b in range(0, p.shape[0], 4000):
            l = slot[nd[b:b + 4000]]
            i = torch.arange(l.numel(), device=dev)
            e = _ranges(noff[l], noff[l + 1] - noff[l])
            ei = torch.repeat_interleave(i, noff[l + 1] - noff[l])
            c = (T["v1"] - T["v0"])[near[1][e]]
            s, t = _ranges(T["v0"][near[1][e]], c), b + torch.repeat_interleave(ei, c)
            todo = [(t, x[s], y[s], g[s], e2[s])]
            e = _ranges(foff[l], foff[l + 1] - foff[l])
            t = b + torch.repeat_interleave(i, foff[l + 1] - foff[l])
            F = far[1][e]
            todo += [(t, T["x" + k][F], T["y" + k][F], T["g" + k][F], torch.zeros_like(T["x"][F])) for k in "pm"]
            for t, sx, sy, sg, s2 in todo:
                dx, dy = p[t, 0] - sx, p[t, 1] - sy
                f = torch.where(sg != 0, sg / (dx * dx + dy * dy + s2), torch.zeros_like(sg))
                u[:, 0].index_add_(0, t, -dy * f)
                u[:, 1].index_add_(0, t, dx * f)
        return u / (2 * math.pi) + torch.tensor(INF, dtype=torch.float64, device=dev)

    gr = _grid(case)
    gx = gr["xmin"] + gr["dxdy"] * torch.arange(gr["xres"], dtype=torch.float64, device=dev)
    gy = gr["ymin"] + gr["dxdy"] * torch.arange(gr["yres"], dtype=torch.float64, device=dev)
    p = torch.stack([gx.repeat(gr["yres"]), gy.repeat_interleave(gr["xres"])], 1)
    m = velocity(p).reshape(gr["yres"], gr["xres"], 2).cpu()
    return dict(points=velocity(torch.from_numpy(_points(case, seed)).to(dev)).cpu(), vx=m[..., 0], vy=m[..., 1])


def _mix64(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _exact_train(case, seed):
    P, X, Y, W, lr = (torch.from_numpy(a).double() for a in _train_data(case, seed))
    cut = np.cumsum([0, 768, 64, 4096, 64, 128, 2, 12, 12, 2])
    part = lambda p: [p[cut[k]:cut[k + 1]] for k in range(9)]  # noqa: E731
    mu, sd, ysd = part(P)[6:]
    p = P[:cut[6]].clone()
    m, v, loss = torch.zeros_like(p), torch.zeros_like(p), []
    slot = np.arange(case["batch"], dtype=np.uint64)
    for k in range(case["steps"]):
        with np.errstate(over="ignore"):
            sk = np.uint64(11) + np.uint64(k) * np.uint64(0x9E3779B97F4A7C15)
            j = _mix64(sk ^ (slot * np.uint64(0xD1B54A32D192ED03))) % np.uint64(case["pairs"])
        j = torch.from_numpy(j.astype(np.int64))
        q = p.clone().requires_grad_(True)
        w1, b1, w2, b2, w3, b3 = part(q)[:6]
        h = torch.nn.functional.silu(((X[j] - mu) / sd) @ w1.reshape(64, 12).T + b1)
        h = torch.nn.functional.silu(h @ w2.reshape(64, 64).T + b2)
        r = h @ w3.reshape(2, 64).T + b3 - Y[j] / ysd
        ls = (W[j] * (r * r).sum(1)).sum() / case["batch"]
        (d,) = torch.autograd.grad(ls, q)
        loss.append(float(ls.detach()))
        m, v = 0.9 * m + 0.1 * d, 0.999 * v + 0.001 * d * d
        p = p - lr[k] * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return dict(loss=np.array(loss), params=torch.cat([p, P[cut[6]:]]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "wake":
        return _exact_wake(case, seed)
    if kind == "probes":
        return _exact_probes(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    return None   # merging and the boundary system in list order take minutes in plain torch
