"""Measured cases: what a user of this package has it do, through its public
entry points (Engine / Context, BatchedSystems, the cost model's learned
order, and the gravity plugin's device call).

A case is a dict of plain values; `kind` picks the path:

  step    one whole round of one system (placement, order, COMs, forces,
          tick), advancing the state from pass to pass as a run loop does.
          The state is cold but moving (a tenth of the virial speed) and dt is
          small, so every pass does the same work.
  forces  one round without the tick from a fixed unsorted snapshot: the
          accelerations.  The FP32 precisions hand them on in float32, which
          is what they resolve.
  batch   one step of many uneven independent systems in one context, as one
          graph replay, in the static or the learned queue order.
  cloud   the gravity plugin: one cloud on itself.
  leaf    the gravity plugin as a tree code calls it: one leaf against the far
          COMs, against its neighbour leaves (both sides) and on itself.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "barnes-hut_amd"))
from barneshut import costmodel, inputs  # noqa: E402
from barneshut.batched import BATCHED_TUNING, BatchedSystems  # noqa: E402
from barneshut.engine import Engine  # noqa: E402
from barneshut.kernels import hiplib  # noqa: E402

DEV = "cuda:0"
FP64_TUNING = dict(p=2, yspan=512, waves_per_cu=32, tail_split=1, tail_items=0)
STATE = ("px", "py", "mass", "vx", "vy", "pid")


def listed():
    return [
        # a toy run: every launch counts
        dict(name="step_2k_fp64_graph", kind="step", n=2000, grid=11, dist="uniform",
             precision="fp64", eps2=0.0, r2_cut=0.0, G=1e-6, dt=1e-5, graph=True),
        # configs/uniform16k_g32_soft.ini: the case a CPU can still run
        dict(name="step_16k_fp64", kind="step", n=16384, grid=32, dist="uniform",
             precision="fp64", eps2=1e-6, r2_cut=0.0, G=1e-6, dt=1e-5, graph=False),
        # a clustered galaxy of ordinary size, forces for a snapshot
        dict(name="forces_262k_fp32", kind="forces", n=262144, grid=256, dist="clusters",
             clusters=16, s_lo=0.001, s_hi=0.03, background=0.2, mass="uniform",
             precision="fp32", eps2=0.0, r2_cut=0.0, G=1e-6),
        # the reference generator's distribution under the CPU law (cutoff), odd size
        dict(name="forces_1m_fp64_cutoff", kind="forces", n=1000003, grid=100, dist="reference",
             precision="fp64", eps2=0.0, r2_cut=1e-5, G=1.0),
        # FP64 on a fine grid, lognormal masses, sizes off every power of two
        dict(name="forces_700k_fp64", kind="forces", n=700001, grid=601, dist="clusters",
             clusters=256, s_lo=0.001, s_hi=0.03, background=0.0, mass="lognormal",
             precision="fp64", eps2=1e-10, r2_cut=0.0, G=1e-6),
        # the reference's logged configuration: 10M particles, 1000 per box
        dict(name="step_10m_fp64", kind="step", n=10000000, grid=120, dist="uniform",
             precision="fp64", eps2=0.0, r2_cut=0.0, G=1e-6, dt=1e-5, graph=False),
        # the bench workload, FP32 and FP64
        dict(name="step_4m_fp32", kind="step", n=4194304, grid=1024, dist="clusters", clusters=64,
             s_lo=0.005, s_hi=0.05, background=0.0, mass="uniform", precision="fp32",
             eps2=1e-10, r2_cut=0.0, G=1e-6, dt=1e-5, graph=False),
        dict(name="step_4m_fp64", kind="step", n=4194304, grid=1024, dist="clusters", clusters=64,
             s_lo=0.005, s_hi=0.05, background=0.0, mass="uniform", precision="fp64",
             eps2=1e-10, r2_cut=0.0, G=1e-6, dt=1e-5, graph=False),
        # 512 uneven systems as one graph replay per step
        dict(name="batch_512_fp32", kind="batch", systems=512, lo=1024, hi=262144, sizes_seed=0,
             precision="fp32", learned=False, eps2=1e-12, G=1e-6, dt=1e-5),
        # a small batch of small systems in the learned order
        dict(name="batch_40_fp32_learned", kind="batch", systems=40, lo=1024, hi=16384,
             sizes_seed=3, precision="fp32", learned=True, eps2=1e-12, G=1e-6, dt=1e-5),
        # direct sum of one cloud, the plugin's largest ordinary call
        dict(name="cloud_100k", kind="cloud", n=100003, eps2=0.0, r2_cut=1e-5),
        # what a tree code asks of the plugin for one leaf
        dict(name="leaf_64", kind="leaf", n=64, far=16384, neighbours=8, eps2=0.0, r2_cut=1e-5),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "forces", "forces", "forces", "batch", "cloud",
                       "leaf"])
    if kind == "batch":
        return dict(kind=kind, systems=int(_log(rng, 3, 512)), lo=1024,
                    hi=int(_log(rng, 8192, 262144)), sizes_seed=rng.randrange(1 << 20),
                    precision="fp32", learned=rng.random() < 0.5, eps2=1e-12, G=1e-6, dt=1e-5)
    if kind == "cloud":
        return dict(kind=kind, n=int(_log(rng, 64, 150000)), eps2=rng.choice([0.0, 1e-6]),
                    r2_cut=1e-5)
    if kind == "leaf":
        return dict(kind=kind, n=int(_log(rng, 1, 1000)), far=int(_log(rng, 64, 65536)),
                    neighbours=rng.choice([3, 5, 8]), eps2=0.0, r2_cut=1e-5)
    n = int(_log(rng, 1000, 4194304))
    per_cell = _log(rng, 3, 1000)
    grid = max(2, min(1024, round(math.sqrt(n / per_cell))))
    # whole steps stand for the largest
    grid = min(grid, int(math.sqrt((3e11 if kind == "forces" else 1.9e12) / n)))
    c = dict(kind=kind, n=n, grid=grid, dist=rng.choice(["uniform", "clusters", "clusters",
                                                         "reference"]),
             precision=rng.choice(["fp32", "fp64"]), eps2=rng.choice([0.0, 1e-12, 1e-10, 1e-8]),
             r2_cut=0.0, G=1e-6)
    if c["dist"] == "clusters":
        c.update(clusters=int(_log(rng, 4, 256)), s_lo=rng.choice([0.002, 0.005]),
                 s_hi=rng.choice([0.03, 0.05]), background=rng.choice([0.0, 0.2]),
                 mass=rng.choice(["uniform", "lognormal"]))
    if c["dist"] == "reference" and rng.random() < 0.5:
        c["r2_cut"] = 1e-5
    if kind == "step":
        c.update(dt=1e-5, graph=rng.random() < 0.3)
    while _near_pairs(c, c["n"], c["grid"]) > 5e10:   # a cluster inside a cell or two
        c["n"] = c["n"] * 2 // 3
    return c


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 11)


def _particles(c, n, seed):
    """px, py, mass, vx, vy of one system as float64 device tensors."""
    g = _gen(seed)

    def rand(*s):
        return torch.rand(*s, generator=g, device=DEV, dtype=torch.float64)

    def randn(*s):
        return torch.randn(*s, generator=g, device=DEV, dtype=torch.float64)

    if c.get("dist", "uniform") == "reference":   # U[0, 499), mass U[0.5, 5], velocity U[-1, 1]
        p = rand(n, 2) * 499.0
        return p[:, 0], p[:, 1], 0.5 + 4.5 * rand(n), 2 * rand(n) - 1, 2 * rand(n) - 1
    if c.get("dist") == "clusters":
        k = c["clusters"]
        nb = round(n * c["background"])
        centre = rand(k, 2)
        sigma = torch.exp(math.log(c["s_lo"]) + math.log(c["s_hi"] / c["s_lo"]) * rand(k))
        lab = torch.randint(0, k, (n,), generator=g, device=DEV)
        p = centre[lab] + randn(n, 2) * sigma[lab][:, None]
        back = torch.randperm(n, generator=g, device=DEV)[:nb]
        p[back] = rand(nb, 2)
        # a point past the box is drawn again inside it: no two rows share a place
        p = torch.where((p < 0) | (p >= 1), rand(n, 2), p)
    else:
        p = rand(n, 2)
    m = torch.exp(0.5 * randn(n)) if c.get("mass") == "lognormal" else 1.0 + rand(n)
    v = 0.1 * math.sqrt(c.get("G", 1e-6) * 1.5 * n) * randn(n, 2)
    return p[:, 0], p[:, 1], m, v[:, 0], v[:, 1]


def _fill(parts, d, o=0):
    n = d[0].numel()
    for k, t in zip(("px", "py", "mass", "vx", "vy"), d):
        parts[k][o:o + n].copy_(t)
    parts["pid"][o:o + n].copy_(torch.arange(n, dtype=torch.int32, device=DEV))


def _sizes(c):
    return inputs.batched_sizes(c["systems"], c["lo"], c["hi"], seed=c["sizes_seed"])


def _rows(n, seed, lo=0.0, hi=1.0):
    g = _gen(seed)
    r = torch.zeros(n, 10, dtype=torch.float64, device=DEV)
    r[:, :2] = lo + (hi - lo) * torch.rand(n, 2, generator=g, device=DEV, dtype=torch.float64)
    r[:, 2] = 1.0 + torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    return r


def _leaf_rows(c, seed):
    """The leaf in the unit cell, its neighbours in the cells around it, far COMs
    over a 128-cell square."""
    own = _rows(c["n"], seed)
    near = []
    for i in range(c["neighbours"]):
        r = _rows(c["n"], seed + 1000 + i)
        r[:, 0] += (-1, 1, 0, 0, -1, -1, 1, 1)[i]
        r[:, 1] += (0, 0, -1, 1, -1, 1, -1, 1)[i]
        near.append(r)
    return own, _rows(c["far"], seed + 2000, 2.0, 130.0), near


def prepare(c, seed):
    if c["kind"] == "cloud":
        return dict(case=c, rows=_rows(c["n"], seed))
    if c["kind"] == "leaf":
        own, far, near = _leaf_rows(c, seed)
        return dict(case=c, own=own, far=far, near=near)
    if c["kind"] == "batch":
        sizes, grids = _sizes(c)
        N = int(sizes.sum())
        one = {k: torch.zeros(N, dtype=torch.float64, device=DEV)
               for k in ("px", "py", "mass", "vx", "vy")}
        one["pid"] = torch.zeros(N, dtype=torch.int32, device=DEV)
        o = 0
        for i, n in enumerate(sizes):
            _fill(one, _particles(c, int(n), seed * 100003 + i), o)
            o += int(n)
        model = None
        if c["learned"]:
            model = costmodel.CostModel.load(
                os.path.join(os.getcwd(), "barnes-hut_amd", "costmodels", "batched512.npz"),
                device=torch.device(DEV))
        b = BatchedSystems(sizes, grids, {k: v.cpu().numpy() for k, v in one.items()},
                           (c["G"], c["eps2"], 0.0), c["precision"], c["dt"],
                           tuning=BATCHED_TUNING, model=model, graph=True)
        return dict(case=c, batch=b)
    # the drop-in's launch shapes: FP64 items are never split, FP32 defaults
    eng = Engine([c["n"]], [c["grid"]], tuning=FP64_TUNING if c["precision"] == "fp64" else None)
    _fill(eng.parts, _particles(c, c["n"], seed))
    torch.cuda.synchronize()
    return dict(case=c, eng=eng)


def run(s):
    c = s["case"]
    if c["kind"] == "cloud":
        s["rows"][:, 5:7].zero_()
        hiplib.cloud_gravity(s["rows"], eps2=c["eps2"], r2_cut=c["r2_cut"])
        return s["rows"]
    if c["kind"] == "leaf":
        own, near = s["own"], s["near"]
        for r in [own] + near:
            r[:, 5:7].zero_()
        hiplib.cloud_gravity(own, s["far"], eps2=c["eps2"], r2_cut=c["r2_cut"])
        for r in near:
            hiplib.cloud_gravity(own, r, eps2=c["eps2"], r2_cut=c["r2_cut"], update_other=True)
        hiplib.cloud_gravity(own, eps2=c["eps2"], r2_cut=c["r2_cut"])
        return [own] + near
    if c["kind"] == "batch":
        s["batch"].step()
        return {k: s["batch"].eng.parts[k] for k in STATE}
    eng = s["eng"]
    if c["kind"] == "step":
        eng.step(c["G"], c["eps2"], c["r2_cut"], c["precision"], c["dt"], True, c["graph"])
        return {k: eng.parts[k] for k in STATE}
    out = eng.other
    eng.ctx.step(eng.parts, out, c["G"], c["eps2"], c["r2_cut"], c["precision"], 0.0, False)
    if c["precision"] == "fp64":
        return dict(ax=out["ax"], ay=out["ay"], pid=out["pid"])
    return dict(ax=out["ax"].float(), ay=out["ay"].float(), pid=out["pid"])


# ---------------------------------------------------------------- floors

def _near_pairs(c, n, grid):
    """Expected pairs in 3x3 cells: 9 n^2 times the integral of the squared
    density over one cell."""
    lump = 1.0
    if c.get("dist") == "clusters":
        w = 1.0 - c["background"]
        inv = (c["s_lo"] ** -2 - c["s_hi"] ** -2) / (2 * math.log(c["s_hi"] / c["s_lo"]))
        lump += w * w * inv / (4 * math.pi * c["clusters"])
    return min(float(n) * n, 9.0 * n * n / grid ** 2 * lump)


def work(c):
    """Each row read and written once; 11 flop a pair for the pairs that the
    method takes one by one (3x3 cells, or all pairs of two clouds), and one
    such term per particle for the far field, which can be summed in groups."""
    if c["kind"] == "cloud":
        return dict(bytes=c["n"] * 72, flops=11 * float(c["n"]) ** 2)
    if c["kind"] == "leaf":
        k = c["neighbours"]
        rows = c["n"] * (1 + k)
        return dict(bytes=rows * 72 + c["far"] * 24,
                    flops=11.0 * c["n"] * (c["far"] + (1 + 2 * k) * c["n"]))
    if c["kind"] == "batch":
        sizes, grids = _sizes(c)
        return dict(bytes=120.0 * float(sizes.sum()),
                    flops=11.0 * sum(_near_pairs(c, int(n), int(g)) + int(n)
                                     for n, g in zip(sizes, grids)))
    return dict(bytes=120.0 * c["n"], flops=11.0 * (_near_pairs(c, c["n"], c["grid"]) + c["n"]))


# ---------------------------------------------------------------- 64-bit values

def _weights(r2, c):
    w = 1.0 / (r2 + c["eps2"])
    return torch.where(r2 > c["r2_cut"], w, torch.zeros_like(w)) if c.get("r2_cut") else w


def _grid_forces(px, py, m, c, G):
    """Placement order and accelerations of the grid method: pairs of the 3x3
    cells one by one, every other non-empty cell by its centre of mass."""
    n = px.numel()
    mnx, mny = px.min(), py.min()
    step = torch.maximum(px.max() - mnx, py.max() - mny) / G
    gx = torch.floor((px - mnx) / step).clamp(0, G - 1).long()
    gy = torch.floor((py - mny) / step).clamp(0, G - 1).long()
    key = gx * G + gy
    o = torch.argsort(px, stable=True)
    o = o[torch.argsort(key[o], stable=True)]
    x, y, m, key = px[o], py[o], m[o], key[o]
    cnt = torch.bincount(key, minlength=G * G)
    off = torch.zeros(G * G + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(cnt, 0)
    M, X, Y = (torch.zeros(G * G, dtype=torch.float64, device=DEV) for _ in range(3))
    M.index_add_(0, key, m)
    X.index_add_(0, key, m * x)
    Y.index_add_(0, key, m * y)
    ne = torch.nonzero(cnt).flatten()
    M, kx, ky = M[ne], ne // G, ne % G
    X, Y = X[ne] / M, Y[ne] / M
    ax, ay = torch.zeros_like(x), torch.zeros_like(x)
    a = 0
    rows = max(1, min(n, int(1.5e8) // max(1, ne.numel())))
    while a < n:
        b = min(n, a + rows)
        cx, cy = key[a:b, None] // G, key[a:b, None] % G
        dx, dy = X[None] - x[a:b, None], Y[None] - y[a:b, None]
        near = ((kx[None] - cx).abs() <= 1) & ((ky[None] - cy).abs() <= 1)
        w = M[None] * _weights(dx * dx + dy * dy, c)
        w.masked_fill_(near, 0.0)
        ax[a:b] += (w * dx).sum(1)
        ay[a:b] += (w * dy).sum(1)
        a = b
    cx, cy = key // G, key % G
    for t in (-1, 0, 1):
        col = cx + t
        ok = (col >= 0) & (col < G)
        base = col.clamp(0, G - 1) * G
        lo = torch.where(ok, off[base + (cy - 1).clamp(min=0)], 0)
        num = torch.where(ok, off[base + (cy + 1).clamp(max=G - 1) + 1], 0) - lo
        by = torch.argsort(num)        # rows of like length together
        a = 0
        while a < n:
            b = min(n, a + 4096)
            while b < n and (b - a) * int(num[by[min(n, 2 * b - a) - 1]]) < 5e7:
                b = min(n, 2 * b - a)
            i = by[a:b]
            k = torch.arange(int(num[i].max()), device=DEV)[None]
            j = (lo[i, None] + k).clamp(max=n - 1)
            keep = (k < num[i, None]) & (j != i[:, None])
            dx, dy = x[j] - x[i, None], y[j] - y[i, None]
            w = m[j] * _weights(torch.where(keep, dx * dx + dy * dy, 1.0), c)
            w = torch.where(keep, w, 0.0)
            ax[i] += (w * dx).sum(1)
            ay[i] += (w * dy).sum(1)
            a = b
    return o, ax * c["G"], ay * c["G"]


def _exact_system(c, n, G, seed, out):
    px, py, m, vx, vy = _particles(c, n, seed)
    o, ax, ay = _grid_forces(px, py, m, dict(c, r2_cut=c.get("r2_cut", 0.0)), G)
    if c["kind"] == "forces":
        out.append(dict(ax=ax, ay=ay, pid=None))
        return
    vx, vy = vx[o] + ax * c["dt"], vy[o] + ay * c["dt"]
    out.append(dict(px=px[o] + vx * c["dt"], py=py[o] + vy * c["dt"], mass=m[o], vx=vx, vy=vy,
                    pid=None))


def _cloud_on(a, b, c, same):
    s = torch.zeros(a.shape[0], 2, dtype=torch.float64, device=DEV)
    for i in range(0, a.shape[0], 1024):
        t = a[i:i + 1024]
        dx, dy = b[None, :, 0] - t[:, None, 0], b[None, :, 1] - t[:, None, 1]
        r2 = dx * dx + dy * dy
        if same:
            k = torch.arange(t.shape[0], device=DEV)
            r2[k, k + i] = 1.0
        w = b[None, :, 2] * _weights(r2, c)
        if same:
            w[k, k + i] = 0.0
        s[i:i + 1024, 0] = (w * dx).sum(1)
        s[i:i + 1024, 1] = (w * dy).sum(1)
    return s


def exact(c, seed):
    """The method's result in 64 bits from its definition, term by term; None
    where that many terms take too long."""
    if c["kind"] == "cloud":
        r = _rows(c["n"], seed)
        r[:, 5:7] = _cloud_on(r, r, c, True)
        return r
    if c["kind"] == "leaf":
        own, far, near = _leaf_rows(c, seed)
        s = _cloud_on(own, far, c, False) + _cloud_on(own, own, c, True)
        back = [_cloud_on(r, own, c, False) for r in near]
        for r in near:
            s += _cloud_on(own, r, c, False)
        own[:, 5:7] = s
        for r, t in zip(near, back):
            r[:, 5:7] = t
        return [own] + near
    if c["kind"] == "batch":
        sizes, grids = _sizes(c)
        jobs = [(int(n), int(g), seed * 100003 + i) for i, (n, g) in enumerate(zip(sizes, grids))]
    else:
        jobs = [(c["n"], c["grid"], seed)]
    if sum(n * min(n, float(g) ** 2) + 4 * _near_pairs(c, n, g) for n, g, _ in jobs) > 2.7e11 \
            or len(jobs) > 100:
        return None
    out = []
    for n, g, sd in jobs:
        _exact_system(c, n, g, sd, out)
    return {k: None if k == "pid" else torch.cat([t[k] for t in out]) for k in out[0]}
