"""The grouped far field (passes of many far terms) against the oracle.

Such passes interpolate the far field on Chebyshev grids instead of taking
every COM on its own.  Tolerances: across a gap of one square the
interpolation leaves about 5.8^-P of a term (P = 12 for fp32: 6.5e-10, P = 20
for fp64: 5e-16), and the FP64 sums round to about 1e-14; both get a factor of
ten, and a particle whose terms cancel may be off by more of its own
acceleration (1e-5 and 1e-9, the library's per-particle targets).
"""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from oracle import oracle as orc  # noqa: E402

NORM = {"fp64": 1e-13, "fp32": 6.5e-9}
EACH = {"fp64": 1e-9, "fp32": 1e-5}


def _engine(n, G, d):
    from barneshut.engine import Engine
    eng = Engine(n, G)
    eng.load(d)
    eng.create_tree()
    eng.summarize()
    return eng


def _pass(eng, law, prec):
    eng.parts["ax"].zero_()
    eng.parts["ay"].zero_()
    eng.evaluate(*law, prec)
    eng.check()
    return eng.fetch()


def _against_oracle(h, G, off, keys, law, prec, seed=3, count=1500):
    """Sampled particles of one system's sorted rows (cells local to it)."""
    com = orc.summarize(off, h["px"], h["py"], h["mass"])
    idx = np.sort(np.random.default_rng(seed).choice(len(h["px"]), count, replace=False))
    rx, ry = orc.forces(G, off, keys, h["px"], h["py"], h["mass"], com, *law, targets=idx)
    num = np.hypot(h["ax"][idx] - rx, h["ay"][idx] - ry)
    den = np.hypot(rx, ry)
    norm = float(np.sqrt((num ** 2).sum() / (den ** 2).sum()))
    each = float((num / den).max())
    print(f"[grouped] {prec} {law}: normwise {norm:.2e}, max {each:.2e}", flush=True)
    return norm, each


def _input(kind):
    n, G = 600001, 193            # a last tile of fewer cells
    if kind == "sparse_columns":   # most tiles empty, some of one cell, a few dense
        rng = np.random.default_rng(41)
        x = np.floor(rng.random(n) * 24) / 24 + 1e-4 * rng.random(n)
        y = rng.random(n) ** 2
        d = inputs._pack(x, y, rng.uniform(1, 2, n))
    else:
        d = inputs.gaussian_mixture(n, 16, (0.005, 0.05), seed=42, background=0.2,
                                    mass="lognormal")
        rng = np.random.default_rng(43)
        clip = (d["px"] == 0) | (d["py"] == 0) | (d["px"] == inputs._UPPER) \
            | (d["py"] == inputs._UPPER)   # no two rows in one place
        d["px"][clip], d["py"][clip] = rng.random(clip.sum()), rng.random(clip.sum())
    if kind == "massless":         # whole cells without mass
        d["mass"][d["px"] < 0.4] = 0.0
    if kind == "signed":           # COMs outside their cells: every term on its own
        d["mass"] *= np.where(np.random.default_rng(44).random(n) < 0.5, -1.0, 1.0)
    if kind == "heavy":
        d["mass"] *= 2.0 ** 400
    return n, G, d


@pytest.mark.parametrize("kind,eps2,r2_cut", [
    ("clusters", 0.0, 0.0), ("clusters", 1e-10, 0.0), ("clusters", 1e-2, 0.0),
    ("clusters", 0.0, 1e-5),       # a cutoff inside a cell
    ("clusters", 1e-8, 1e-2),      # a cutoff past a tile: every term on its own
    ("sparse_columns", 0.0, 0.0), ("massless", 0.0, 0.0), ("signed", 1e-10, 0.0),
    ("heavy", 0.0, 0.0)])
def test_grouped_pass_against_oracle(kind, eps2, r2_cut):
    n, G, d = _input(kind)
    eng = _engine([n], [G], d)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    law = (1e-6 if kind != "heavy" else 1e-6 * 2.0 ** -400, eps2, r2_cut)
    for prec in ("fp64", "fp32"):
        h = _pass(eng, law, prec)
        if prec == "fp32":
            assert int(eng.ctx.stats()[6]) == 0
            again = _pass(eng, law, prec)
            np.testing.assert_array_equal(h["ax"], again["ax"])
            np.testing.assert_array_equal(h["ay"], again["ay"])
        norm, each = _against_oracle(h, G, off, keys, law, prec)
        # signed masses cancel in every particle: FP64 sums of 2e4 terms
        assert norm <= (1e-11 if kind == "signed" else NORM[prec])
        assert each <= (1e-5 if kind == "signed" else EACH[prec])
    eng.close()


@pytest.mark.parametrize("n,G,precisions", [
    (70001, 600, "64"),          # 0.2 particles a cell: tiles of 24 cells
    (600001, 60, "64"),          # 167: 5, near the least far terms that are grouped
    (150001, 500, "64 32"),      # 0.6: 22 and 14
    (400001, 301, "64 32"),      # 4.4: 13 and 8
    (1000003, 97, "64"),         # 106: 6
    (2500001, 90, "64 32")])     # 309: 4 and 4, a last tile of two cells
def test_tile_sizes(n, G, precisions):
    """The tile side follows from particles per cell, by precision."""
    d = inputs.uniform(n, seed=47)
    eng = _engine([n], [G], d)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    for prec in ("fp" + p for p in precisions.split()):
        law = (1e-6, 1e-10, 0.0)
        norm, each = _against_oracle(_pass(eng, law, prec), G, off, keys, law, prec, count=700)
        assert norm <= NORM[prec] and each <= EACH[prec]
    eng.close()


def test_grouped_pass_of_moved_particles():
    """Particles that left their tile since the placement take every COM on
    its own: the pass still evaluates the placed cells at the new positions."""
    n, G, d = _input("clusters")
    eng = _engine([n], [G], d)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    com = eng.com()
    eng.parts["px"][::5000] += 0.3
    law = (1e-6, 1e-10, 0.0)
    h = _pass(eng, law, "fp64")
    idx = np.arange(0, n, 5000)
    rx, ry = orc.forces(G, off, keys, h["px"], h["py"], h["mass"], com, *law, targets=idx)
    num, den = np.hypot(h["ax"][idx] - rx, h["ay"][idx] - ry), np.hypot(rx, ry)
    assert np.sqrt((num ** 2).sum() / (den ** 2).sum()) <= NORM["fp64"]
    assert (num / den).max() <= EACH["fp64"]
    eng.close()


def test_grouped_batch_of_uneven_systems():
    """One context with systems of one tile (grids under 32), of a few tiles
    and of several levels; parts of a pass, a graph replay and an order give
    the bits of one eager pass."""
    import torch
    sizes, grids = [40, 300000, 700, 33000, 5000, 420000], [3, 210, 31, 32, 33, 180]
    d = inputs.batched_uniform(sizes, seed=45)
    law = (1e-6, 1e-12, 0.0)
    eng = _engine(sizes, grids, d)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    for prec in ("fp64", "fp32"):
        h = _pass(eng, law, prec)
        p0 = c0 = 0
        for n, G in zip(sizes, grids):
            sl = slice(p0, p0 + n)
            norm, each = _against_oracle({k: h[k][sl] for k in ("px", "py", "mass", "ax", "ay")}, G,
                                         off[c0:c0 + G * G + 1] - off[c0], keys[sl] - c0, law, prec,
                                         count=min(n, 500))
            assert norm <= NORM[prec] and each <= EACH[prec]
            p0 += n
            c0 += G * G
        eng.ctx.build_items()
        order = torch.arange(int(eng.ctx.stats()[2]) - 1, -1, -1, dtype=torch.int32, device="cuda")
        full = torch.zeros(eng.ctx.query(4), dtype=torch.int32, device="cuda")
        full[:order.numel()] = order
        for parts in (1, 7):
            eng.parts["ax"].zero_()
            eng.parts["ay"].zero_()
            for k in range(parts):
                eng.ctx.force_pass(eng.parts, *law, prec, full, part=k, nparts=parts)
            g = eng.fetch()
            np.testing.assert_array_equal(g["ax"], h["ax"])
            np.testing.assert_array_equal(g["ay"], h["ay"])
    eng.close()
    runs = []
    from barneshut.engine import Engine
    for graph in (False, True):
        e = Engine(sizes, grids)
        e.load(d)
        for _ in range(4):
            e.step(*law, precision="fp32", dt=1e-5, graph=graph)
            torch.cuda.synchronize()
        e.check()
        runs.append(e.fetch())
        e.close()
    for k in ("px", "py", "vx", "vy", "pid"):
        np.testing.assert_array_equal(runs[0][k], runs[1][k])


def test_recompute_call_after_a_grouped_pass():
    """A deferred recompute after a grouped FP32 pass has nothing to do; after
    an FP64 pass it is refused as before."""
    from barneshut.kernels.hiplib import BhError
    n, G, d = _input("clusters")
    eng = _engine([n], [G], d)
    law = (1e-6, 1e-10, 0.0)
    eng.ctx.set_recompute(1.5, deferred=True)
    h = _pass(eng, law, "fp32")
    eng.ctx.recompute(eng.parts, *law)
    g = eng.fetch()
    np.testing.assert_array_equal(g["ax"], h["ax"])
    assert int(eng.ctx.stats()[6]) == 0
    _pass(eng, law, "fp64")
    with pytest.raises(BhError):
        eng.ctx.recompute(eng.parts, *law)
    eng.close()
