"""Placement, merge passes and work items at the sizes where their launches
change: sets below and above the small-set limit, systems that end inside a
wave, cells of one run, of eight runs and beyond (merge passes), columns whose
items are plain runs and columns cut by the row span.  Everything is an integer
or an order: exact."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from oracle import oracle as orc  # noqa: E402


def _greedy_items(counts, offsets, sizes, grids, pitem, yspan):
    """Runs of pitem particles of a column, closed yspan rows below their first."""
    out, c0 = [], 0
    for s, G in enumerate(grids):
        for x in range(G):
            it = None
            for y in range(G):
                c = c0 + x * G + y
                n, p = int(counts[c]), int(offsets[c])
                if n and it is not None and y - it[4] >= yspan:
                    out.append(it)
                    it = None
                while n:
                    if it is None:
                        it = [p, 0, s, x, y, y]
                    t = min(n, pitem - it[1])
                    it[1] += t
                    it[5] = y
                    p += t
                    n -= t
                    if it[1] == pitem:
                        out.append(it)
                        it = None
            if it is not None:
                out.append(it)
        c0 += G * G
    return np.array(out, np.int32).reshape(-1, 6)


@pytest.mark.parametrize("sizes,grids,p,yspan", [
    ([1000], [7], 1, 512), ([1000], [7], 1, 3), ([5000], [40], 2, 40), ([5000], [40], 2, 39),
    ([70001], [50], 4, 512), ([3, 900, 64, 5000, 2], [2, 11, 1, 30, 9], 1, 512),
    ([300, 20000], [600, 20], 2, 512), ([300001], [300], 2, 16)])
def test_items_and_placement(sizes, grids, p, yspan):
    from barneshut.engine import Engine
    d = inputs.batched_uniform(sizes, seed=71)
    eng = Engine(sizes, grids, tuning=dict(p=p, yspan=yspan, waves_per_cu=8, tail_split=1,
                                           tail_items=0))
    eng.load(d)
    for _ in range(2):   # the second time from the sorted rows
        src = eng.fetch()
        eng.create_tree()
        eng.summarize()
        eng.ctx.build_items()
        eng.check()
    counts, offsets, items = eng.counts(), eng.offsets(), eng.items()
    np.testing.assert_array_equal(items[:, :6],
                                  _greedy_items(counts, offsets, sizes, grids, 64 * p, yspan))
    h, com, box = eng.fetch(), eng.com(), eng.bbox()
    p0 = c0 = 0
    for s, (n, G) in enumerate(zip(sizes, grids)):
        sl = slice(p0, p0 + n)
        bb = orc.bbox(src["px"][sl], src["py"][sl], G)
        assert tuple(box[s][[0, 1, 2, 4]]) == (bb[0], bb[1], bb[2], bb[4])
        _, _, key = orc.place(src["px"][sl], src["py"][sl], bb[0], bb[1], bb[4], G)
        np.testing.assert_array_equal(counts[c0:c0 + G * G], np.bincount(key, minlength=G * G))
        order = orc.sort_perm(key, [src[k][sl] for k in ("px", "py", "mass", "vx", "vy", "ax", "ay",
                                                         "pid")])
        np.testing.assert_array_equal(h["pid"][sl], src["pid"][sl][order])
        empty = counts[c0:c0 + G * G] == 0
        assert (com[c0:c0 + G * G][empty] == 0.0).all()
        p0 += n
        c0 += G * G
    eng.close()


@pytest.mark.parametrize("n,G", [(1024, 1), (1025, 1), (8192, 1), (8193, 1), (30000, 1),
                                 (70000, 1), (200000, 2), (300000, 1)])
def test_merge_passes(n, G):
    """One or four cells of up to 300,000 rows, many of them tied in px and py."""
    from barneshut.engine import Engine
    rng = np.random.default_rng(n)
    d = inputs.uniform(n, seed=72)
    d["px"] = np.round(d["px"], 2)
    d["py"] = np.round(d["py"], 1)
    d["mass"] = rng.integers(1, 4, n).astype(np.float64)
    eng = Engine([n], [G])
    eng.load(d)
    eng.create_tree()
    eng.check()
    h, keys = eng.fetch(), eng.keys()
    o = np.lexsort((h["pid"], h["mass"], h["py"], h["px"], keys))
    np.testing.assert_array_equal(o, np.arange(n))
    np.testing.assert_array_equal(np.sort(h["pid"]), np.arange(n))
    eng.close()


@pytest.mark.parametrize("kind", ["px", "px_pairs", "px_py", "rows"])
def test_equal_keys_by_cell_size(kind):
    """One cell a system, of 2 to 1,026 rows, whose px, px and py or whole rows
    tie; a first row elsewhere gives the box an extent."""
    from barneshut.engine import Engine
    rng = np.random.default_rng(5)
    sizes = [2, 3, 7, 8, 9, 10, 15, 16, 17, 18, 64, 66, 1023, 1024, 1025, 1026]
    d = inputs.batched_uniform(sizes, seed=73)
    if kind == "px_pairs":
        d["px"] = np.round(d["px"] * 64) / 64
    else:
        d["px"][:] = 0.25
    if kind in ("px_py", "rows"):
        d["py"][:] = 0.5
    first = np.cumsum([0] + sizes[:-1])
    d["px"][first] = d["py"][first] = 1.0
    d["mass"][:] = 1.0 if kind == "rows" else rng.integers(1, 9, len(d["px"]))
    eng = Engine(sizes, [1] * len(sizes))
    eng.load(d)
    src = eng.fetch()
    eng.create_tree()
    eng.check()
    h = eng.fetch()
    p0 = 0
    for n in sizes:
        sl = slice(p0, p0 + n)
        order = orc.sort_perm(np.zeros(n, np.int64), [src[k][sl] for k in (
            "px", "py", "mass", "vx", "vy", "ax", "ay", "pid")])
        for k in ("pid", "px", "py", "mass"):
            np.testing.assert_array_equal(h[k][sl], src[k][sl][order])
        p0 += n
    eng.close()


@pytest.mark.parametrize("big", [1023, 1024, 1025, 5000])
def test_com_of_large_cells(big):
    """Cells of a few and of `big` rows side by side.  Any order of adding n
    positive numbers is off by at most n ulp, so the quotients by 2 n."""
    from barneshut.engine import Engine
    rng = np.random.default_rng(big)
    G = 9
    cnt = np.where(rng.random(G * G) < 0.2, big, rng.integers(0, 40, G * G))
    cnt[0] = cnt[-1] = 3
    cell = np.repeat(np.arange(G * G), cnt)
    n = len(cell)
    x, y = cell // G + 0.1 + 0.8 * rng.random(n), cell % G + 0.1 + 0.8 * rng.random(n)
    x[0] = y[0] = 0.0
    x[-1] = y[-1] = G   # the box
    d = inputs._pack(x, y, rng.uniform(1, 2, n))
    eng = Engine([n], [G])
    eng.load(d)
    eng.create_tree()
    eng.summarize()
    eng.check()
    h, com, off = eng.fetch(), eng.com(), eng.offsets()
    eng.close()
    np.testing.assert_array_equal(np.diff(off), cnt)
    for c in np.nonzero(cnt)[0]:
        sl = slice(off[c], off[c + 1])
        m = h["mass"][sl].astype(np.longdouble)
        tol = 2 * (cnt[c] + 3) * 2.0 ** -52
        for k, f in ((0, "px"), (1, "py")):
            ref = float((m * h[f][sl]).sum() / m.sum())
            assert abs(com[c][k] - ref) <= tol * abs(ref)
        assert abs(com[c][2] - float(m.sum())) <= tol * float(m.sum())


@pytest.mark.parametrize("n", [2, 511, 513, 2049, 262143, 262145])
def test_unsorted_rows_over_many_cells(n):
    """Every second row in one of three cells, the others over 512^2 cells."""
    from barneshut.engine import Engine
    G = 512
    rng = np.random.default_rng(n)
    x, y = rng.random(n), rng.random(n)
    x[::2] = (rng.integers(0, 3, len(x[::2])) * 100 + 50.2 + 0.6 * rng.random(len(x[::2]))) / G
    y[::2] = (77.2 + 0.6 * rng.random(len(x[::2]))) / G
    eng = Engine([n], [G])
    eng.load(inputs._pack(x, y, rng.uniform(1, 2, n)))
    src = eng.fetch()
    eng.create_tree()
    eng.check()
    bb = orc.bbox(src["px"], src["py"], G)
    _, _, key = orc.place(src["px"], src["py"], bb[0], bb[1], bb[4], G)
    order = orc.sort_perm(key, [src[k] for k in ("px", "py", "mass", "vx", "vy", "ax", "ay",
                                                 "pid")])
    np.testing.assert_array_equal(eng.counts(), np.bincount(key, minlength=G * G))
    np.testing.assert_array_equal(eng.fetch()["pid"], src["pid"][order])
    eng.close()


@pytest.mark.parametrize("sizes,grids", [
    ([2], [1]), ([2], [90]), ([1023], [11]), ([1025], [11]), ([4095], [1]), ([4096], [90]),
    ([4097], [90]), ([4096], [91]), ([3000], [600]), ([70001], [40]), ([500, 9000, 2], [1000, 31, 1]),
    ([500, 66000, 2], [400, 500, 130])])
def test_steps_equal_their_phases(sizes, grids):
    """A step joins the placement of a small system and the items of few columns
    with their neighbours; the phases one by one give the same bits."""
    from barneshut.engine import Engine
    d = inputs.batched_uniform(sizes, seed=74)
    law = (1e-6, 1e-10, 0.0)
    runs = []
    for whole in (True, False):
        eng = Engine(sizes, grids)
        eng.load(d)
        for _ in range(3):
            if whole:
                eng.step(*law, precision="fp64", dt=1e-4)
            else:
                eng.create_tree()
                eng.summarize()
                eng.evaluate(*law, "fp64")
                eng.timestep(1e-4)
            st = eng.check()
        runs.append(dict(eng.fetch(), counts=eng.counts(), offsets=eng.offsets(), com=eng.com(),
                         keys=eng.keys(), items=eng.items(), perm=eng.perm(), box=eng.bbox(),
                         stats=np.array([st[1], st[2], st[4]])))
        eng.close()
    for k, v in runs[0].items():
        np.testing.assert_array_equal(v, runs[1][k])


@pytest.mark.parametrize("n,G", [(500, 5), (524000, 3), (524800, 3)])
def test_cost_order_of_few_and_many_items(n, G):
    """Orders of up to 8,192 items (one block) and of more: a permutation by
    falling cost, to within a bin of the range; the static order if a cost is
    not finite."""
    import torch
    from barneshut.engine import Engine
    eng = Engine([n], [G], tuning=dict(p=1, yspan=512, waves_per_cu=8, tail_split=1, tail_items=0))
    eng.load(inputs.uniform(n, seed=75))
    eng.create_tree()
    eng.ctx.build_items()
    items = int(eng.check()[2])
    cap = eng.ctx.query(4)
    cost = np.random.default_rng(n).normal(size=cap).astype(np.float32)
    cost[:items][:: max(items // 50, 1)] = 0.25   # ties
    order = torch.full((cap,), -1, dtype=torch.int32, device="cuda")
    eng.ctx.order_by_cost(torch.as_tensor(cost, device="cuda"), order)
    o = order.cpu().numpy()
    np.testing.assert_array_equal(np.sort(o[:items]), np.arange(items))
    assert (o[items:] == -1).all()
    c = cost[:items][o[:items]]
    assert (np.diff(c) <= np.ptp(cost[:items]) / 4095 * 1.001).all()
    cost[items // 2] = np.nan
    eng.ctx.order_by_cost(torch.as_tensor(cost, device="cuda"), order)
    np.testing.assert_array_equal(order.cpu().numpy()[:items], np.arange(items))
    eng.close()
