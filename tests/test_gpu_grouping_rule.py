"""Which passes are grouped: a rule on all systems of a context, which bh_query
tells (6 and 7: nodes per square side of FP64 and FP32 passes, 8 and 9: cells
per tile side of the first system; 0: term by term).  A system's result does not
depend on its neighbours beyond rounding: bit for bit where the form is the same,
to the grouped forms' accuracy where it differs."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from test_gpu_grouped import EACH, NORM, _engine, _pass  # noqa: E402


@pytest.mark.parametrize("sizes,grids,nodes,tiles", [
    ([262144], [256], (0, 0), (0, 0)),                  # the largest of the step without allocation
    ([262145], [256], (20, 0), (13, 0)),
    ([262144] * 2, [256] * 2, (20, 12), (13, 9)),       # 3.4e10 far terms together
    ([555000], [60], (0, 0), (0, 0)),                   # 1.998e9
    ([556000], [60], (20, 0), (5, 0)),                  # 2.0016e9
    ([600001], [182], (20, 0), (9, 0)),                 # 1.987e10
    ([600001], [183], (20, 12), (9, 6)),                # 2.009e10
    ([3000, 2000], [12, 9], (0, 0), (0, 0))])
def test_rule(sizes, grids, nodes, tiles):
    from barneshut.kernels.hiplib import BhError, Context
    c = Context()
    c.set_systems(sizes, grids)
    assert (c.query(6), c.query(7)) == nodes
    assert (c.query(8), c.query(9)) == tiles
    with pytest.raises(BhError):
        c.query(10)
    c.close()


@pytest.mark.parametrize("n,G,prec,same", [
    (3000, 12, "fp64", True), (3000, 12, "fp32", True),
    (20000, 90, "fp64", True),         # 1.6e8 far terms each: two stay below the line
    (100000, 100, "fp64", False),      # 1e9 each: two are on it
    (100000, 150, "fp64", False),      # 2.25e9 each, a single one within the other step's limits
    (600001, 193, "fp64", True), (600001, 193, "fp32", True),   # grouped by themselves
    (262144, 230, "fp32", False)])     # 1.4e10 each
def test_a_system_and_its_copies(n, G, prec, same):
    d = inputs.uniform(n, seed=85)
    law = (1e-6, 1e-9, 0.0)
    runs = []
    for k in (1, 2):
        eng = _engine([n] * k, [G] * k, {f: np.tile(v, k) for f, v in d.items()})
        runs.append(_pass(eng, law, prec))
        eng.close()
    one, two = runs
    for f in ("px", "ax", "ay"):
        np.testing.assert_array_equal(two[f][:n], two[f][n:])
    if same:
        np.testing.assert_array_equal(two["ax"][:n], one["ax"])
        np.testing.assert_array_equal(two["ay"][:n], one["ay"])
        return
    num = np.hypot(two["ax"][:n] - one["ax"], two["ay"][:n] - one["ay"])
    den = np.hypot(one["ax"], one["ay"])
    norm = float(np.sqrt((num ** 2).sum() / (den ** 2).sum()))
    print(f"[rule] {n} {G} {prec}: {norm:.2e}, max {(num / den).max():.2e}", flush=True)
    assert 0 < norm <= (NORM["fp64"] if prec == "fp64" else 1e-6)   # fp32 by terms: 4e-8
    assert (num / den).max() <= EACH[prec]


@pytest.mark.parametrize("n,G,prec,tile", [
    (262144, 256, "fp64", None), (262145, 256, "fp64", 13),
    (600001, 193, "fp32", 6), (600001, 193, "fp64", 9)])   # (c G^2 / n)^(1/4): 6.08, 9.48
def test_benchmark_counts_the_form_that_ran(n, G, prec, tile):
    """The benchmark's accounting of a pass follows the library's form, on
    clusters too, where few cells hold particles."""
    import bench
    d = inputs.gaussian_mixture(n, 8, (0.005, 0.03), seed=86)
    r = bench.measure(d, G, prec, None, 1, 0)
    if tile is None:
        assert r["grouped"] is None
        assert r["flop_per_launch"] == bench.FLOP_PER_INTERACTION * (r["near"][0] + r["far"][0])
    else:
        assert r["grouped"]["tile_side"] == tile
        assert r["grouped"]["near_terms"] == r["near"][0]
