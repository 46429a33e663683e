"""The cutoff on far terms.  A COM outside a particle's 3x3 cells is usually a
cell side away and beyond a smaller cutoff, but not always: masses of both
signs put COMs outside their cells, and a particle may have moved since it was
placed.  The law drops such terms too.  Tolerances as in test_gpu_grouped.py
(FP64 sums of at most 2e4 terms; signed masses cancel in every particle)."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from test_gpu_grouped import EACH, NORM, _engine, _pass  # noqa: E402


@pytest.mark.parametrize("n,G,r2_cut,precisions", [
    (20001, 60, 1e-4, ["fp64"]),              # term by term, 0.36 cell sides squared
    (600001, 193, 1e-5, ["fp64", "fp32"])])   # grouped, 0.37
@pytest.mark.parametrize("kind", ["signed", "moved", "moved_summarized"])
def test_far_terms_within_the_cutoff_are_dropped(kind, n, G, r2_cut, precisions):
    d = inputs.uniform(n, seed=71)
    if kind == "signed":
        d["mass"] *= np.where(np.random.default_rng(72).random(n) < 0.5, -1.0, 1.0)
    eng = _engine([n], [G], d)
    if kind != "signed":
        eng.parts["px"][::50] += 0.3
    if kind == "moved_summarized":   # then COMs leave their cells too
        eng.ctx.summarize(eng.parts)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    com = eng.com()
    idx = np.arange(0, n, 50)[:400]
    for law in ((1e-6, 0.0, r2_cut), (1e-6, 1e-8, r2_cut)):
        for prec in precisions:
            h = _pass(eng, law, prec)
            rx, ry = orc.forces(G, off, keys, h["px"], h["py"], h["mass"], com, *law, targets=idx)
            num, den = np.hypot(h["ax"][idx] - rx, h["ay"][idx] - ry), np.hypot(rx, ry)
            norm = float(np.sqrt((num ** 2).sum() / (den ** 2).sum()))
            print(f"[cutoff] {kind} {G} {prec}: {norm:.2e}, max {(num / den).max():.2e}", flush=True)
            assert norm <= (1e-11 if kind == "signed" else NORM[prec])
            assert (num / den).max() <= (1e-5 if kind == "signed" else EACH[prec])
    eng.close()


def test_cutoff_just_below_a_tile_side():
    """A grouped pass keeps every distant term where the cutoff ends before a
    tile's side h, so it must end before the closest that a distant COM can
    come: a particle 3e-5 h past its tile's edge still counts as inside."""
    n, G, T = 300000, 90, 8          # 2.4e9 far terms, tiles of (130000 G^2 / n)^(1/4) cells
    d = inputs.uniform(n, seed=73)
    h = T / G
    y = 4.5 / G
    d["px"][:4] = [0.0, 1.0, h - 1e-8, 2 * h + 1e-8]   # the box, the particle, a heavy source
    d["py"][:4] = [0.0, 1.0, y, y]
    d["mass"][3] = 1e9
    eng = _engine([n], [G], d)
    i = int(np.nonzero(eng.fetch()["pid"] == d["pid"][2])[0][0])
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    assert keys[i] == (T - 1) * G + 4
    com = eng.com()
    for moved in (0.0, 3e-5 * h):
        eng.parts["px"][i] = h - 1e-8 + moved
        law = (1e-6, 0.0, 0.99996 * h * h)
        r = _pass(eng, law, "fp64")
        rx, ry = orc.forces(G, off, keys, r["px"], r["py"], r["mass"], com, *law,
                            targets=np.array([i]))
        err = np.hypot(r["ax"][i] - rx, r["ay"][i] - ry)[0] / np.hypot(rx, ry)[0]
        print(f"[cutoff] tile side, moved {moved:.1e}: {err:.2e}", flush=True)
        assert err <= EACH["fp64"]
    eng.close()
