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
