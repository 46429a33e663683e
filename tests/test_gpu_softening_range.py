"""Softening at the ends of its range.  Several terms share a reciprocal, whose
denominator is the product of theirs: it must not leave a double's range where
the terms themselves do not.  Tiny softening, there only to keep coincident
particles from dividing by zero, and softening far beyond the box.  Tolerance:
FP64 sums of at most 2e4 terms (1e-13 normwise; a particle whose terms cancel,
the library's 1e-9), grouped FP32 passes as in test_gpu_grouped.py."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from test_gpu_grouped import EACH, NORM, _engine, _pass  # noqa: E402


@pytest.mark.parametrize("n,G,prec", [
    (5001, 3, "fp64"),       # chunks of one column, by quads
    (9001, 40, "fp64"),      # a walk per lane
    (300001, 90, "fp64"),    # grouped
    (600001, 193, "fp32")])
@pytest.mark.parametrize("eps2", [1e-300, 1e-80, 1e74, 1e90])
@pytest.mark.parametrize("r2_cut", [0.0, 1e-6])
def test_extreme_softening(n, G, prec, eps2, r2_cut):
    d = inputs.uniform(n, seed=91)
    for k in ("px", "py"):           # groups of eight in one place
        for j in range(1, 8):
            d[k][j:800:8] = d[k][0:800:8]
    eng = _engine([n], [G], d)
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    com = eng.com()
    law = (max(1.0, eps2), eps2, r2_cut)   # G brings the sums back into range
    h = _pass(eng, law, prec)
    eng.close()
    idx = np.unique(np.concatenate([np.nonzero(h["pid"] < 800)[0][:200], np.arange(0, n, n // 200)]))
    rx, ry = orc.forces(G, off, keys, h["px"], h["py"], h["mass"], com, *law, targets=idx)
    num, den = np.hypot(h["ax"][idx] - rx, h["ay"][idx] - ry), np.hypot(rx, ry)
    assert np.isfinite(den).all()
    print(f"[softening] {prec} {n} {G} {eps2} {r2_cut}: finite {np.isfinite(num).mean():.2f}, "
          f"{np.sqrt((num ** 2).sum() / (den ** 2).sum()):.2e}, max {(num / den).max():.2e}", flush=True)
    assert np.sqrt((num ** 2).sum() / (den ** 2).sum()) <= NORM[prec]
    assert (num / den).max() <= EACH[prec]
