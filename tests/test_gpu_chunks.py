"""Passes by shared chunks (64 particles of one system per block) against the
oracle, at the sizes where chunks, quads and ranges end: one particle, a
chunk less or more one, odd remainders, dense cells (union walk), sparse ones
(a walk per lane), several systems whose chunks start off multiples of 64.
Tolerance: FP64 sums of at most a few thousand terms, each rounded a few times
(1e-13 normwise); a particle whose terms cancel, the library's 1e-9."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from oracle import oracle as orc  # noqa: E402

LAWS = [(1.0, 0.0, 0.0), (0.7, 1e-4, 0.0), (1.0, 0.0, 1e-5), (1.0, 1e-6, 1e-2)]


@pytest.mark.parametrize("prec,norm,each", [("fp64", 1e-13, 1e-9), ("fp32", 1e-6, 1e-5)])
@pytest.mark.parametrize("law", LAWS)
@pytest.mark.parametrize("sizes,grids", [
    ([2], [1]), ([3], [2]), ([63], [3]), ([64], [4]), ([65], [4]), ([129], [2]),
    ([1001], [3]), ([1000], [40]), ([4099], [2]), ([5003], [9]),
    ([2, 65, 7, 1030, 64, 301], [1, 5, 2, 6, 9, 20]),
])
def test_chunks_against_oracle(sizes, grids, law, prec, norm, each):
    from barneshut.engine import Engine
    d = inputs.batched_uniform(sizes, seed=61)
    d["mass"][::7] = 0.0
    eng = Engine(sizes, grids)
    eng.load(d)
    eng.create_tree()
    eng.summarize()
    eng.evaluate(*law, prec)
    eng.check()
    h = eng.fetch()
    off, keys = eng.offsets().astype(np.int64), eng.keys().astype(np.int64)
    p0 = c0 = 0
    for n, G in zip(sizes, grids):
        sl = slice(p0, p0 + n)
        o = off[c0:c0 + G * G + 1] - off[c0]
        com = orc.summarize(o, h["px"][sl], h["py"][sl], h["mass"][sl])
        rx, ry = orc.forces(G, o, keys[sl] - c0, h["px"][sl], h["py"][sl], h["mass"][sl], com,
                            *law)
        num, den = np.hypot(h["ax"][sl] - rx, h["ay"][sl] - ry), np.hypot(rx, ry)
        assert np.sqrt((num ** 2).sum()) <= norm * np.sqrt((den ** 2).sum())
        assert (num <= each * den).all()
        p0 += n
        c0 += G * G
    # parts of a pass give the same bits
    eng.ctx.build_items()
    for k in ("ax", "ay"):
        eng.parts[k].zero_()
    for k in range(3):
        eng.ctx.force_pass(eng.parts, *law, prec, part=k, nparts=3)
    g = eng.fetch()
    np.testing.assert_array_equal(g["ax"], h["ax"])
    np.testing.assert_array_equal(g["ay"], h["ay"])
    eng.close()
