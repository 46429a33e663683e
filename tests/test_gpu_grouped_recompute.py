"""The FP64 recompute of grouped FP32 passes (2e10 far terms and more): done
inside the pass, deferred or not, its count in stats [8].  Recomputed particles
carry the FP64 path's value to 1e-9, as after a term-by-term pass
(test_gpu_recompute.py)."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut import inputs  # noqa: E402
from test_gpu_grouped import _engine, _input, _pass  # noqa: E402


def _rel(a, b):
    return np.hypot(a["ax"] - b["ax"], a["ay"] - b["ay"]) / np.hypot(b["ax"], b["ay"])


@pytest.mark.parametrize("kind,law", [
    ("clusters", (1e-6, 1e-10, 0.0)), ("clusters", (0.7, 0.0, 1e-5)), ("massless", (1e-6, 0.0, 0.0)),
    ("heavy", (1e-6 * 2.0 ** -400, 0.0, 0.0)), ("batch", (1e-6, 1e-12, 0.0))])
def test_kappa_holds_for_grouped_passes(kind, law):
    if kind == "batch":
        n, G = [40, 300000, 700, 420000], [3, 210, 31, 180]
        d = inputs.batched_uniform(n, seed=81)
    else:
        n, G, d = _input(kind)
        n, G = [n], [G]
    eng = _engine(n, G, d)
    r64 = _pass(eng, law, "fp64")

    def fp32(kappa, deferred=False):
        eng.ctx.set_recompute(kappa, deferred)
        h = _pass(eng, law, "fp32")
        return h, int(eng.ctx.stats()[8])
    off, none = fp32(0.0)
    assert none == 0
    on, some = fp32(1.5)
    changed = (on["ax"] != off["ax"]) | (on["ay"] != off["ay"])
    print(f"[grouped recompute] {kind}: {some} recomputed, {changed.sum()} changed, their max "
          f"{_rel(on, r64)[changed].max():.2e} (without {_rel(off, r64)[changed].max():.2e})", flush=True)
    assert 0 < changed.sum() <= some < sum(n)
    assert _rel(on, r64)[changed].max() < 1e-9
    late, _ = fp32(1.5, deferred=True)
    np.testing.assert_array_equal(late["ax"], on["ax"])
    every, count = fp32(1e-30)
    assert count == sum(n)
    assert _rel(every, r64).max() < 1e-9
    eng.ctx.set_recompute(1.5)
    _pass(eng, law, "fp64")
    assert int(eng.ctx.stats()[8]) == 0
    eng.close()


def test_parts_of_two_grouped_passes_are_not_mixed():
    """FP64 and FP32 passes form their far fields in one scratch: a part whose
    far field the other precision has replaced is refused, and nothing is added."""
    from barneshut.kernels.hiplib import BhError
    n, G, d = _input("clusters")
    eng = _engine([n], [G], d)
    eng.ctx.build_items()
    law = (1e-6, 1e-10, 0.0)
    want = {p: _pass(eng, law, p) for p in ("fp64", "fp32")}
    for p, other in (("fp64", "fp32"), ("fp32", "fp64")):
        eng.ctx.force_pass(eng.parts, *law, p, part=0, nparts=2)
        eng.ctx.force_pass(eng.parts, *law, other)
        for k in ("ax", "ay"):
            eng.parts[k].zero_()
        with pytest.raises(BhError):
            eng.ctx.force_pass(eng.parts, *law, p, part=1, nparts=2)
        assert not eng.parts["ax"].any()
        for part in range(2):
            eng.ctx.force_pass(eng.parts, *law, p, part=part, nparts=2)
        np.testing.assert_array_equal(eng.fetch()["ax"], want[p]["ax"])
        eng.parts["ax"].zero_()
    eng.close()
