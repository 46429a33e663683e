"""Large clouds take their sources in pairs that share a reciprocal: against the
oracle at the line where that starts, with odd remainders, pairs that the cutoff
drops, coincident rows, and coordinates whose squared products leave a double's
range (those rows go one by one).  Tolerance: each row within 1e-12 of the sum
of its terms' magnitudes, as for the rows taken one by one."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

from barneshut.kernels import hiplib  # noqa: E402
from oracle import oracle as orc  # noqa: E402


def _rows(n, seed, scale):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 10))
    r[:, :2] = rng.random((n, 2)) * scale
    r[:, 2] = rng.uniform(1.0, 2.0, n)
    r[1::97, :2] = r[0, :2]          # coincident rows
    r[:, 5:7] = rng.normal(size=(n, 2)) * 1e-30   # added to, not overwritten
    return r


def _magnitude(a, b, eps2, r2_cut, same):
    """Sum of |term| per row of a."""
    out = np.zeros(len(a))
    for i in range(0, len(a), 512):
        d = b[None, :, :2] - a[i:i + 512, None, :2]
        r2 = (d ** 2).sum(-1)
        keep = r2 > r2_cut if r2_cut > 0 else np.ones_like(r2, bool)
        if same:
            k = np.arange(len(r2))
            keep[k, k + i] = False
        with np.errstate(divide="ignore", invalid="ignore"):
            t = np.where(keep, b[None, :, 2] * np.sqrt(r2) / (r2 + eps2), 0.0)
        out[i:i + 512] = t.sum(1)
    return out


@pytest.mark.parametrize("scale,eps2,r2_cut", [
    (1.0, 0.0, 1e-5), (1.0, 1e-6, 1e-5), (1.0, 1e-6, 0.0), (30.0, 0.0, 1e-3),
    (1e-90, 1e-190, 0.0),            # Q near 1e-360
    (1e80, 0.0, 1e-5)])              # Q near 1e320
@pytest.mark.parametrize("n", [6000, 6001, 8193])
def test_cloud_on_itself_in_pairs(n, scale, eps2, r2_cut):
    import torch
    a = _rows(n, n, scale)
    dev = torch.as_tensor(a, device="cuda")
    hiplib.cloud_gravity(dev, G=1.0, eps2=eps2, r2_cut=r2_cut)
    acc = orc.cloud_gravity(a, None, 1.0, eps2, r2_cut)[0]
    got = dev.cpu().numpy()
    assert np.isfinite(acc).all()
    mag = _magnitude(a, a, eps2, r2_cut, True)
    err = np.abs(got[:, 5:7] - (a[:, 5:7] + acc))
    assert (err <= 1e-12 * mag[:, None] + 1e-40).all()
    np.testing.assert_array_equal(got[:, [0, 1, 2, 3, 4, 7, 8, 9]], a[:, [0, 1, 2, 3, 4, 7, 8, 9]])


def test_two_clouds_both_sides_in_pairs():
    """Both directions of one call, also where the two are views of one array."""
    import torch
    a, b = _rows(6500, 1, 1.0), _rows(7001, 2, 1.0)
    da, db = torch.as_tensor(a, device="cuda"), torch.as_tensor(b, device="cuda")
    hiplib.cloud_gravity(da, db, eps2=0.0, r2_cut=1e-5, update_other=True)
    one, two = torch.as_tensor(a, device="cuda"), torch.as_tensor(b, device="cuda")
    hiplib.cloud_gravity(one, db, eps2=0.0, r2_cut=1e-5)
    hiplib.cloud_gravity(two, da, eps2=0.0, r2_cut=1e-5)
    np.testing.assert_array_equal(da.cpu().numpy(), one.cpu().numpy())
    np.testing.assert_array_equal(db.cpu().numpy(), two.cpu().numpy())
    whole = torch.as_tensor(np.concatenate([a, b]), device="cuda")
    u, v = whole[:9000], whole[4000:]          # 5,000 rows in both
    first, second = u.clone(), v.clone()
    hiplib.cloud_gravity(u, v, eps2=1e-6, r2_cut=0.0, update_other=True)
    w = torch.as_tensor(np.concatenate([a, b]), device="cuda")
    hiplib.cloud_gravity(w[:9000], second, eps2=1e-6, r2_cut=0.0)
    hiplib.cloud_gravity(w[4000:], first, eps2=1e-6, r2_cut=0.0)
    np.testing.assert_array_equal(whole.cpu().numpy(), w.cpu().numpy())


@pytest.mark.parametrize("n", [6001, 30011, 70000])
def test_rounding_does_not_grow_with_the_cloud(n):
    """Sums by tiles of 256 rows: at most 16 + n / 256 roundings in a lane's
    chain, of independent signs, so a few 1e-16 of the sums at any size."""
    import torch
    rng = np.random.default_rng(n)
    rows = np.zeros((n, 10))
    rows[:, :2], rows[:, 2] = rng.random((n, 2)), rng.uniform(1, 2, n)
    dev = torch.as_tensor(rows, device="cuda")
    hiplib.cloud_gravity(dev, None, eps2=0.0, r2_cut=1e-5)
    got = dev.cpu().numpy()
    x, y, m = (rows[:, k].astype(np.longdouble) for k in range(3))
    num = den = 0.0
    for i in rng.choice(n, 60, replace=False):
        dx, dy = x - x[i], y - y[i]
        r2 = dx * dx + dy * dy
        w = np.where(r2 > 1e-5, m / np.where(r2 > 0, r2, 1), 0)
        ex, ey = (dx * w).sum(), (dy * w).sum()
        num += (got[i, 5] - ex) ** 2 + (got[i, 6] - ey) ** 2
        den += ex * ex + ey * ey
    assert float((num / den) ** 0.5) <= 4e-16
