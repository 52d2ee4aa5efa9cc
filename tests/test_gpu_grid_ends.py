"""Linear-grid tools towards the band ends: a damped table of levels inside the
band, where the double sums nearly cancel for |x| -> 1, against sums in extended
precision.  The tools may not be further off than six times the oracle's double
sums, which add the same terms in the same form: the host's functions are right to
about half a unit in the last place, the device's to two, and the order of the
sums differs."""
import numpy as np
import pytest

import linqt_amd as lq

pytestmark = pytest.mark.gpu

PI = np.longdouble("3.14159265358979323846264338327950288")


def _table(M, seed):
    rng = np.random.default_rng(seed)
    J = 96
    tx, ty = np.arccos(rng.uniform(-0.93, 0.93, J)), np.arccos(rng.uniform(-0.93, 0.93, J))
    w = (rng.normal(size=J) + 1j * rng.normal(size=J)) / J
    m = np.arange(M)
    t = (np.cos(np.outer(m, tx)) * w) @ np.cos(np.outer(m, ty)).T
    mu = 2.0 * (t + t.conj().T)
    mu[0] *= 0.5
    mu[:, 0] *= 0.5
    p = np.pi / (M + 1.0)
    g = ((M - m + 1) * np.cos(p * m) + np.sin(p * m) / np.tan(p)) * p / np.pi
    return mu * np.outer(g, g)


def _exact(kind, mu, n, W, x):
    """The tools' kernels at x, scaled, in extended precision."""
    M = mu.shape[0]
    x = x.astype(np.longdouble)
    th, f = np.arccos(x), np.sqrt((1 - x) * (1 + x))
    m = np.arange(M).astype(np.longdouble)
    c, s = np.cos(np.outer(th, m)), np.sin(np.outer(th, m))
    re, im = mu.real.astype(np.longdouble), mu.imag.astype(np.longdouble)
    zr, zi = c @ re, c @ im
    a = np.longdouble(W) / 2
    if kind == 6:
        return PI * n / a / a * (c * zr).sum(1) / (PI * f) ** 2
    if kind == 2:
        fi = c * (m * f[:, None]) - s * x[:, None]  # Im of (x + i m f) e^{-i m theta}
        fr = c * x[:, None] + s * (m * f[:, None])
        return -2 * n / a / a * (fi * zi - fr * zr).sum(1) / f**3 / (PI * f)
    return -n / a / a * (-s * zi - c * zr).sum(1) / f / (PI * f)


@pytest.mark.parametrize("kind,M,nd", [(1, 64, 801), (6, 64, 801), (6, 97, 1501), (2, 97, 3000)])
def test_band_ends(ctx, oracle, kind, M, nd):
    print("[case] band ends", kind, M, nd, flush=True)
    mu, n, W = _table(M, 3), 5000, 9.2
    xb = 0.99 if kind == 2 else 1.0
    x = -xb + np.arange(nd) * (2 * xb) / (nd - 1)
    ends = np.abs(x) > 0.96
    k = _exact(kind, mu, n, W, np.clip(x, -0.9999999, 0.9999999))
    if kind == 2:  # the running sum printed on the low end's rows
        want = np.cumsum(k[:-1] * np.diff(x.astype(np.longdouble)))
        rows = ends[:-1] & (x[:-1] < 0)
    elif kind == 6:  # means of neighbours; x = +-1 has no value
        want = (k[1:] + k[:-1]) / 2
        rows = ends[:-1] & ends[1:]
        rows[[0, -1]] = False
    else:
        want, rows = k[:-1], ends[:-1].copy()
        rows[0] = False
    _, got = lq.linear_grid(ctx, kind, mu, n, W, 0.0, nd)
    _, ref = oracle.linear_grid(kind, mu, n, W, 0.0, nd)
    err = np.abs(got[rows] - want[rows]).max()
    limit = np.abs(ref[rows] - want[rows]).max()
    assert 0 < limit < 1e-9 * np.abs(want).max()
    assert err <= 6 * limit


@pytest.mark.parametrize("kind,M1", [(2, 3), (5, 1), (6, 2)])
def test_most_orders(ctx, oracle, kind, M1):
    """4096 orders, the most a block's left vectors hold."""
    print("[case] most orders", kind, M1, flush=True)
    rng = np.random.default_rng(M1)
    mu = (rng.normal(size=(4096, M1)) + 1j * rng.normal(size=(4096, M1))) * np.exp(-np.arange(4096) / 300.0)[:, None]
    E, v = lq.linear_grid(ctx, kind, mu, 5000, 9.2, 0.3, 41)
    Eo, vo = oracle.linear_grid(kind, mu, 5000, 9.2, 0.3, 41)
    assert np.allclose(E, Eo, rtol=0, atol=1e-13)
    fin = np.isfinite(vo)
    assert np.array_equal(np.isfinite(v), fin)
    if kind != 5:
        assert fin.sum() >= len(vo) - 2 and np.abs(v - vo)[fin].max() < 1e-9 * np.abs(vo[fin]).max()
