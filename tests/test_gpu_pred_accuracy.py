"""The error of a prediction's variances is that of a forward substitution which
subtracts 64 columns of the factor at a time, in each of the three solves (a few points,
16 and 64 columns a workgroup).

Both errors are against the substitution in 80-bit arithmetic with the device's own
factor and cross covariance.  The substitution is restated operation by operation (fused
multiply-adds, a 64-column product summed before it is subtracted, the inverse of each
diagonal block, the squares summed by 64 lanes), so its error is the device's but for the
order inside a block; one sum over all columns in a row is 2.3 to 4 times further off at
these sizes.  The line lies between the two."""

import numpy as np
import pytest

import gplite_amd as G

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _fma(a, b, c):
    """a b + c in float64, rounded once (up to the products' last bits in 80)."""
    return (a.astype(LD) * b + c).astype(float)


def _blocked_variance(L, b, kd):
    n, m = b.shape
    y = np.zeros((-(-n // 64) * 64, m))
    y[:n] = b
    for i in range(0, n, 64):
        e = min(i + 64, n)
        inv = _exact(L[i:e, i:e], np.eye(e - i)).astype(float)
        x = np.zeros((e - i, m))
        for k in range(e - i):
            x = _fma(inv[:, k, None], y[i + k], x)
        y[i:e] = x
        if e < n:
            s = np.zeros((n - e, m))
            for k in range(i, e):
                s = _fma(L[e:, k, None], y[k], s)
            y[e:n] -= s
    s = np.zeros((64, m))
    for i in range(0, n, 64):
        s = _fma(y[i:i + 64], y[i:i + 64], s)
    for o in (32, 16, 8, 4, 2, 1):
        s = s[:o] + s[o:2 * o]
    return kd - s[0]


def _exact(L, b):
    L, y = L.astype(LD), b.astype(LD)
    for k in range(len(L)):
        y[k] /= L[k, k]
        y[k + 1:] -= L[k + 1:, k, None] * y[k]
    return y


@pytest.mark.parametrize("n,m", [(640, 48), (640, 200), (640, 4800), (1500, 40), (1500, 100), (1500, 2100)])
def test_variance_error(n, m):
    sigma, use = 0.125, 40  # a power of two: the scaling between the two factors is exact
    dev, ref = 0.0, 0.0
    for seed in range(3):
        r = np.random.default_rng(seed)
        x, xt = r.uniform(-1, 1, (n, 3)), r.uniform(-1, 1, (m, 3))
        g = G.gp_fit(G.gp_init(G.cf_matern52(lscale=0.7), G.lik_gaussian(sigma=sigma)), x, np.sin(3 * x.sum(1)))
        var = G.gp_pred(g, xt, var=True)["var"][:use]
        Lb = np.tril(g.fit.C_chol) / sigma
        kt = G.eval_cf(g.cfs, x, xt[:use]) / sigma
        kd = G.eval_cf(g.cfs, xt[:use], xt[:use], diag_only=True)
        want = kd.astype(LD) - (_exact(Lb, kt) ** 2).sum(0)
        dev += float(((var - want) ** 2).sum())
        ref += float(((_blocked_variance(Lb, kt, kd) - want) ** 2).sum())
    print(f"n={n} m={m}: {np.sqrt(dev / ref):.2f}", flush=True)
    assert np.sqrt(dev / ref) <= 1.5
