"""Predictions of more points than the pinned result block holds (2 m + 1 doubles of
131072) give the bits that the same points give in small predictions: a substitution,
a kept inverse, and a fit with split sites."""

import numpy as np
import pytest

import gplite_amd as G

pytestmark = pytest.mark.gpu


def _model(kind):
    r = np.random.default_rng(3)
    if kind == "split":
        x = np.sort(r.uniform(-3, 3, 100))
        mu = 1 / (1 + np.exp(-3.0 - 0.5 * np.sin(x)))
        y = r.binomial(10, r.beta(mu / 0.2, (1 - mu) / 0.2)).astype(float)
        y[[10, 50, 90]] = 0.0
        return G.gp_fit(G.gp_init(G.cf_sexp(lscale=1.0), G.lik_betabinom(phi=0.2)), x, y, trials=np.full(100, 10.0))
    x = r.uniform(-3, 3, 130)
    y = np.sin(x) + 0.1 * r.standard_normal(130)
    return G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.5), G.lik_gaussian(sigma=0.2)), x, y, want_grad=kind == "inverse")


@pytest.mark.parametrize("kind", ["substitution", "inverse", "split"])
@pytest.mark.parametrize("m", [65535, 65536, 66001])
def test_more_points_than_the_pinned_block(kind, m):
    g = _model(kind)
    xt = np.random.default_rng(m).uniform(-3.5, 3.5, m)
    p = G.gp_pred(g, xt, var=True)
    np.testing.assert_array_equal(G.gp_pred(g, xt)["mean"], p["mean"])
    for a in (0, m // 2, m - 300):
        q = G.gp_pred(g, xt[a:a + 300], var=True)
        np.testing.assert_array_equal(p["mean"][a:a + 300], q["mean"])
        np.testing.assert_array_equal(p["var"][a:a + 300], q["var"])
