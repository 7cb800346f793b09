"""A predicted point's mean and variance are the same bits whatever the number of
points asked for with it: the solves for a few points, 16 columns and 64 columns at
a time, on one and on many row blocks of the factor."""

import numpy as np
import pytest

import gplite_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 64, 65, 130, 640, 1000, 2500])
def test_any_number_of_points(n):
    r = np.random.default_rng(n)
    x, xt = r.uniform(-1, 1, (n, 3)), r.uniform(-1, 1, (1500, 3))
    y = np.sin(3 * x.sum(1)) + 0.1 * r.standard_normal(n)
    g = G.gp_fit(G.gp_init(G.cf_matern52(lscale=0.5), G.lik_gaussian(sigma=0.2)), x, y)
    want = G.gp_pred(g, xt, var=True)
    for m in (1, 2, 3, 8, 17, 32, 63, 64, 65, 200):
        for _ in range(2):
            p = G.gp_pred(g, xt[:m], var=True)
            np.testing.assert_array_equal(p["mean"], want["mean"][:m])
            np.testing.assert_array_equal(p["var"], want["var"][:m])
