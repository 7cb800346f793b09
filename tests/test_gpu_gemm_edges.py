"""The FP64 product kernel through the calls that use it, at sizes on both sides
of its tile choice: 64x64 output tiles below and above 128 (16- and 32-wide
waves), and 128x128 ones above 600 with a long inner dimension (64-wide)."""

import numpy as np
import pytest
import scipy.linalg as sla

import gplite_amd as G

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,m", [(130, 1), (960, 70), (1030, 577), (1450, 2049), (4500, 1100)])
def test_prediction_and_gradient_at_tile_edges(n, m):
    r = np.random.default_rng(n)
    x, xt = r.uniform(-1, 1, (n, 3)), r.uniform(-1, 1, (m, 3))
    y = np.sin(3 * x.sum(1)) + 0.3 * r.standard_normal(n)
    ls, sig = 0.4, 0.3

    def kern(a, b):
        s = sum((a[:, k, None] - b[None, :, k]) ** 2 for k in range(3))
        return np.exp(-0.5 * s / ls ** 2), s

    K, s = kern(x, x)
    C = K + (sig ** 2 + 1e-6) * np.eye(n)
    Lc = sla.cholesky(C, lower=True)
    a = sla.cho_solve((Lc, True), y)
    Ci = sla.cho_solve((Lc, True), np.eye(n))
    P = Ci - np.outer(a, a)
    grad = np.array([0.5 * np.sum(P * K * s) / ls ** 2, np.sum(P * K), sig ** 2 * np.trace(P)])
    Kt, _ = kern(xt, x)
    v = sla.solve_triangular(Lc, Kt.T, lower=True)
    mean, var = Kt @ a, 1.0 - np.sum(v * v, axis=0)
    # both sides carry errors of about n eps cond(C), cond(C) <= (n + sig^2) / sig^2
    tol = 4 * n * EPS * (n + sig ** 2) / sig ** 2
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=ls), G.lik_gaussian(sigma=sig)), x, y, want_grad=True)
    gr = G.gp_energy_grad(g, include_prior=False)
    assert np.abs(gr - grad).max() <= tol * np.abs(grad).max()
    f = G.gp_fit(G.gp_init(G.cf_sexp(lscale=ls), G.lik_gaussian(sigma=sig)), x, y)
    for h in (g, f):  # through L^-1, and by substitution
        p = G.gp_pred(h, xt, var=True)
        assert np.abs(p["mean"] - mean).max() <= tol * np.abs(mean).max()
        assert np.abs(p["var"] - var).max() <= tol
