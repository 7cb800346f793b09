"""L^-1 without scratch, by doubling (its products lie transposed above the
diagonal), through the posterior variances of EP: one 64-row block, a short last
block at one and at several levels, whole powers of two, and the sizes where the
leading half runs beside the factor."""

import numpy as np
import pytest

import gplite_amd as G

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("n", [50, 100, 190, 256, 330, 700, 1090, 2100])
def test_ep_variances_are_those_of_the_final_sites(n):
    r = np.random.default_rng(n)
    x = r.uniform(-1, 1, (n, 2))
    y = (r.uniform(size=n) < 1 / (1 + np.exp(-2 * np.sin(3 * x.sum(1))))).astype(float)
    ls = 0.5
    f = G.gp_fit(G.gp_init(G.cf_sexp(lscale=ls), G.lik_bernoulli("probit"), approx=G.approx_ep()), x, y).fit
    V = f.V
    K = np.exp(-0.5 * ((x[:, None] - x[None]) ** 2).sum(-1) / ls ** 2) + 1e-6 * np.eye(n)
    s = 1 / np.sqrt(V)
    B = np.eye(n) + s[:, None] * K * s
    # fvar = V (1 - diag B^-1); both inverses carry errors of about n eps cond(B), cond(B) <= 1 + n / min V
    tol = 4 * n * EPS * (1 + n / V.min()) * V
    assert np.all(np.abs(f.fvar - V * (1 - np.diag(np.linalg.inv(B)))) <= tol)
