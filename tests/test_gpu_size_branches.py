"""Branches that only size reaches: the substitution of a prediction in more than one
launch (n m > 2^28), and the step-ending kernels at the edges of their workgroups of 256
threads (up to 256 points end without partial sums) and past 128 of them (n > 32768:
every thread takes more than one point)."""

import numpy as np
import pytest
from scipy.special import gammaln

import gplite_amd as G
from tests import test_gpu_step_edges as steps

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,m", [(4090, 65601), (2500, 210001)])
def test_substitution_in_several_launches(n, m):
    r = np.random.default_rng(n)
    x = r.uniform(-1, 1, (n, 2))
    g = G.gp_fit(G.gp_init(G.cf_matern52(lscale=0.5), G.lik_gaussian(sigma=0.2)), x, np.sin(3 * x.sum(1)))
    xt = r.uniform(-1, 1, (m, 2))
    p = G.gp_pred(g, xt, var=True)
    # the starts, ends and halves of the launches, and the last points
    for a in (0, 32700, 32832 - 30, 65536 - 30, m // 2 // 64 * 64 - 30, m // 2 - 10, m - 200):
        q = G.gp_pred(g, xt[a:a + 200], var=True)
        np.testing.assert_array_equal(p["mean"][a:a + 200], q["mean"])
        np.testing.assert_array_equal(p["var"][a:a + 200], q["var"])


@pytest.mark.parametrize("n", [255, 256, 257, 512, 513])
def test_evidence_at_workgroup_edges(n):
    steps.test_laplace_evidence(n)
    steps.test_ep_evidence(n)


N_LARGE = 33001


def test_gaussian_evidence_past_128_workgroups():
    # inputs far apart: K = I, so every result has a closed form
    n, s2, jit = N_LARGE, 0.25, 1e-6
    y = np.random.default_rng(1).standard_normal(n)
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.1), G.lik_gaussian(sigma=0.5)), 10.0 * np.arange(n), y).fit
    c = 1.0 + jit + s2
    terms = np.concatenate([-0.5 * y * y / c, np.full(n, -0.5 * np.log(2 * np.pi * c))])
    # a handful of roundings a point, and n in the sums
    np.testing.assert_allclose(g.alpha, y / c, rtol=16 * EPS)
    np.testing.assert_allclose(g.fmean, y * (1 + jit) / c, rtol=32 * EPS)
    assert abs(g.log_evidence - terms.sum()) <= (n + 64) * EPS * np.abs(terms).sum()


def test_laplace_evidence_past_128_workgroups():
    n, jit = N_LARGE, 1e-6
    r = np.random.default_rng(2)
    y = r.poisson(np.exp(r.standard_normal(n))).astype(float)
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.1), G.lik_poisson(), approx=G.approx_laplace(maxiter=50, tol=1e-8)),
                 10.0 * np.arange(n), y).fit
    f, V = g.fmean, g.V
    terms = np.concatenate([y * f - np.exp(f) - gammaln(y + 1), -0.5 * f * g.alpha, -0.5 * np.log1p((1 + jit) / V)])
    assert abs(g.log_evidence - terms.sum()) <= (n + 64) * EPS * np.abs(terms).sum()
    np.testing.assert_allclose(f, (1 + jit) * g.alpha, rtol=32 * EPS)
    # the mode: d log p = alpha at every point, to the last Newton step's change
    np.testing.assert_allclose(y - np.exp(f), g.alpha, atol=1e-7)
