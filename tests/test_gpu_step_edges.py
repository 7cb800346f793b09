"""The scalars that end a Newton step and an EP sweep, and the state they leave, at
sizes around one workgroup's 1024 threads: the returned evidence is that of the
returned vectors."""

import numpy as np
import pytest
from scipy.special import gammaln, ndtr

import gplite_amd as G
from gplite_amd import _lib as L

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _setup(n, offset):
    r = np.random.default_rng(n)
    x = r.uniform(-1, 1, (n, 2))
    f = np.sin(3 * x.sum(1))
    off = 0.3 * r.standard_normal(n) if offset else None
    K = np.exp(-0.5 * ((x[:, None] - x[None]) ** 2).sum(-1) / 0.5 ** 2) + 1e-6 * np.eye(n)
    return r, x, f, off, K


def _logdet(K, V):
    s = 1 / np.sqrt(V)
    B = np.eye(len(V)) + s[:, None] * K * s
    return np.linalg.slogdet(B)[1], 4 * len(V) * EPS * (1 + len(V) / V.min())


@pytest.mark.parametrize("n", [1, 70, 1023, 1025, 2100])
def test_laplace_evidence(n):
    r, x, f, off, K = _setup(n, True)
    y = r.poisson(np.exp(f + off)).astype(float)
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.5), G.lik_poisson(), approx=G.approx_laplace(maxiter=50, tol=1e-8)), x, y,
                 offset=off).fit
    h = g.fmean + off
    ld, tol = _logdet(K, g.V)
    terms = np.concatenate([y * h - np.exp(h) - gammaln(y + 1), -0.5 * g.fmean * g.alpha, [-0.5 * ld]])
    # the factor's error, and that of K alpha and the sums relative to the sum of absolute terms
    assert abs(g.log_evidence - terms.sum()) <= tol * np.abs(terms).sum() + tol
    assert np.abs(K @ g.alpha - g.fmean).max() <= 4 * n * EPS * np.abs(g.alpha).sum()


@pytest.mark.parametrize("n", [2, 70, 1023, 1025, 2100])
def test_ep_evidence(n):
    r, x, f, _, K = _setup(n, False)
    y = (r.uniform(size=n) < ndtr(f)).astype(float)
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.5), G.lik_bernoulli("probit"), approx=G.approx_ep()), x, y).fit
    gx, gw = np.polynomial.hermite_e.hermegauss(11)
    cm, cv, V, z = g.vector(L.VEC_CAVITY_MEAN), g.vector(L.VEC_CAVITY_VAR), g.V, g.z
    lz = np.log(ndtr((2 * y - 1)[:, None] * (cm[:, None] + np.sqrt(cv)[:, None] * gx)) @ (gw / gw.sum()))
    ld, tol = _logdet(K, V)
    c = cv + V
    terms = np.concatenate([lz + 0.5 * np.log(c) + 0.5 * (cm - z) ** 2 / c - 0.5 * np.log(V), -0.5 * z * g.alpha,
                            [-0.5 * ld]])
    assert abs(g.log_evidence - terms.sum()) <= tol * np.abs(terms).sum() + tol
    assert np.abs(K @ g.alpha - g.fmean).max() <= 4 * n * EPS * np.abs(g.alpha).sum()
