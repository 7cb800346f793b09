"""FITC at the edges of its kernels: the passes over A = Lz^-1 K_zx at each number
of rows a wave holds (up to 128, 256, 512, 1024, and the split form above), one and
several partial Gram products, one and two blocks of columns, short last parts."""

import numpy as np
import pytest
import scipy.linalg as sla

import gplite_amd as G

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,m", [(40, 1), (65, 64), (700, 65), (1000, 200), (3000, 257), (5001, 513), (1500, 1100),
                                 (33000, 1000)])
def test_fitc_gaussian_fit_and_prediction(n, m):
    r = np.random.default_rng(n + m)
    d, ls, sig = 6, 0.8, 0.2
    x, xt = r.uniform(-1, 1, (n, d)), r.uniform(-1, 1, (90, d))
    z = x[r.permutation(n)[:m]]
    y = np.sin(x.sum(1)) + sig * r.standard_normal(n)

    def kern(a, b):
        return np.exp(-0.5 * (np.sum(a * a, 1)[:, None] + np.sum(b * b, 1) - 2 * a @ b.T) / ls ** 2)

    jit = 1e-6
    Kz = kern(z, z) + jit * np.eye(m)
    Lz = sla.cholesky(Kz, lower=True)
    A = sla.solve_triangular(Lz, kern(z, x), lower=True)
    S = 1 + jit - np.sum(A * A, 0) + sig ** 2
    Gm = np.eye(m) + (A / S) @ A.T
    Lc = sla.cholesky(Gm, lower=True)
    w0 = sla.cho_solve((Lc, True), A @ (y / S))
    alpha = y / S - (A.T @ w0) / S
    w = A @ alpha
    ev = -0.5 * (y @ alpha) - 0.5 * (np.log(S).sum() + 2 * np.log(np.diag(Lc)).sum()) - 0.5 * n * np.log(2 * np.pi)
    At = sla.solve_triangular(Lz, kern(z, xt), lower=True)
    v = sla.solve_triangular(Lc, At, lower=True)
    mean, var = At.T @ w, 1 - np.sum(At * At, 0) + np.sum(v * v, 0)
    # both sides carry the errors of A (about m eps cond Kz) through G's solve (cond G); |At| <= 1
    cz, cg = np.linalg.cond(Kz), np.linalg.cond(Gm)
    tol = 8 * max(m, 64) * EPS * (cz + cg)
    f = G.gp_fit(G.gp_init(G.cf_sexp(lscale=ls), G.lik_gaussian(sigma=sig), method=G.method_fitc(inducing=z)), x, y)
    p = G.gp_pred(f, xt, var=True)
    assert np.abs(p["mean"] - mean).max() <= tol * max(1.0, np.linalg.norm(w))
    assert np.abs(p["var"] - var).max() <= tol
    assert abs(f.fit.log_evidence - ev) <= tol * (abs(ev) + n)
