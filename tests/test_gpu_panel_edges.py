"""The single-launch Cholesky panel at the edges of its column blocks, panels and
outer blocks: the factor against the matrix it factors, the carried forward
solve, and the failing minor reported from every position of a panel."""

import numpy as np
import pytest

import gplite_amd as G
from gplite_amd import _lib as L

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _problem(n, seed=0):
    r = np.random.default_rng(seed)
    x = r.uniform(-1, 1, (n, 2))
    y = np.sin(3 * x.sum(1)) + 0.1 * r.standard_normal(n)
    d = ((x[:, None] - x[None]) ** 2).sum(-1)
    C = np.exp(-0.5 * d / 0.3 ** 2) + (1e-6 + 0.01) * np.eye(n)
    return x, y, C


# one column block, two, one panel (256), an outer block (512), each with a row more and less
@pytest.mark.parametrize("n", [64, 65, 128, 192, 193, 255, 256, 257, 320, 448, 511, 512, 513, 576, 769, 1025])
@pytest.mark.parametrize("want_grad", [False, True])
def test_factor_and_solve_at_block_edges(n, want_grad):
    x, y, C = _problem(n)
    g = G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.3), G.lik_gaussian(sigma=0.1)), x, y, want_grad=want_grad)
    Lc = np.tril(g.fit.C_chol)
    # Cholesky's backward error: |L L^T - C|_ij <= (n + 1) eps sqrt(C_ii C_jj) (Higham, 2002, Thm 10.5), and
    # 4 eps for the covariance entries themselves, evaluated in another order here
    assert np.abs(Lc @ Lc.T - C).max() <= (n + 5) * EPS * C.max()
    # the residual of a solve with that factor: 3 (n + 1) eps |L| |L^T| |alpha| (Thm 10.4), and through B = S C S
    a = g.fit.alpha
    bound = 4 * (n + 5) * EPS * (np.abs(Lc) @ (np.abs(Lc).T @ np.abs(a))) + 4 * (n + 5) * EPS * (np.abs(C) @ np.abs(a))
    assert np.all(np.abs(C @ a - y) <= bound + 4 * EPS * np.abs(y))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("k", [1, 63, 64, 65, 130, 255, 256, 300, 511, 512, 600, 767])
def test_failing_minor_is_reported(k, precision):
    # inputs far apart except x_k = x_0: B = (2 + jitter) I plus a 1 at (k, 0), so with jitter -1.1 every pivot
    # is 0.9 but that of row k, 0.9 - 1 / 0.9 < 0
    n = 768
    x = 10.0 * np.arange(n)
    x[k] = x[0]
    with pytest.raises(L.GplError) as e:
        G.gp_fit(G.gp_init(G.cf_sexp(lscale=0.1), G.lik_gaussian(sigma=1.0)), x, np.zeros(n), jitter=-1.1,
                 precision=precision)
    assert e.value.code == L.GPL_ERR_NOT_PD
    assert e.value.minor == k + 1


@pytest.mark.parametrize("n", [576, 960, 2049])
def test_factor_has_the_same_bits_every_time(n):
    # the waves of a panel's workgroups read each other's columns of one LDS block while they factor it
    x, y, _ = _problem(n)
    gp = G.gp_init(G.cf_sexp(lscale=0.3), G.lik_gaussian(sigma=0.1))
    want = None
    for _ in range(150):
        a = G.gp_fit(gp, x, y).fit.alpha
        want = a if want is None else want
        np.testing.assert_array_equal(a, want)
