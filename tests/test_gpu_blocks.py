"""Device blocks that freed models leave for the next one: fits into reused blocks
give what fits into fresh ones give, for every kind of model, and unused blocks go
back to the device."""

import gc

import numpy as np
import pytest
import torch

import gplite_amd as G

pytestmark = pytest.mark.gpu


def _fits(kind, n):
    r = np.random.default_rng(n)
    x = r.uniform(-1, 1, (n, 3))
    f = np.sin(3 * x.sum(1))
    cf = G.cf_matern52(lscale=0.6)
    if kind == "laplace":
        return lambda: G.gp_fit(G.gp_init(cf, G.lik_poisson()), x, r0.poisson(np.exp(f)).astype(float))
    if kind == "ep":
        return lambda: G.gp_fit(G.gp_init(cf, G.lik_bernoulli("probit"), approx=G.approx_ep()), x,
                                (r0.uniform(size=n) < 0.5 + 0.4 * f).astype(float))
    y = f + 0.1 * r.standard_normal(n)
    if kind == "fitc":
        return lambda: G.gp_fit(G.gp_init(cf, G.lik_gaussian(sigma=0.2), method=G.method_fitc(inducing=x[:n // 4])), x, y)
    prec = "mixed" if kind == "mixed" else "fp64"
    return lambda: G.gp_fit(G.gp_init(cf, G.lik_gaussian(sigma=0.2)), x, y, precision=prec, want_grad=kind != "gaussian")


r0 = None


def _run(fit, xt):
    global r0
    r0 = np.random.default_rng(5)
    g = fit()
    p = G.gp_pred(g, xt, var=True)
    return g, np.concatenate([[G.gp_energy(g)], g.fit.alpha, p["mean"], p["var"]])


@pytest.mark.parametrize("kind", ["gaussian", "grad", "mixed", "laplace", "ep", "fitc"])
def test_reused_blocks_give_the_same_results(kind):
    xt = np.random.default_rng(9).uniform(-1, 1, (70, 3))
    fits = [_fits(kind, n) for n in (900, 960, 700)]
    kept = [_run(f, xt) for f in fits]  # alive together: no block is used twice
    ref = [k[1] for k in kept]
    del kept
    gc.collect()
    for _ in range(2):
        for f, want in zip(fits, ref):
            g, got = _run(f, xt)
            del g
            np.testing.assert_array_equal(got, want)


def test_unused_blocks_are_given_back():
    big, small = _fits("grad", 3000), _fits("gaussian", 100)
    xt = np.zeros((1, 3))
    for f in (big, small):
        _run(f, xt)
    gc.collect()
    for _ in range(20):
        _run(small, xt)
    gc.collect()
    free0 = torch.cuda.mem_get_info()[0]
    _run(big, xt)  # about 220 MB
    gc.collect()
    for _ in range(20):
        _run(small, xt)
    gc.collect()
    assert torch.cuda.mem_get_info()[0] >= free0 - (32 << 20)
