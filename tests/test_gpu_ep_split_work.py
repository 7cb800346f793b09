"""An EP sweep whose sites split (some pseudo-variance <= 0) runs the split's products
only: no factor of the full B, inverse or product with K beside them.  The first sweep of
these fits, from the prior, is the one whose sites do not split."""

import numpy as np
import pytest

import gplite_amd as G
from gplite_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [100, 700])
def test_no_full_factor_in_split_sweeps(n):
    r = np.random.default_rng(3)
    x = np.sort(r.uniform(-3, 3, n))
    mu = 1 / (1 + np.exp(-3.0 - 0.5 * np.sin(x)))
    y = r.binomial(10, r.beta(mu / 0.2, (1 - mu) / 0.2)).astype(float)
    y[::10] = 0.0
    gp = G.gp_init(G.cf_sexp(lscale=1.0, magn=1.0), G.lik_betabinom(phi=0.2), approx=G.approx_ep())
    L.profile(enable=True, reset=True)
    try:
        g = G.gp_fit(gp, x, y, trials=np.full(n, 10.0))
        prof = L.profile()
    finally:
        L.profile(enable=False, reset=True)
    sweeps = prof["ep_sites"]["launches"]
    full = prof.get("symv", {"launches": 0})["launches"]
    print(f"n={n}: {sweeps} sweeps, {(g.fit.V < 0).sum()} V < 0, {full} with the full factor", flush=True)
    assert sweeps == g.fit.iters > 2
    assert full == 1
