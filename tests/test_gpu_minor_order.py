"""The failing minor is the lowest one although the workgroups that factor the later
diagonal blocks of a panel, which hold NaN by then, report theirs in no fixed order:
beside the other streams' products of a large factorization, many times over."""

import numpy as np
import pytest

import gplite_amd as G
from gplite_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(256, 1), (256, 70), (2304, 1), (2304, 512), (2304, 1100)])
def test_lowest_minor(n, k):
    # as in the panel's edge tests: every pivot is 0.9 but that of row k, and all that follow are NaN
    x = 10.0 * np.arange(n)
    x[k] = x[0]
    gp = G.gp_init(G.cf_sexp(lscale=0.1), G.lik_gaussian(sigma=1.0))
    for _ in range(20):
        with pytest.raises(L.GplError) as e:
            G.gp_fit(gp, x, np.zeros(n), jitter=-1.1)
        assert e.value.code == L.GPL_ERR_NOT_PD
        assert e.value.minor == k + 1
