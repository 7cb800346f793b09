"""The native column means and standard deviations are numpy's, bit for bit (they
enter every kernel value), for each remainder of the column groups."""

import numpy as np
import pytest

from gplite_amd import _lib as L


@pytest.mark.parametrize("n,d", [(2, 2), (3, 3), (1000, 7), (4097, 8), (5000, 13), (70000, 16)])
def test_matches_numpy(n, d):
    x = np.random.default_rng(n + d).normal(size=(n, d)) * 3 + 1
    m, s = np.empty(d), np.empty(d)
    L.lib().gpl_col_scales(L.dptr(x), n, d, L.dptr(m), L.dptr(s))
    np.testing.assert_array_equal(m, x.mean(axis=0))
    np.testing.assert_array_equal(s, x.std(axis=0, ddof=1))
