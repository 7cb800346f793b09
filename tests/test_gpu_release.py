"""Device blocks that freed models leave: a call gives them back, and the contexts of a
process share one limit of 1/32 of the device's memory."""

import ctypes as C
import gc

import numpy as np
import pytest
import torch

import gplite_amd as G
from gplite_amd import _lib as L
from gplite_amd import api

pytestmark = pytest.mark.gpu

SLACK = 64 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_release_memory():
    r = np.random.default_rng(0)
    x = r.uniform(-1, 1, (3000, 2))
    y = np.sin(3 * x.sum(1)) + 0.1 * r.standard_normal(3000)
    gp = G.gp_init(G.cf_matern52(lscale=0.5), G.lik_gaussian(sigma=0.2))

    def fit():
        return G.gp_energy_grad(G.gp_fit(gp, x, y, want_grad=True))

    G.release_memory()
    small = G.gp_fit(gp, x[:100], y[:100])  # the context and its workspaces exist
    want = fit()
    gc.collect()
    G.release_memory()
    free0 = _free()
    fit()
    gc.collect()
    assert _free() < free0 - (100 << 20)  # three matrices of 72 MB wait for the next fit
    G.release_memory()
    assert _free() >= free0 - SLACK
    np.testing.assert_array_equal(fit(), want)
    del small


def test_contexts_share_the_limit():
    lib = L.lib()
    gc.collect()
    G.release_memory()
    r = np.random.default_rng(1)
    n = 16384  # three matrices of 2.1 GB a model
    x = r.uniform(0, 1, (n, 4))
    y = np.sin(3 * x.sum(1))
    terms, nt, xp, _ = api._program([G.cf_matern52(lscale=0.5)], x)
    lik = api._lik_struct(G.lik_gaussian(sigma=0.3))
    opts = L.Opts()
    lib.gpl_opts_default(C.byref(opts))
    opts.flags = 1
    ctxs, models = [], []
    for _ in range(2):
        c, m, e = L._vp(), L._vp(), C.c_double()
        L.check(lib.gpl_ctx_create(0, C.byref(c)))
        ctxs.append(c)
        L.check(lib.gpl_fit(c, terms, nt, L.dptr(xp), n, xp.shape[1], L.dptr(y), None, None, C.byref(lik), C.byref(opts),
                            C.byref(m), C.byref(e)))
        models.append(m)
    held = sum(lib.gpl_model_bytes(m) for m in models)
    limit = torch.cuda.mem_get_info()[1] // 32
    assert held > limit
    free0 = _free()
    for m in models:
        lib.gpl_model_free(m)
    assert _free() - free0 >= held - limit - SLACK
    for c in ctxs:
        lib.gpl_ctx_destroy(c)
    assert _free() - free0 >= held - SLACK
