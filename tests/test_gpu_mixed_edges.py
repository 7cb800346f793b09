"""The mixed form's FP64 diagonal tiles and panel steps at their edges, single fits
and batches: one to eighteen 64-row blocks, so that the updates run at depths 64,
128, 256 and 512 on one block and on several."""

import numpy as np
import pytest
import scipy.linalg as sla

import gplite_amd as G
from gplite_amd.batch import GPBatch

pytestmark = pytest.mark.gpu

EPS32 = float(np.finfo(np.float32).eps)
SIZES = [50, 64, 100, 190, 256, 300, 513, 640, 1090]


def _problem(n):
    r = np.random.default_rng(n)
    x = r.uniform(-1, 1, (n, 3))
    y = np.sin(3 * x.sum(1)) + 0.5 * r.standard_normal(n)
    C = np.exp(-0.5 * ((x[:, None] - x[None]) ** 2).sum(-1) / 0.6 ** 2) + (0.25 + 1e-6) * np.eye(n)
    Lc = sla.cholesky(C, lower=True)
    a = sla.cho_solve((Lc, True), y)
    e = 0.5 * y @ a + np.log(np.diag(Lc)).sum() + 0.5 * n * np.log(2 * np.pi)
    # the refined solution is good to about 1e-8; the n pivots carry FP32 errors of the off-diagonal blocks
    return x, y, a, e, 4 * n * EPS32


def _gp():
    return G.gp_init(G.cf_sexp(lscale=0.6), G.lik_gaussian(sigma=0.5))


@pytest.mark.parametrize("n", SIZES)
def test_mixed_fit(n):
    x, y, a, e, tol = _problem(n)
    g = G.gp_fit(_gp(), x, y, precision="mixed", want_grad=True)
    assert g.fit.precision_info["precision"] == "mixed"
    assert np.abs(g.fit.alpha - a).max() <= 1e-7 * np.abs(a).max()
    assert abs(G.gp_energy(g, include_prior=False) - e) <= tol


def test_batch_of_all_sizes():
    ps = [_problem(n) for n in SIZES + [513, 64]]
    e, _ = GPBatch([_gp()] * len(ps), [p[0] for p in ps], [p[1] for p in ps]).energy_grad(include_prior=False)
    assert np.all(np.abs(e - [p[3] for p in ps]) <= [p[4] for p in ps])


# the solves of the rows below a diagonal block: none, one and several row blocks, the last one padded or whole
@pytest.mark.parametrize("n", [65, 128, 129, 192, 321, 1025])
@pytest.mark.parametrize("copies", [1, 3])
def test_batched_panel_solve(n, copies):
    x, y, _, e, tol = _problem(n)
    got, _ = GPBatch([_gp()] * copies, [x] * copies, [y] * copies).energy_grad(include_prior=False)
    assert np.all(np.abs(got - e) <= tol)


# 256 row blocks below the diagonal blocks of a launch, and more: one launch with the factor and two
@pytest.mark.parametrize("copies", [127, 128, 129])
def test_batched_step_at_its_line(copies):
    x, y, _, e, tol = _problem(180)
    got, _ = GPBatch([_gp()] * copies, [x] * copies, [y] * copies).energy_grad(include_prior=False)
    assert np.all(np.abs(got - e) <= tol)


# 64x64 tiles of a launch, of one problem and of all, on both sides of the line between the two FP32 products
@pytest.mark.parametrize("n,copies", [(64, 300), (130, 60), (500, 12), (1400, 2), (1500, 2)])
def test_a_problem_alone_and_among_copies(n, copies):
    x, y = _problem(n)[:2]
    one = GPBatch([_gp()], [x], [y]).energy_grad(include_prior=False)
    e, g = GPBatch([_gp()] * copies, [x] * copies, [y] * copies).energy_grad(include_prior=False)
    # the factor and the inverses have one order of sums; alpha is refined to 1e-8 in any
    np.testing.assert_allclose(e, np.full(copies, one[0][0]), rtol=1e-8)
    np.testing.assert_allclose(g, np.tile(one[1][0], (copies, 1)), rtol=0, atol=1e-7 * np.abs(one[1]).max())
