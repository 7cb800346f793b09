"""Performance cases of the dense GP core: what a program that uses gplite_amd has it do.

A case is a dict of plain values; its "kind" picks one of the paths below.  `prepare` makes what such a
program holds before the call (data, the model object, a fitted model to predict from, a batch handle),
`run` is one pass through the public entry points, `work` counts the bytes and operations that a pass
cannot do without, and `exact` restates the result in plain FP64 on the CPU.

kinds
  regress   gp_fit with the Gaussian likelihood, then energy, optionally the gradient and a prediction
  latent    gp_fit with a non-Gaussian likelihood (Laplace or EP)
  predict   gp_pred (mean and variance) from a fitted model that is kept
  batch     energy and gradient of many regressions in one device pass (GPBatch)
  fitc      gp_fit with method_fitc and given inducing inputs, then a prediction

Data are smooth random functions (a few random cosines) of uniform or normal inputs plus noise, the
regime that the benchmark's and the tests' workloads have.
"""

import math

import numpy as np
import torch

import gplite_amd as G
from gplite_amd.batch import GPBatch

JITTER = 1e-6  # gp_fit's default


def listed():
    return [
        # A script's first contact: 200 points in one dimension, fit, evidence and a plotting grid with
        # variances.  Latency: allocations, launches and host work count, not arithmetic.
        dict(name="regress_small", kind="regress", n=200, d=1, cf="sexp", ard=False, precision="fp64", grad=False, m=300),
        # One step of hyperparameter optimisation on an ordinary table, a sum of kernels (the generic
        # gradient kernel), a size that is no multiple of any tile.
        dict(name="regress_grad_mid", kind="regress", n=1507, d=3, cf="sexp+lin", ard=True, precision="fp64", grad=True, m=0),
        # The benchmark's regression, energy and gradient in plain FP64.
        dict(name="regress_grad_large", kind="regress", n=8192, d=8, cf="matern52", ard=True, precision="fp64", grad=True, m=0),
        # The same in the mixed-precision form.
        dict(name="regress_grad_large_mixed", kind="regress", n=8192, d=8, cf="matern52", ard=True, precision="mixed", grad=True, m=0),
        # Many small independent regressions of uneven size (folds, per-group models), one pass.
        dict(name="batch_ragged", kind="batch", problems=128, nmin=64, nmax=2048, d=8, ard=False, restarts=False),
        # The benchmark's headline form: 16 hyperparameter restarts of one regression, one pass.
        dict(name="batch_restarts", kind="batch", problems=16, nmin=8192, nmax=8192, d=8, ard=True, restarts=True),
        # The benchmark's classification, Laplace to a tight mode tolerance.
        dict(name="laplace_class", kind="latent", n=4096, d=4, lik="bernoulli_logit", approx="laplace", tol=1e-8),
        # Count regression on a small table with exposures, default tolerance.
        dict(name="laplace_counts_small", kind="latent", n=500, d=2, lik="poisson", approx="laplace", tol=1e-4),
        # Probit classification by EP: a factor and the posterior variances in every sweep.
        dict(name="ep_class", kind="latent", n=1200, d=3, lik="bernoulli_probit", approx="ep", tol=1e-4),
        # Serving: a request of 1000 points with variances on a resident model.
        dict(name="predict_serving", kind="predict", n=4096, d=6, m=1000),
        # Serving's smallest request: one point on a small model.
        dict(name="predict_one", kind="predict", n=640, d=3, m=1),
        # Sparse regression at the size where the dense form ends.
        dict(name="fitc_large", kind="fitc", n=131072, d=8, m=1024, mt=4096),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["regress", "regress_grad", "regress_grad", "batch_ragged", "batch_restarts", "latent", "ep", "predict", "fitc"])
    if kind == "regress":
        d = rng.randint(1, 4)
        return dict(kind="regress", n=_logu(rng, 32, 1200), d=d, cf=rng.choice(["sexp", "matern52"]), ard=rng.random() < 0.5,
                    precision="fp64", grad=False, m=_logu(rng, 1, 600))
    if kind == "regress_grad":
        cf = rng.choice(["matern52", "matern52", "sexp+lin"])
        return dict(kind="regress", n=_logu(rng, 600, 8192), d=rng.randint(3, 8), cf=cf, ard=True,
                    precision=rng.choice(["fp64", "fp64", "mixed"]), grad=True, m=0)
    if kind == "batch_ragged":
        return dict(kind="batch", problems=_logu(rng, 8, 128), nmin=64, nmax=_logu(rng, 256, 2048), d=rng.randint(3, 8), ard=False, restarts=False)
    if kind == "batch_restarts":
        n = _logu(rng, 1000, 4096)
        return dict(kind="batch", problems=rng.randint(4, 12), nmin=n, nmax=n, d=rng.randint(4, 8), ard=True, restarts=True)
    if kind == "latent":
        lik = rng.choice(["bernoulli_logit", "bernoulli_probit", "poisson"])
        return dict(kind="latent", n=_logu(rng, 200, 4096), d=rng.randint(2, 4), lik=lik, approx="laplace", tol=rng.choice([1e-4, 1e-8]))
    if kind == "ep":
        return dict(kind="latent", n=_logu(rng, 150, 1500), d=rng.randint(2, 4), lik="bernoulli_probit", approx="ep", tol=1e-4)
    if kind == "predict":
        return dict(kind="predict", n=_logu(rng, 300, 4096), d=rng.randint(2, 6), m=_logu(rng, 1, 4096))
    return dict(kind="fitc", n=_logu(rng, 5000, 131072), d=rng.randint(6, 8), m=_logu(rng, 100, 1024), mt=_logu(rng, 100, 4096))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _smooth(x, r, terms=16):
    """A random smooth function of the rows of x with standard deviation near 1."""
    w = r.standard_normal((x.shape[1], terms)) * (2.0 / math.sqrt(x.shape[1]))
    b = r.uniform(0, 2 * math.pi, terms)
    return np.cos(x @ w + b) @ (r.standard_normal(terms) * math.sqrt(2.0 / terms))


def _lscale(case, r, lo=0.3, hi=1.0):
    """Length-scales that grow with the dimension, as fitted ones do."""
    g = math.sqrt(max(case["d"], 2) / 2.0)
    return r.uniform(lo, hi, case["d"]) * g if case.get("ard") else float(r.uniform(lo, hi)) * g


def _cfs(case, ls):
    if case["cf"] == "sexp":
        return [G.cf_sexp(lscale=ls, magn=1.0)]
    if case["cf"] == "matern52":
        return [G.cf_matern52(lscale=ls, magn=1.0)]
    return [G.cf_sexp(lscale=ls, magn=1.0), G.cf_lin(magn=0.5)]


def _regress_inputs(case, seed):
    r = np.random.default_rng(seed)
    x = r.uniform(-1, 1, (case["n"], case["d"]))
    sigma = 0.1 if case["n"] < 4096 else 0.05
    y = _smooth(x, r) + sigma * r.standard_normal(case["n"])
    ls = _lscale(case, r)
    xt = r.uniform(-1, 1, (max(case["m"], 1), case["d"]))
    return x, y, ls, sigma, xt


def _latent_inputs(case, seed):
    r = np.random.default_rng(seed)
    n = case["n"]
    x = r.standard_normal((n, case["d"]))
    f = 1.5 * _smooth(x, r)
    if case["lik"] == "poisson":
        off = np.log(r.uniform(0.5, 3.0, n))
        y = r.poisson(np.exp(0.7 * f + off)).astype(float)
    else:
        off = None
        y = (r.uniform(size=n) < 1 / (1 + np.exp(-f))).astype(float)
    ls, magn = float(r.uniform(0.7, 1.1)) * math.sqrt(case["d"] / 2.0), 1.5
    return x, y, off, ls, magn


def _lik(name):
    return {"poisson": G.lik_poisson, "bernoulli_logit": lambda: G.lik_bernoulli("logit"),
            "bernoulli_probit": lambda: G.lik_bernoulli("probit")}[name]()


def _predict_inputs(case, seed):
    return _regress_inputs(dict(case, cf="matern52", ard=True), seed)


def _batch_inputs(case, seed):
    r = np.random.default_rng(seed)
    k, d = case["problems"], case["d"]
    xs, ys, lss, sigma = [], [], [], 0.05 if case["restarts"] else 0.1
    if case["restarts"]:
        x = r.uniform(0, 1, (case["nmin"], d))
        y = _smooth(x, r) + sigma * r.standard_normal(case["nmin"])
        base = r.uniform(0.3, 1.0, d)
        for _ in range(k):
            xs.append(x)
            ys.append(y)
            lss.append(base * np.exp(0.2 * r.standard_normal(d)))
    else:
        for i in range(k):
            # sizes spread evenly over the logarithm, so that every seed has the same work
            n = int(round(math.exp(math.log(case["nmin"]) + (math.log(case["nmax"]) - math.log(case["nmin"])) * (i + 0.5) / k)))
            di = 1 + i % d
            x = r.uniform(-2, 2, (n, di))
            xs.append(x)
            ys.append(np.sin(x.sum(1)) + sigma * r.standard_normal(n))
            lss.append(float(r.uniform(0.3, 1.5)))
    return xs, ys, lss, sigma


def _fitc_inputs(case, seed):
    r = np.random.default_rng(seed)
    x = r.uniform(0, 1, (case["n"], case["d"]))
    y = _smooth(x, r) + 0.1 * r.standard_normal(case["n"])
    z = x[r.choice(case["n"], case["m"], replace=False)]
    ls = r.uniform(0.2, 0.6, case["d"])  # short enough that Kz is well conditioned
    xt = r.uniform(0, 1, (case["mt"], case["d"]))
    return x, y, z, ls, xt


def prepare(case, seed):
    k = case["kind"]
    G.require_device()
    if k == "regress":
        x, y, ls, sigma, xt = _regress_inputs(case, seed)
        return dict(case=case, gp=G.gp_init(_cfs(case, ls), G.lik_gaussian(sigma=sigma)), x=x, y=y, xt=xt)
    if k == "latent":
        x, y, off, ls, magn = _latent_inputs(case, seed)
        approx = G.approx_ep() if case["approx"] == "ep" else G.approx_laplace(maxiter=50, tol=case["tol"])
        return dict(case=case, gp=G.gp_init(G.cf_sexp(lscale=ls, magn=magn), _lik(case["lik"]), approx=approx), x=x, y=y, off=off)
    if k == "predict":
        x, y, ls, sigma, xt = _predict_inputs(case, seed)
        gf = G.gp_fit(G.gp_init(G.cf_matern52(lscale=ls, magn=1.0), G.lik_gaussian(sigma=sigma)), x, y)
        G.gp_pred(gf, xt[:1], var=True)  # a served model has predicted before
        return dict(case=case, gf=gf, xt=xt)
    if k == "batch":
        xs, ys, lss, sigma = _batch_inputs(case, seed)
        gps = [G.gp_init(G.cf_matern52(lscale=ls, magn=1.0), G.lik_gaussian(sigma=sigma)) for ls in lss]
        b = GPBatch(gps, xs, ys, refine_iters=3 if case["restarts"] else 6)
        if case["restarts"]:  # the benchmark's persisted choice for one large size
            b.load_tuning([dict(n=-(-case["nmin"] // 64) * 64, tile=128, panel=512)])
        return dict(case=case, b=b)
    x, y, z, ls, xt = _fitc_inputs(case, seed)
    return dict(case=case, gp=G.gp_init(G.cf_matern52(lscale=ls, magn=1.0), G.lik_gaussian(sigma=0.1), method=G.method_fitc(inducing=z)),
                x=x, y=y, xt=xt)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "regress":
        gf = G.gp_fit(s["gp"], s["x"], s["y"], precision=case["precision"], want_grad=case["grad"])
        out = {"energy": G.gp_energy(gf, include_prior=False), "alpha": gf.fit.alpha}
        if case["grad"]:
            out["grad"] = G.gp_energy_grad(gf, include_prior=False)
        if case["m"]:
            out["pred"] = G.gp_pred(gf, s["xt"], var=True)
        return out
    if k == "latent":
        gf = G.gp_fit(s["gp"], s["x"], s["y"], offset=s["off"])
        out = {"energy": G.gp_energy(gf, include_prior=False), "fmean": gf.fit.fmean, "alpha": gf.fit.alpha}
        if case["approx"] == "ep":
            out["fvar"] = gf.fit.fvar
        return out
    if k == "predict":
        return G.gp_pred(s["gf"], s["xt"], var=True)
    if k == "batch":
        e, g = s["b"].energy_grad(include_prior=False)
        return {"energy": e, "grad": g}
    gf = G.gp_fit(s["gp"], s["x"], s["y"])
    return {"energy": G.gp_energy(gf, include_prior=False), "fmean": gf.fit.fmean, "pred": G.gp_pred(gf, s["xt"], var=True)}


# ---------------------------------------------------------------------------
# work that a pass cannot do without
# ---------------------------------------------------------------------------

def _chol(n):
    return n ** 3 / 3.0


def work(case):
    k = case["kind"]
    if k == "regress":
        n, d, m = case["n"], case["d"], case["m"]
        fl = _chol(n) * (3 if case["grad"] else 1) + 4.0 * n * n + (1.0 * n * n * m + 2.0 * n * m if m else 0)
        return {"bytes": 8.0 * (n * (d + 2) + m * (d + 2)), "flops": fl}
    if k == "latent":
        n = case["n"]
        # a handful of Newton steps; an EP sweep also needs diag(B^-1).  Counted at the usual number of passes.
        if case["approx"] == "ep":
            return {"bytes": 8.0 * n * (case["d"] + 5), "flops": 10 * (2 * _chol(n) + 4.0 * n * n)}
        return {"bytes": 8.0 * n * (case["d"] + 4), "flops": (7 if case["tol"] < 1e-6 else 5) * (_chol(n) + 4.0 * n * n)}
    if k == "predict":
        n, m = case["n"], case["m"]
        return {"bytes": 8.0 * (n * n / 2 + n * (case["d"] + 1) + m * (case["d"] + 2)), "flops": 1.0 * n * n * m + 2.0 * n * m}
    if k == "batch":
        ns = [math.exp(math.log(case["nmin"]) + (math.log(case["nmax"]) - math.log(case["nmin"])) * (i + 0.5) / case["problems"])
              for i in range(case["problems"])]
        return {"bytes": 8.0 * sum(n * (case["d"] + 1) for n in ns), "flops": sum(n ** 3 + 4 * n * n for n in ns)}
    n, m, mt = case["n"], case["m"], case["mt"]
    # K_zx S^-1 K_xz (symmetric) and Lz^-1 K_zx (triangular), m x m factors, the prediction
    return {"bytes": 8.0 * (n * (case["d"] + 2) + mt * (case["d"] + 2)), "flops": 2.0 * n * m * m + 4 * _chol(m) + 2.0 * m * m * mt}


# ---------------------------------------------------------------------------
# the same results in plain FP64
# ---------------------------------------------------------------------------

def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64)


def _sq(a, b, ls):
    """sum_k (a_ik - b_jk)^2 / l_k^2 by differences."""
    a, b = _t(a), _t(b)
    ls = np.broadcast_to(np.asarray(ls, float), (a.shape[1],))
    s = torch.zeros(a.shape[0], b.shape[0], dtype=torch.float64)
    for k in range(a.shape[1]):
        df = (a[:, k, None] - b[None, :, k]) / float(ls[k])
        s.addcmul_(df, df)
    return s


def _k_sexp(s, magn=1.0):
    return magn ** 2 * torch.exp(-0.5 * s)


def _k_m52(s):
    u = torch.sqrt(5.0 * s)
    return (1 + u + u * u / 3) * torch.exp(-u)


def _dk_m52(s):
    """dK / d s."""
    u = torch.sqrt(5.0 * s)
    return -(5.0 / 6.0) * (1 + u) * torch.exp(-u)


def _kern(case, a, b, ls):
    s = _sq(a, b, ls)
    if case["cf"] == "matern52":
        return _k_m52(s), s
    K = _k_sexp(s)
    if case["cf"] == "sexp+lin":
        K = K + 0.25 * _t(a) @ _t(b).T
    return K, s


def _kdiag(case, xt):
    d = torch.ones(xt.shape[0], dtype=torch.float64)
    return d + 0.25 * (_t(xt) ** 2).sum(1) if case["cf"] == "sexp+lin" else d


def _gauss_exact(case, x, y, ls, sigma, grad, xt=None):
    n = x.shape[0]
    K, s = _kern(case, x, x, ls)
    y = _t(y)
    C = K.clone()
    C.diagonal().add_(JITTER + sigma ** 2)
    L = torch.linalg.cholesky(C)
    del C
    a = torch.cholesky_solve(y[:, None], L)[:, 0]
    out = {"energy": float(0.5 * y @ a + torch.log(L.diagonal()).sum() + 0.5 * n * math.log(2 * math.pi)), "alpha": a.numpy()}
    if grad:
        P = torch.cholesky_inverse(L)
        P.addr_(a, a, alpha=-1.0)  # dE/dtheta = 1/2 tr(P dC/dtheta)
        g = []
        E = _dk_m52(s) if case["cf"] == "matern52" else -0.5 * _k_sexp(s)
        E *= P
        lsv = np.atleast_1d(np.asarray(ls, float))
        if lsv.size == 1:
            g.append(0.5 * float((E * s).sum()) * -2.0)
        else:
            xx = _t(x)
            for k in range(x.shape[1]):
                df = (xx[:, k, None] - xx[None, :, k]) / float(lsv[k])
                g.append(0.5 * -2.0 * float((E * df * df).sum()))
        del E
        if case["cf"] == "sexp+lin":
            Kl = 0.25 * _t(x) @ _t(x).T
            g.append(float((P * (K - Kl)).sum()))
            g.append(float((P * Kl).sum()))
        else:
            g.append(float((P * K).sum()))
        g.append(sigma ** 2 * float(P.diagonal().sum()))
        out["grad"] = np.array(g)
    if xt is not None:
        Kt, _ = _kern(case, xt, x, ls)
        v = torch.linalg.solve_triangular(L, Kt.T.contiguous(), upper=False)
        out["pred"] = {"mean": (Kt @ a).numpy(), "var": (_kdiag(case, xt) - (v * v).sum(0)).numpy()}
    return out


def _ndtr(f):
    return 0.5 * torch.erfc(-f / math.sqrt(2.0))


def _loglik(lik, f, y):
    if lik == "poisson":
        return y * f - torch.exp(f) - torch.lgamma(y + 1)
    sgn = 2 * y - 1
    if lik == "bernoulli_logit":
        return -torch.nn.functional.softplus(-sgn * f)
    return torch.log(_ndtr(sgn * f))


def _dloglik(lik, f, y):
    if lik == "poisson":
        return y - torch.exp(f)
    if lik == "bernoulli_logit":
        return y - torch.sigmoid(f)
    sgn = 2 * y - 1
    return sgn * torch.exp(-0.5 * f * f) / math.sqrt(2 * math.pi) / _ndtr(sgn * f)


def _site_solve(K, V):
    s = 1 / torch.sqrt(V)
    B = s[:, None] * K * s[None, :]
    B.diagonal().add_(1.0)
    return torch.linalg.cholesky(B), s


def _laplace_exact(case, x, y, off, ls, magn):
    n = x.shape[0]
    K = _k_sexp(_sq(x, x, ls), magn)
    K.diagonal().add_(JITTER)
    y = _t(y)
    o = torch.zeros(n, dtype=torch.float64) if off is None else _t(off)
    f = torch.zeros(n, dtype=torch.float64)
    for _ in range(50):
        g = _dloglik(case["lik"], f + o, y)
        g2 = (_dloglik(case["lik"], f + 1e-6 + o, y) - g) / 1e-6  # the package's curvature is this difference
        V, z = -1 / g2, f - g / g2
        L, s = _site_solve(K, V)
        a = s * torch.cholesky_solve((s * z)[:, None], L)[:, 0]
        new = K @ a
        diff = float((new - f).abs().max())
        f = new
        if diff < case["tol"]:
            break
    ev = float(_loglik(case["lik"], f + o, y).sum() - 0.5 * f @ a - torch.log(L.diagonal()).sum())
    return {"energy": -ev, "fmean": f.numpy(), "alpha": a.numpy()}


def _ep_exact(case, x, y, ls, magn):
    n = x.shape[0]
    K = _k_sexp(_sq(x, x, ls), magn)
    K.diagonal().add_(JITTER)
    y = _t(y)
    gx, gw = np.polynomial.hermite_e.hermegauss(11)
    gx, gw = _t(gx), _t(gw / gw.sum())
    zo, Po, fm, fv = torch.zeros(n, dtype=torch.float64), torch.zeros(n, dtype=torch.float64), torch.zeros(n, dtype=torch.float64), K.diagonal().clone()
    damp, old = 0.9, math.inf
    for it in range(1, 101):
        cp = 1 / fv - Po
        cm, cv = (fm / fv - zo * Po) / cp, 1 / cp
        fg = cm[:, None] + torch.sqrt(cv)[:, None] * gx[None, :]
        lk = torch.exp(_loglik(case["lik"], fg, y[:, None]))
        Z = lk @ gw
        mt = (fg * lk) @ gw / Z
        vt = ((fg - mt[:, None]) ** 2 * lk) @ gw / Z
        P = damp * (1 / vt - 1 / cv) + (1 - damp) * Po
        nu = damp * (mt / vt - cm / cv) + (1 - damp) * zo * Po
        z, V = nu / P, 1 / P
        L, s = _site_solve(K, V)
        a = s * torch.cholesky_solve((s * z)[:, None], L)[:, 0]
        f = K @ a
        var = V * (1 - torch.cholesky_inverse(L).diagonal())
        ev = float(-torch.log(L.diagonal()).sum() - 0.5 * torch.log(V).sum() - 0.5 * z @ a + torch.log(Z).sum()
                   + 0.5 * torch.log(cv + V).sum() + 0.5 * ((cm - z) ** 2 / (cv + V)).sum())
        new = float((f - fm).abs().max())
        if new > old:
            damp *= 0.9
            continue
        damp = max(damp, 0.1)
        fm, fv, zo, Po, old = f, var, z, P, new
        if new < 1e-4:
            break
    if it == 100:
        ev = -math.inf
    return {"energy": -ev, "fmean": f.numpy(), "alpha": a.numpy(), "fvar": var.numpy()}


def _fitc_exact(case, x, y, z, ls, xt):
    n, m = x.shape[0], z.shape[0]
    y = _t(y)
    Kz = _k_m52(_sq(z, z, ls))
    Kz.diagonal().add_(JITTER)
    Lz = torch.linalg.cholesky(Kz)
    U = torch.cat([_k_m52(_sq(x[i:i + 16384], z, ls)) for i in range(0, n, 16384)])
    A = torch.linalg.solve_triangular(Lz, U.T.contiguous(), upper=False)  # Lz^-1 K_zx
    D = 1.0 + JITTER - (A * A).sum(0)
    S = D + 0.01
    H = A @ (A / S).T
    G_ = H.clone()
    G_.diagonal().add_(1.0)
    Lg = torch.linalg.cholesky(G_)  # C^-1 = S^-1 - S^-1 A^T G^-1 A S^-1
    q = A @ (y / S)
    al = y / S - (A.T @ torch.cholesky_solve(q[:, None], Lg)[:, 0]) / S
    w = A @ al
    f = A.T @ w + D * al
    r = (y - f) / 0.1
    ll = float((-0.5 * r * r).sum()) - n * (0.5 * math.log(2 * math.pi) + math.log(0.1))
    logdet = float(torch.log(S).sum() + 2 * torch.log(Lg.diagonal()).sum())
    ev = ll - 0.5 * float(f @ al) + 0.5 * (n * math.log(0.01) - logdet)
    T = torch.linalg.solve_triangular(Lz, _k_m52(_sq(z, xt, ls)), upper=False)
    # A C^-1 A^T = H - H G^-1 H = I - G^-1, applied to T: var = 1 - |T|^2 + T^T G^-1 T
    v = torch.linalg.solve_triangular(Lg, T, upper=False)
    return {"energy": -ev, "fmean": f.numpy(), "pred": {"mean": (T.T @ w).numpy(), "var": (1.0 - (T * T).sum(0) + (v * v).sum(0)).numpy()}}


def exact(case, seed):
    k = case["kind"]
    if k == "regress":
        x, y, ls, sigma, xt = _regress_inputs(case, seed)
        return _gauss_exact(case, x, y, ls, sigma, case["grad"], xt if case["m"] else None)
    if k == "latent":
        x, y, off, ls, magn = _latent_inputs(case, seed)
        return _ep_exact(case, x, y, ls, magn) if case["approx"] == "ep" else _laplace_exact(case, x, y, off, ls, magn)
    if k == "predict":
        x, y, ls, sigma, xt = _predict_inputs(case, seed)
        return _gauss_exact(dict(case, cf="matern52"), x, y, ls, sigma, False, xt)["pred"]
    if k == "batch":
        if case["problems"] * case["nmax"] ** 3 > 4e11 and case["restarts"]:
            return None  # minutes on the CPU
        xs, ys, lss, sigma = _batch_inputs(case, seed)
        o = [_gauss_exact(dict(cf="matern52"), x, y, ls, sigma, True) for x, y, ls in zip(xs, ys, lss)]
        return {"energy": np.array([v["energy"] for v in o]), "grad": np.stack([v["grad"] for v in o])}
    return _fitc_exact(case, *_fitc_inputs(case, seed))
