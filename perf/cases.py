"""Performance cases: the work that users of probit_amd have it do, by size and direction.

Every case goes through the package's public entry points (LaplaceGP, VBGP,
sample_prior, ServingEngine / serve_async).  Inputs are synthetic: a latent
function from random Fourier features of the kernel, ordinal labels by
cutpoints or Gaussian targets, as in the repository's own data sets
(probit_amd/data.py).  `op` says what one pass does:

  posterior  approximate_posterior, then predict at M test points
  evidence   value_and_grad of the objective: one hyperparameter step
  predict    predict at M points from a posterior that is already resident
  covariance predict_covariance at M points from a resident posterior
  sweep      value_and_grad_batch over a grid of lengthscales
  prior      sample_prior: Gram matrix, Cholesky factor, L z
  serve      a stream of uneven requests through the batching engine
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from probit_amd import (EQ, LaplaceGP, Matern12, VBGP, log_gaussian_likelihood,
                        log_probit_likelihood)
from probit_amd.prior import sample_prior
from probit_amd.serving import ServingEngine, serve_async

TOLERANCE = 1e-5
MAXITER = 100
PROBIT_FLOOR = 1e-10
PRIOR_JITTER = 1e-6


def _case(name, op, **kw):
    c = {"name": name, "op": op, "gp": "laplace", "precision": "fp64", "N": 0, "D": 1, "M": 0,
         "kernel": "EQ", "ard": False, "lengthscale": 1.0, "variance": 1.0, "period": 0.0, "J": 0,
         "noise": 0.2, "x": "uniform", "count": 0}
    c.update(kw)
    return c


def listed():
    return [
        # the plain regression example: 20 points, periodic kernel, 1000 test points
        _case("regression_n20", "posterior", N=20, M=1000, period=0.5),
        # one optimiser step on a data set of the classification examples' size
        _case("evidence_n300", "evidence", N=300, D=2, J=3, noise=0.63, x="normal"),
        # an ordinary ordinal regression, ragged sizes, ARD lengthscales
        _case("posterior_n1537", "posterior", N=1537, D=3, M=501, J=5, noise=0.5, ard=True),
        # the ordinal data set of 8192 points in the mixed-precision mode
        _case("posterior_n8192_fp32", "posterior", N=8192, D=2, M=4096, J=3, kernel="Matern12",
              noise=math.sqrt(0.4), x="normal", precision="fp32"),
        # the single large mixed-precision fit
        _case("posterior_n16384_bf16", "posterior", N=16384, D=8, M=1024, J=5, ard=True,
              noise=math.sqrt(0.1), precision="bf16"),
        # an optimiser step on a large data set: fit, evidence and adjoint
        _case("evidence_n4096", "evidence", N=4096, D=4, J=3, lengthscale=0.8, variance=1.5,
              noise=math.sqrt(0.4), x="normal"),
        # the variational approximation: fixed point, objective and predict
        _case("vb_n1024", "posterior", gp="vb", N=1024, D=2, M=256, J=3, noise=0.8, x="normal"),
        # many test points against a posterior that stays resident
        _case("predict_n3000", "predict", N=3000, D=4, M=5000, noise=0.2),
        # the joint predictive covariance, for sampling from the posterior
        _case("covariance_n2000", "covariance", N=2000, D=3, M=1000, J=3, noise=0.5,
              kernel="Matern12"),
        # a lengthscale sweep of the evidence and its gradient
        _case("sweep_n512", "sweep", N=512, D=2, J=3, noise=0.63, x="normal", count=16),
        # the data generators' exact prior draw (8192 training and 4096 test points)
        _case("prior_n12288", "prior", N=12288, D=2, M=1, kernel="Matern12", x="normal"),
        # the serving stream: N log-uniform on [64, 4096], 256 test points each
        _case("serve_256_fp32", "serve", N=4096, M=256, count=256, precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    op = rng.choice(["posterior", "posterior", "posterior", "evidence", "evidence", "predict",
                     "covariance", "sweep", "prior", "serve", "vb"])
    J = rng.choice([0, 2, 3, 4, 5])
    kw = {"D": rng.randint(1, 8), "kernel": rng.choice(["EQ", "Matern12"]), "J": J,
          "lengthscale": round(math.exp(rng.uniform(math.log(0.4), math.log(2.0))), 3),
          "variance": round(rng.uniform(0.8, 1.6), 3),
          "noise": round(rng.uniform(0.4, 0.7) if J else rng.uniform(0.2, 0.4), 3),
          "x": rng.choice(["uniform", "normal"]), "ard": rng.random() < 0.3}
    if op == "posterior":
        p = rng.choice(["fp64", "fp64", "fp32", "bf16"])
        return _case("", op, N=_log_int(rng, 20, {"fp64": 6000, "fp32": 9000, "bf16": 12000}[p]),
                     M=_log_int(rng, 16, 4096), precision=p, **kw)
    if op == "evidence":
        return _case("", op, N=_log_int(rng, 100, 4096), **kw)
    if op == "predict":
        return _case("", op, N=_log_int(rng, 200, 4096), M=_log_int(rng, 64, 5000), **kw)
    if op == "covariance":
        return _case("", op, N=_log_int(rng, 200, 3000), M=_log_int(rng, 64, 1500), **kw)
    if op == "sweep":
        return _case("", op, N=_log_int(rng, 64, 700), count=rng.randint(6, 24), **kw)
    if op == "prior":
        kw.update(J=0, noise=0.0, kernel="Matern12")
        return _case("", op, N=_log_int(rng, 100, 12288), M=_log_int(rng, 1, 32), **kw)
    if op == "vb":  # the plain fixed-point iteration needs noise against the signal
        kw.update(J=rng.choice([2, 3, 4, 5]), noise=round(rng.uniform(0.8, 1.2), 3), variance=1.0)
        return _case("", "posterior", gp="vb", N=_log_int(rng, 64, 1500), M=_log_int(rng, 16, 512),
                     **kw)
    return _case("", "serve", N=_log_int(rng, 1024, 4096), M=rng.randint(64, 256),
                 count=rng.randint(48, 256), precision=rng.choice(["fp32", "fp32", "fp64"]))


# ---- inputs ------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _points(g, n, D, x):
    if x == "normal":
        return torch.randn((n, D), dtype=torch.float64, device="cuda", generator=g)
    return 2.0 * torch.rand((n, D), dtype=torch.float64, device="cuda", generator=g) - 1.0


def _lengthscales(case, seed):
    if not case["ard"]:
        return case["lengthscale"]
    r = random.Random(int(seed))
    return np.exp([r.uniform(math.log(0.3), math.log(3.0)) for _ in range(case["D"])])


def _latent(g, X, kernel, ls, var, features=256):
    D = X.shape[1]
    w = torch.randn((features, D), dtype=torch.float64, device="cuda", generator=g)
    if kernel == "Matern12":
        w = w / torch.randn((features, 1), dtype=torch.float64, device="cuda", generator=g).abs()
    w = w / torch.as_tensor(ls, dtype=torch.float64, device="cuda")
    b = 2.0 * math.pi * torch.rand(features, dtype=torch.float64, device="cuda", generator=g)
    return math.sqrt(2.0 * var / features) * torch.cos(X @ w.t() + b).sum(1)


def _targets(g, f, J, noise):
    """Gaussian targets, or labels of J classes with equal counts and their cutpoints."""
    t = f + noise * torch.randn(f.shape[0], dtype=torch.float64, device="cuda", generator=g)
    if not J:
        return t, None
    s = torch.sort(t).values
    n = s.shape[0]
    k = torch.tensor([(n * j) // J for j in range(1, J)], device="cuda")
    inner = 0.5 * (s[k - 1] + s[k])
    cut = np.concatenate([[-np.inf], inner.cpu().numpy(), [np.inf]])
    return torch.bucketize(t, inner, right=True).to(torch.float64), cut


def _data(case, seed):
    g = _generator(seed)
    ls = _lengthscales(case, seed)
    X = _points(g, case["N"], case["D"], case["x"])
    f = _latent(g, X, case["kernel"], ls, case["variance"])
    y, cut = _targets(g, f, case["J"], case["noise"])
    Xt = _points(g, max(1, case["M"]), case["D"], case["x"])
    lik = (case["noise"],) if cut is None else (case["noise"], cut)
    return X, y, Xt, (ls, case["variance"]), lik


def _prior(case):
    base = EQ if case["kernel"] == "EQ" else Matern12

    def prior(theta):
        k = theta[1] * base().stretch(theta[0])
        return k.periodic(case["period"]) if case["period"] else k

    return prior


def _sweep_parameters(case, theta, lik):
    grid = np.exp(np.linspace(math.log(0.5), math.log(2.0), case["count"]))
    return [((float(s) * theta[0], theta[1]), lik) for s in grid]


def _requests(case, seed):
    """The serving stream's requests: uneven N and D, both likelihoods and kernels
    (the case sets the sizes, the seed the data)."""
    r, g = random.Random(case["count"]), _generator(seed)
    out = []
    for tag in range(case["count"]):
        N, D, M = _log_int(r, 64, case["N"]), r.randint(1, 8), case["M"]
        kind = r.choice(["EQ", "Matern12"])
        ls = math.exp(r.uniform(math.log(0.2), math.log(2.0)))
        J = r.choice([0, 0, 0, 0, 2, 3, 4, 5])
        noise = 0.5 if J else 0.2
        X, Xt = _points(g, N, D, "uniform"), _points(g, M, D, "uniform")
        y, cut = _targets(g, _latent(g, X, kind, ls, 1.0, features=64), J, noise)
        out.append((tag, X, y, kind, ls, 1.0, "probit" if J else "gaussian", noise, cut, Xt, None))
    return out


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    if case["op"] == "serve":
        s.requests = _requests(case, seed)
        s.engine = ServingEngine(precision=case["precision"], capacity=512)
        return s
    if case["op"] == "prior":
        g = _generator(seed)
        s.X = _points(g, case["N"], case["D"], case["x"])
        s.z = torch.randn((case["N"], case["M"]), dtype=torch.float64, device="cuda", generator=g)
        s.kernel = _prior(case)((_lengthscales(case, seed), case["variance"]))
        return s
    X, y, s.Xt, s.theta, s.lik = _data(case, seed)
    s.gp = (VBGP if case["gp"] == "vb" else LaplaceGP)(
        data=(X, y), prior=_prior(case), precision_mode=case["precision"], tolerance=TOLERANCE,
        log_likelihood=log_probit_likelihood if case["J"] else log_gaussian_likelihood)
    if case["op"] == "evidence":
        s.step = s.gp.value_and_grad()
    elif case["op"] == "sweep":
        s.step = s.gp.value_and_grad_batch()
        s.grid = _sweep_parameters(case, s.theta, s.lik)
    elif case["op"] in ("predict", "covariance"):
        s.posterior = s.gp.approximate_posterior((s.theta, s.lik))
    return s


def run(state):
    s, case = state, state.case
    op = case["op"]
    if op == "posterior":
        weight, precision = s.gp.approximate_posterior((s.theta, s.lik))
        mean, var = s.gp.predict(s.Xt, (s.theta, s.lik), weight, precision)
        return {"weight": weight, "precision": precision, "mean": mean, "var": var}
    if op == "evidence":
        value, ((gls, gvar), glik) = s.step((s.theta, s.lik))
        return {"value": value, "lengthscale": gls, "variance": gvar, "noise": glik[0],
                "cutpoints": glik[1] if len(glik) > 1 else None}
    if op == "sweep":
        values, grads = s.step(s.grid)
        return {"values": values,
                "lengthscale": np.stack([np.atleast_1d(g[0][0]) for g in grads]),
                "variance": np.stack([g[0][1] for g in grads]),
                "noise": np.stack([g[1][0] for g in grads]),
                "cutpoints": np.stack([g[1][1] for g in grads]) if case["J"] else None}
    if op == "predict":
        return list(s.gp.predict(s.Xt, (s.theta, s.lik), *s.posterior))
    if op == "covariance":
        return s.gp.predict_covariance(s.Xt, (s.theta, s.lik), *s.posterior)
    if op == "prior":
        return sample_prior(s.kernel, s.X, s.z, jitter=PRIOR_JITTER)
    done = serve_async(s.engine, s.requests)
    done = [done[r[0]] for r in s.requests]
    return {"mean": torch.stack([c.mean for c in done]), "var": torch.stack([c.var for c in done]),
            "weight": torch.cat([c.weight for c in done]),
            "precision": torch.cat([c.precision for c in done])}


# ---- the work a pass cannot do without ---------------------------------------------
def _fit_work(N, D, J, refits):
    """Gram matrix, `refits` factorisations of N^3 / 3 and the two solves of each."""
    n = float(N)
    return 8.0 * n * (D + 3), n * n * (3 * D + 4) / 2 + refits * (n ** 3 / 3 + 4 * n * n)


def work(case):
    N, D, M, J, op = case["N"], case["D"], case["M"], case["J"], case["op"]
    n, m = float(N), float(M)
    refits = 6 if J else 1
    if op == "prior":
        return {"bytes": 8 * n * (D + 2 * m), "flops": n * n * (3 * D + 4) / 2 + n ** 3 / 3 + n * n * m}
    if op == "serve":
        b = fl = 0.0
        for r in range(case["count"]):  # the sizes' quantiles
            q = math.exp(math.log(64) + (r + 0.5) / case["count"] * math.log(N / 64))
            fb, ff = _fit_work(q, 4.5, 3, 3.5)
            b += fb + 8 * m * 6.5
            fl += ff + q * q * m
        return {"bytes": b, "flops": fl}
    pred = n * n * m + n * m * (3 * D + 4)
    fb, ff = _fit_work(N, D, J, refits)
    if op == "predict":
        return {"bytes": 4 * n * n + 8 * m * (D + 2), "flops": pred}
    if op == "covariance":
        return {"bytes": 4 * n * n + 8 * m * (D + m), "flops": pred + m * m * n}
    if op == "evidence":
        return {"bytes": fb, "flops": ff + n ** 3}
    if op == "sweep":
        return {"bytes": fb * case["count"], "flops": (ff + n ** 3) * case["count"]}
    if case["gp"] == "vb":  # one factorisation of sigma^2 I + K, its inverse, the B factor
        return {"bytes": fb + 8 * m * (D + 2), "flops": 4 * n ** 3 / 3 + 20 * 4 * n * n + pred}
    return {"bytes": fb + 8 * m * (D + 2), "flops": ff + pred}


# ---- the same results from plain torch in 64 bits --------------------------------------
def _gram(kernel, X, Z, ls, var, period=0.0):
    ls = torch.as_tensor(ls, dtype=torch.float64, device=X.device).expand(X.shape[1])
    r2 = torch.zeros((X.shape[0], Z.shape[0]), dtype=torch.float64, device=X.device)
    for d in range(X.shape[1]):
        q = X[:, d, None] - Z[None, :, d]
        if period:
            q = 2.0 * torch.sin(math.pi * q / period)
        r2 = r2 + (q / ls[d]) ** 2
    if kernel == "EQ":
        return var * torch.exp(-0.5 * r2)
    # the square root's derivative at 0 is taken as 0
    r = torch.sqrt(torch.where(r2 > 0, r2, torch.ones_like(r2)))
    return var * torch.exp(-torch.where(r2 > 0, r, torch.zeros_like(r)))


def _likelihood(f, y, noise, cut):
    """(log p, d log p / df, W = -d2 log p / df2)."""
    if cut is None:
        r = (y - f) / noise
        return (-0.5 * r * r - torch.log(noise) - 0.5 * math.log(2.0 * math.pi), r / noise,
                torch.ones_like(f) / noise ** 2)
    lab = y.to(torch.int64)
    lo, hi = cut[lab], cut[lab + 1]
    has_lo, has_hi = torch.isfinite(lo), torch.isfinite(hi)
    zero, one = torch.zeros_like(f), torch.ones_like(f)
    z1 = (torch.where(has_lo, lo, zero) - f) / noise
    z2 = (torch.where(has_hi, hi, zero) - f) / noise

    def cdf(z):
        return 0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))

    def pdf(z, has):
        return torch.where(has, torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi), zero)

    p = torch.where(has_hi, cdf(z2), one) - torch.where(has_lo, cdf(z1), zero) + PROBIT_FLOOR
    p1, p2 = pdf(z1, has_lo), pdf(z2, has_hi)
    d1 = (p1 - p2) / noise / p
    return torch.log(p), d1, d1 * d1 - (z1 * p1 - z2 * p2) / noise ** 2 / p


def _laplace(K, y, noise, cut):
    """The Newton fixed point: (weight, W there)."""
    a = torch.zeros_like(y)
    eye = torch.eye(K.shape[0], dtype=K.dtype, device=K.device)
    for _ in range(MAXITER):
        _, d1, W = _likelihood(K @ a, y, noise, cut)
        s = torch.sqrt(W)
        L = torch.linalg.cholesky(eye + s[:, None] * K * s)
        r = d1 - a
        u = torch.cholesky_solve((s * (K @ r))[:, None], L)[:, 0]
        step = r - s * u
        a = a + step
        if float(step.norm()) <= TOLERANCE:
            break
    return a, _likelihood(K @ a, y, noise, cut)[2]


def _vb(K, y, noise, cut):
    a = torch.zeros_like(y)
    eye = torch.eye(K.shape[0], dtype=K.dtype, device=K.device)
    L = torch.linalg.cholesky(noise ** 2 * eye + K)
    for _ in range(MAXITER):
        f = K @ a
        rhs = f + noise * _likelihood(f, y, noise, cut)[1]
        new = torch.cholesky_solve(rhs[:, None], L)[:, 0]
        step, a = float((new - a).norm()), new
        if step <= TOLERANCE:
            break
    return a, torch.ones_like(a) / noise ** 2


def _predictive(K, Kfs, W, weight):
    """(mean, V) with the predictive covariance Kss - V^T V."""
    s = torch.sqrt(W)
    L = torch.linalg.cholesky(torch.eye(K.shape[0], dtype=K.dtype, device=K.device)
                              + s[:, None] * K * s)
    V = torch.linalg.solve_triangular(L, s[:, None] * Kfs, upper=False)
    return Kfs.t() @ weight, V


def _evidence(case, X, y, ls, var, noise, cut):
    """The objective at the Laplace fixed point and its gradient, by automatic
    differentiation through one Newton step taken at the fixed point."""
    leaves = [torch.as_tensor(v, dtype=torch.float64, device=X.device).clone().requires_grad_(True)
              for v in (ls, var, noise)]
    cuts = None if cut is None else cut.clone().requires_grad_(True)
    K = _gram(case["kernel"], X, X, leaves[0], leaves[1])
    eye = torch.eye(K.shape[0], dtype=K.dtype, device=K.device)
    with torch.no_grad():
        a0, W0 = _laplace(K, y, leaves[2], cuts)
        s0 = torch.sqrt(W0)
        L0 = torch.linalg.cholesky(eye + s0[:, None] * K * s0)
    r = _likelihood(K @ a0, y, leaves[2], cuts)[1] - a0
    # (I + W K)^-1 r, linear in r, with the matrix held at the fixed point
    t = s0 * (K.detach() @ r)
    a = a0 + r - s0 * torch.cholesky_solve(t[:, None], L0)[:, 0]
    f = K @ a
    ll, _, W = _likelihood(f, y, leaves[2], cuts)
    s = torch.sqrt(W)
    L = torch.linalg.cholesky(eye + s[:, None] * K * s)
    value = -ll.sum() + 0.5 * f @ a + torch.log(torch.diagonal(L)).sum()
    grads = torch.autograd.grad(value, leaves + ([] if cuts is None else [cuts]))
    grads = [v.detach().cpu().numpy() for v in grads]
    return float(value.detach()), grads


def exact(case, seed):
    op = case["op"]
    if op == "serve":
        return _exact_serve(case, seed)
    if op == "prior":
        g = _generator(seed)
        X = _points(g, case["N"], case["D"], case["x"])
        z = torch.randn((case["N"], case["M"]), dtype=torch.float64, device="cuda", generator=g)
        K = _gram(case["kernel"], X, X, _lengthscales(case, seed), case["variance"])
        K.diagonal().add_(PRIOR_JITTER)
        return torch.linalg.cholesky(K) @ z
    X, y, Xt, (ls, var), lik = _data(case, seed)
    noise = torch.tensor(lik[0], dtype=torch.float64, device=X.device)
    cut = torch.as_tensor(lik[1], device=X.device) if len(lik) > 1 else None
    if op == "evidence":
        v, gr = _evidence(case, X, y, ls, var, noise, cut)
        return {"value": v, "lengthscale": gr[0], "variance": gr[1], "noise": gr[2],
                "cutpoints": gr[3] if cut is not None else None}
    if op == "sweep":
        out = [_evidence(case, X, y, th[0], th[1], noise, cut)
               for th, _ in _sweep_parameters(case, (ls, var), lik)]
        return {"values": np.array([v for v, _ in out]),
                "lengthscale": np.stack([np.atleast_1d(g[0]) for _, g in out]),
                "variance": np.stack([g[1] for _, g in out]),
                "noise": np.stack([g[2] for _, g in out]),
                "cutpoints": np.stack([g[3] for _, g in out]) if cut is not None else None}
    K = _gram(case["kernel"], X, X, ls, var, case["period"])
    Kfs = _gram(case["kernel"], X, Xt, ls, var, case["period"])
    weight, W = (_vb if case["gp"] == "vb" else _laplace)(K, y, noise, cut)
    mean, V = _predictive(K, Kfs, W, weight)
    if op == "covariance":
        return _gram(case["kernel"], Xt, Xt, ls, var, case["period"]) - V.t() @ V
    out = var - (V * V).sum(0)
    if op == "predict":
        return [mean, out]
    return {"weight": weight, "precision": W, "mean": mean, "var": out}


def _exact_serve(case, seed):
    mean, var, weight, prec = [], [], [], []
    for _, X, y, kind, ls, v, _, noise, cut, Xt, _ in _requests(case, seed):
        noise = torch.tensor(noise, dtype=torch.float64, device=X.device)
        cut = None if cut is None else torch.as_tensor(cut, device=X.device)
        K, Kfs = _gram(kind, X, X, ls, v), _gram(kind, X, Xt, ls, v)
        a, W = _laplace(K, y, noise, cut)
        m, V = _predictive(K, Kfs, W, a)
        mean.append(m)
        var.append(v - (V * V).sum(0))
        weight.append(a)
        prec.append(W)
    return {"mean": torch.stack(mean), "var": torch.stack(var), "weight": torch.cat(weight),
            "precision": torch.cat(prec)}
