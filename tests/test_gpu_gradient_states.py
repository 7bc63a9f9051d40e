"""The Laplace gradient at states that its other tests do not reach: precisions
that are zero or negative, a factor stored in FP32, small Gaussian noise."""

import numpy as np
import pytest

from oracle import gp_oracle as O
from tests.helpers import lik_kind, make_prior, oracle_spec, rel_err, small_problem

pytestmark = pytest.mark.gpu


def _closed_form(spec, X, y, lp, w):
    """O.laplace_objective_gradient where some W = -d2 are not positive: the
    W^1/2 of the factor and of C is sqrt(max(W, 0))."""
    K = O.gram(spec, X)
    N = len(K)
    d = O.lik_derivs(O.PROBIT, K @ w, y, lp, order=3)
    s = np.sqrt(np.maximum(-d["d2"], 0.0))
    Cm = s[:, None] * np.linalg.inv(np.eye(N) + s[:, None] * K * s) * s
    sig = np.diag(K) - np.einsum("ij,ji->i", K, Cm @ K)
    s2 = -0.5 * sig * d["d3"]
    s2 = s2 - Cm @ (K @ s2)
    out = [-0.5 * w @ Kd @ w + 0.5 * np.sum(Cm * Kd) + s2 @ (Kd @ w)
           for _, Kd in O.gram_param_derivs(spec, X)]
    Lp, Lfp, Lffp = d["sigma"]
    out.append(-np.sum(Lp) + 0.5 * np.sum(sig * -Lffp) + s2 @ (K @ Lfp))
    return -d["d2"], [name for name, _ in O.gram_param_derivs(spec, X)], np.array(out)


# a weight set from outside, some of whose latents lie so far outside their
# points' class that the probability is its floor (W < 0), or
# so far inside that W = 0 exactly: one such column, a few, most of them.
# (the tolerance of tests/test_gpu_laplace.py, 1e-7)
@pytest.mark.parametrize("N,wrong,noise", [(64, 1, 0.1), (130, 4, 0.1), (321, 12, 0.1),
                                           (321, 200, 1.0), (200, 0, 0.01)])
def test_gradient_where_precisions_are_not_positive(N, wrong, noise):
    import torch

    import probit_amd as P
    rng = np.random.default_rng(N)
    X = rng.normal(size=(N, 2))
    spec = oracle_spec("EQ", 1.3, 0.8, 2)
    w = rng.normal(size=N) * 0.2
    f = O.gram(spec, X) @ w
    cut = np.array([-np.inf, -0.7, 0.9, np.inf])
    y = np.searchsorted(cut[1:-1], f).astype(np.float64)
    if noise == 1.0:
        cut = np.array([-np.inf, -7.2, 0.9, np.inf])
    # the lowest class for the points nearest to 7.3 noise above it
    y[np.argsort(np.abs(f - cut[1] - 7.3 * noise))[:wrong]] = 0.0
    lp = (noise, cut)
    W, names, ref = _closed_form(spec, X, y, lp, w)
    assert np.sum(W <= 0.0) >= max(wrong, 1) and np.any(W > 0.0)
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"),
                     log_likelihood=P.log_probit_likelihood)
    ks, ls = gp._structs(((0.8, 1.3), lp))
    gp._set_state(ks, ls, torch.from_numpy(w), None, fixed_point=True)
    got = np.asarray(gp._grad(ks, ls))
    at = {"variance": 0, "lengthscale0": 1, "lengthscale1": 2}
    mine = np.array([got[at[n]] for n in names] + [got[1 + 2 * 2]])
    assert np.all(np.abs(mine - ref) <= 1e-7 * np.maximum(1.0, np.abs(ref)))


# FP32 factors: the gradient's error against the oracle at the FP64 fixed point
# is the factor's, eps32 times the condition of B, of the largest entry (8: the
# factor, the inverse and the products each bring one such error)
@pytest.mark.parametrize("N", [64, 130, 321, 577])
@pytest.mark.parametrize("lik", ["gaussian", "probit"])
def test_gradient_from_an_fp32_factor(N, lik):
    import probit_amd as P
    D = 2
    X, y, theta, lp, spec = small_problem(N, N, D, lik)
    ll = P.log_gaussian_likelihood if lik == "gaussian" else P.log_probit_likelihood
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), log_likelihood=ll, tolerance=1e-10,
                     precision_mode="fp32")
    _, ((g_ls, g_var), g_lik) = gp.value_and_grad()((theta, lp))
    K = O.gram(spec, X)
    w = O.laplace_weight_converged(K, y, lik_kind(lik), lp)
    ref = O.laplace_objective_gradient(spec, X, y, lik_kind(lik), lp, w)
    got = [g_ls, g_var, g_lik[0]]
    want = [sum(ref[f"lengthscale{d}"] for d in range(D)), ref["variance"], ref["noise_std"]]
    if lik == "probit":
        got += list(np.asarray(g_lik[1])[1:-1])
        want += list(np.asarray(ref["cutpoints"])[1:-1])
    s = np.sqrt(-O.lik_derivs(lik_kind(lik), K @ w, y, lp)["d2"])
    cond = np.linalg.cond(np.eye(N) + s[:, None] * K * s)
    assert rel_err(got, want) < 8 * 2.0 ** -24 * cond


# FP64 at small noise, where the sums behind diag Sigma cancel: eps64 times the
# condition of B the same way
@pytest.mark.parametrize("noise", [1e-1, 1e-2, 1e-3])
def test_gradient_at_small_gaussian_noise(noise):
    import probit_amd as P
    N, D = 200, 2
    X, y, theta, lp, spec = small_problem(N, N, D, "gaussian", noise=noise)
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), tolerance=1e-11,
                     log_likelihood=P.log_gaussian_likelihood)
    _, ((g_ls, g_var), g_lik) = gp.value_and_grad()((theta, lp))
    K = O.gram(spec, X)
    w = np.linalg.solve(K + noise ** 2 * np.eye(N), y)
    ref = O.laplace_objective_gradient(spec, X, y, O.GAUSSIAN, lp, w)
    want = [sum(ref[f"lengthscale{d}"] for d in range(D)), ref["variance"], ref["noise_std"]]
    cond = np.linalg.cond(np.eye(N) + K / noise ** 2)
    assert rel_err([g_ls, g_var, g_lik[0]], want) < 8 * 2.0 ** -53 * cond
