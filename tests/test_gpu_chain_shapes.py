"""The column chain of the Cholesky (workgroup per block row, super-steps) and
the segmented triangular solves at the sizes where their schedules change:
one to three blocks, whole and ragged segments of four block rows, whole and
ragged super-steps, one row past each."""

import numpy as np
import pytest

from oracle import gp_oracle as O
from tests.helpers import lik_kind, make_prior, rel_err, small_problem

pytestmark = pytest.mark.gpu

SIZES = [1, 64, 65, 129, 192, 256, 257, 320, 321, 512, 513, 576, 640, 641, 769, 833]


# the fit's tolerances against the oracle: FP64 1e-9; FP32 factors keep the
# FP64 fixed point, the variance to 1e-5
@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("mode,tol,vtol", [("fp64", 1e-9, 1e-9), ("fp32", 1e-5, 1e-5)])
def test_fit_at_schedule_edges(N, mode, tol, vtol):
    import probit_amd as P
    D = 2
    X, y, theta, lp, spec = small_problem(N, max(N, 4), D, "probit")
    if N < 4:  # (the classes' cutpoints need a few points)
        X, y = X[:N], y[:N]
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode=mode,
                     log_likelihood=P.log_probit_likelihood, tolerance=1e-8)
    w, p = gp.approximate_posterior((theta, lp))
    K = O.gram(spec, X)
    w_ref, _, _ = O.laplace_weight(K, y, lik_kind("probit"), lp, tol=1e-8)
    p_ref, _ = O.laplace_precision(K, y, lik_kind("probit"), lp, w_ref)
    assert rel_err(w.cpu().numpy(), w_ref) < tol
    assert rel_err(p.cpu().numpy(), p_ref) < tol
    Xt = np.random.default_rng(7).normal(size=(33, D))
    mean, var = gp.predict(Xt, (theta, lp), w, p)
    m_ref, v_ref = O.predict(spec, X, Xt, w_ref, p_ref)
    assert rel_err(mean.cpu().numpy(), m_ref) < tol
    assert rel_err(var.cpu().numpy(), v_ref) < vtol


# the gradient's tolerance against the closed form of the oracle
# (tests/test_gpu_laplace.py: 1e-7)
@pytest.mark.parametrize("N", [64, 130, 200, 321, 577])
@pytest.mark.parametrize("lik", ["gaussian", "probit"])
def test_gradient_at_doubling_edges(N, lik):
    import probit_amd as P
    D = 2
    X, y, theta, lp, spec = small_problem(N, N, D, lik)
    ll = P.log_gaussian_likelihood if lik == "gaussian" else P.log_probit_likelihood
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), log_likelihood=ll, tolerance=1e-11)
    val, ((g_ls, g_var), g_lik) = gp.value_and_grad()((theta, lp))
    K = O.gram(spec, X)
    w = O.laplace_weight_converged(K, y, lik_kind(lik), lp)
    ref = O.laplace_objective_gradient(spec, X, y, lik_kind(lik), lp, w)
    ref_ls = sum(ref[f"lengthscale{d}"] for d in range(D))
    assert abs(val - O.objective_LA(spec, X, y, lik_kind(lik), lp, w)) < 1e-9 * abs(val)
    for got, want in [(g_ls, ref_ls), (g_var, ref["variance"]), (g_lik[0], ref["noise_std"])]:
        assert abs(got - want) <= 1e-7 * max(1.0, abs(want))
    if lik == "probit":
        cut = np.asarray(g_lik[1])[1:-1]
        want = np.asarray(ref["cutpoints"])[1:-1]
        assert np.max(np.abs(cut - want)) <= 1e-7 * max(1.0, np.max(np.abs(want)))


# the wide solves of predict: one block row, whole and ragged column tiles,
# and the edge of a launch's 128 column tiles (the fit's tolerances above)
@pytest.mark.parametrize("N,M", [(64, 300), (65, 1025), (300, 8192), (300, 8193), (130, 16449)])
@pytest.mark.parametrize("mode,tol,vtol", [("fp64", 1e-9, 1e-9), ("fp32", 1e-5, 1e-5)])
def test_predict_at_column_tile_edges(N, M, mode, tol, vtol):
    import probit_amd as P
    D = 2
    X, y, theta, lp, spec = small_problem(N, N, D, "probit")
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode=mode,
                     log_likelihood=P.log_probit_likelihood, tolerance=1e-8)
    w, p = gp.approximate_posterior((theta, lp))
    K = O.gram(spec, X)
    w_ref, _, _ = O.laplace_weight(K, y, lik_kind("probit"), lp, tol=1e-8)
    p_ref, _ = O.laplace_precision(K, y, lik_kind("probit"), lp, w_ref)
    Xt = np.random.default_rng(M).normal(size=(M, D))
    mean, var = gp.predict(Xt, (theta, lp), w, p)
    m_ref, v_ref = O.predict(spec, X, Xt, w_ref, p_ref)
    assert rel_err(mean.cpu().numpy(), m_ref) < tol
    assert rel_err(var.cpu().numpy(), v_ref) < vtol


# a batch whose outer updates together fill the chip takes the 128-tiles (odd
# and even block counts below the first super-step), each member alone the
# 64-tiles: the same bits
@pytest.mark.parametrize("mode,count", [("fp64", 5), ("fp32", 8), ("bf16", 6)])
def test_outer_update_tilings_agree(mode, count):
    import torch

    import probit_amd as P
    from probit_amd.serving import ServingEngine
    sizes = [1600 + 50 * (k % 2) - k for k in range(count)]
    probs = [small_problem(200 + k, N, 2, "probit", "EQ", noise=0.5) for k, N in enumerate(sizes)]
    eng = ServingEngine(precision=mode, capacity=8)
    for tag, (X, y, theta, lp, _) in enumerate(probs):
        assert eng.submit(tag, X, y, "EQ", theta[0], theta[1], "probit", lp[0], lp[1])
    out = {}
    while eng.in_flight:
        for c in eng.step():
            out[c.tag] = c
    eng.close()
    for tag, (X, y, theta, lp, _) in enumerate(probs):
        gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode=mode,
                         log_likelihood=P.log_probit_likelihood)
        w, p = gp.approximate_posterior((theta, lp))
        assert torch.equal(w, out[tag].weight) and torch.equal(p, out[tag].precision), tag


# super-steps that carry a part of the outer update (odd and even trailing
# block counts, all of it and a part, before and after the rows below) against
# the two-launch form, which carries none: the same bits
@pytest.mark.parametrize("mode,N", [("fp64", 1300), ("fp64", 4450), ("fp64", 7000),
                                    ("fp32", 4450), ("fp32", 9000), ("bf16", 7000)])
def test_superstep_with_outer_tiles_agrees(mode, N):
    import torch

    import probit_amd as P
    from probit_amd import autotune as at
    X, y, theta, lp, _ = small_problem(N, N, 2, "probit", "EQ", noise=0.5)
    saved, out = at.get(mode, 1), []
    try:
        for merge in (1, 2):
            at.set_entry(mode, 1, dict(saved, column_merge=merge))
            gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode=mode,
                             log_likelihood=P.log_probit_likelihood)
            out.append(gp.approximate_posterior((theta, lp)))
    finally:
        at.set_entry(mode, 1, saved)
    for a, b in zip(*out):
        assert torch.equal(a, b)


# FP32 solves of 5 to 15 and of 16 and more column tiles in one launch against
# a launch per block row and per super-step (PGP_TRSM_WAVEFRONT=0): same bits
_WIDE_FP32 = """
import hashlib, sys
import numpy as np
import probit_amd as P
from tests.helpers import make_prior, small_problem
for N in (64, 300, 1111):
    X, y, theta, lp, _ = small_problem(N, N, 2, "probit")
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode="fp32",
                     log_likelihood=P.log_probit_likelihood)
    w, p = gp.approximate_posterior((theta, lp))
    for M in (257, 960, 961, 2000):
        out = gp.predict(np.random.default_rng(M).normal(size=(M, 2)), (theta, lp), w, p)
        print("H", N, M, *(hashlib.md5(t.cpu().numpy().tobytes()).hexdigest() for t in out))
"""


def test_wide_fp32_solves_agree_with_the_launch_schedules():
    import os
    import subprocess
    import sys
    from pathlib import Path
    root = Path(__file__).resolve().parent.parent
    out = []
    for on in ("0", "1"):
        r = subprocess.run([sys.executable, "-c", _WIDE_FP32], cwd=root, capture_output=True,
                           text=True, timeout=100,
                           env={**os.environ, "PGP_TRSM_WAVEFRONT": on,
                                "PYTHONPATH": str(root)})
        assert r.returncode == 0, r.stderr
        out.append([ln for ln in r.stdout.splitlines() if ln.startswith("H ")])
    assert len(out[0]) == 12 and out[0] == out[1]
