"""Predicts whose solves take several launches or uneven column tiles."""

import numpy as np
import pytest

from oracle import gp_oracle as O
from tests.helpers import make_prior, oracle_spec, rel_err, small_problem

pytestmark = pytest.mark.gpu


# 516 block rows, past the 512 of one launch of the transposed solve.  The
# inputs are 66 groups too far apart to have any covariance, in random order:
# each group's posterior is exact by itself, while the factor has entries of
# all groups in every tile.  (the tolerances of FP32 fits elsewhere: mean and
# variance to 1e-5)
def test_predict_beyond_one_launch_of_block_rows():
    import probit_amd as P
    G, n, ls, var, noise, M = 66, 500, 0.8, 1.3, 0.3, 100
    N = G * n
    rng = np.random.default_rng(5)
    group = rng.permutation(np.repeat(np.arange(G), n))
    X = rng.normal(size=(N, 1)) + 100.0 * group[:, None]
    y = np.sin(X[:, 0]) + noise * rng.normal(size=N)
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode="fp32",
                     log_likelihood=P.log_gaussian_likelihood, tolerance=1e-8)
    params = ((ls, var), (noise,))
    w, p = gp.approximate_posterior(params)
    tg = rng.integers(0, G, size=M)
    Xt = 3.0 * rng.normal(size=(M, 1)) + 100.0 * tg[:, None]
    mean, v = gp.predict(Xt, params, w, p)
    spec = oracle_spec("EQ", var, ls, 1)
    m_ref, v_ref = np.empty(M), np.empty(M)
    for g in np.unique(tg):
        i, j = group == g, tg == g
        K = O.gram(spec, X[i])
        w_ref = np.linalg.solve(K + noise ** 2 * np.eye(n), y[i])
        m_ref[j], v_ref[j] = O.predict(spec, X[i], Xt[j], w_ref, np.full(n, noise ** -2.0))
    assert rel_err(mean.cpu().numpy(), m_ref) < 1e-5
    assert rel_err(v.cpu().numpy(), v_ref) < 1e-5


# requests with few and many test points in one serving step (1, 5, 18 and 141
# column tiles: each of FP32's groupings, two launches of column tiles): each
# as when it is served alone, bit for bit, and as the oracle's
@pytest.mark.parametrize("mode,tol", [("fp64", 1e-9), ("fp32", 1e-5), ("bf16", None)])
def test_uneven_test_points_in_one_serving_step(mode, tol):
    from probit_amd.serving import ServingEngine
    reqs = []
    for k, (N, M) in enumerate([(700, 40), (641, 300), (650, 1100), (704, 40), (600, 9000)]):
        X, y, theta, lp, spec = small_problem(60 + k, N, 2, "gaussian")
        reqs.append((X, y, theta, lp, spec, np.random.default_rng(70 + k).normal(size=(M, 2))))

    def run(idx):
        eng = ServingEngine(precision=mode, capacity=8, hbm_budget_bytes=1 << 33)
        for i in idx:
            X, y, theta, lp, _, Xt = reqs[i]
            assert eng.submit(i, X, y, "EQ", theta[0], theta[1], "gaussian", lp[0], None, Xt)
        out = {}
        while eng.in_flight:
            for c in eng.step():
                out[c.tag] = c
        eng.close()
        return out

    mix = run(range(len(reqs)))
    for i, (X, y, theta, lp, spec, Xt) in enumerate(reqs):
        alone = run([i])[i]
        for k in ("mean", "var"):
            assert np.array_equal(getattr(alone, k).cpu().numpy(),
                                  getattr(mix[i], k).cpu().numpy()), (i, k)
        if tol is not None:
            w_ref = np.linalg.solve(O.gram(spec, X) + lp[0] ** 2 * np.eye(len(X)), y)
            m_ref, v_ref = O.predict(spec, X, Xt, w_ref, np.full(len(X), lp[0] ** -2.0))
            assert rel_err(mix[i].mean.cpu().numpy(), m_ref) < tol
            assert rel_err(mix[i].var.cpu().numpy(), v_ref) < tol


# a state formed in memory with any contents starts with the triangular
# solves' published values (the last 16 bytes a padded row of an FP64
# workspace) cleared
@pytest.mark.parametrize("N", [1, 64, 130, 1000])
def test_published_values_are_cleared_with_a_new_state(N):
    import torch

    import probit_amd as P
    X, y, theta, lp, _ = small_problem(N, max(N, 4), 2, "gaussian")
    X, y = X[:N], y[:N]
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"),
                     log_likelihood=P.log_gaussian_likelihood)
    ws = gp._workspace()
    ws.fill_(0xA5)
    w = torch.zeros(N, dtype=torch.float64)
    gp.predict(X, (theta, lp), w, torch.full((N,), lp[0] ** -2.0, dtype=torch.float64))
    Np = (N + 63) // 64 * 64
    assert not bool(ws[-16 * Np:].any())


# FP64 solves of 5 to 15 and of 16 and more column tiles in one launch against
# a launch per block row and per super-step (PGP_TRSM_WAVEFRONT=0), which take
# the sums off the right-hand side in the same groups: the same bits
_WIDE_FP64 = """
import hashlib
import numpy as np
import probit_amd as P
from tests.helpers import make_prior, small_problem
for N in (64, 300, 1111):
    X, y, theta, lp, _ = small_problem(N, N, 2, "probit")
    gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"),
                     log_likelihood=P.log_probit_likelihood)
    w, p = gp.approximate_posterior((theta, lp))
    for M in (257, 960, 961, 2000):
        out = gp.predict(np.random.default_rng(M).normal(size=(M, 2)), (theta, lp), w, p)
        print("H", N, M, *(hashlib.md5(t.cpu().numpy().tobytes()).hexdigest() for t in out))
"""


def test_wide_fp64_solves_agree_with_the_launch_schedules():
    import os
    import subprocess
    import sys
    from pathlib import Path
    root = Path(__file__).resolve().parent.parent
    out = []
    for on in ("0", "1"):
        r = subprocess.run([sys.executable, "-c", _WIDE_FP64], cwd=root, capture_output=True,
                           text=True, timeout=100,
                           env={**os.environ, "PGP_TRSM_WAVEFRONT": on,
                                "PYTHONPATH": str(root)})
        assert r.returncode == 0, r.stderr
        out.append([ln for ln in r.stdout.splitlines() if ln.startswith("H ")])
    assert len(out[0]) == 12 and out[0] == out[1]
