"""Predicts whose solves take several launches or uneven column tiles."""

import numpy as np
import pytest

from oracle import gp_oracle as O
from tests.helpers import make_prior, oracle_spec, rel_err

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
