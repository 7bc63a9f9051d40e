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
