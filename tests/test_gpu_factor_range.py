"""The FP64 factor of matrices whose entries are far from 1."""

import numpy as np
import pytest

from oracle import gp_oracle as O
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


# D A D, D a power of two for every row: the factor is D chol(A) to the factor
# test's tolerance for A itself (1e-12), entries between 2^-900 and 2^900, as
# one scale and as rows of very different scales side by side
@pytest.mark.parametrize("N", [64, 192])
@pytest.mark.parametrize("scale", [-450, -300, 300, 450, "rows"])
def test_potrf_over_the_range_of_fp64(N, scale):
    import torch

    from probit_amd import _lib
    rng = np.random.default_rng(N)
    X = rng.normal(size=(N, 2))
    s = np.sqrt(rng.uniform(0.5, 5.0, size=N))
    A = np.eye(N) + s[:, None] * O.gram(O.KernelSpec.make(O.EQ, 1.0, 0.7, 2), X) * s
    k = rng.integers(-250, 251, size=N) if scale == "rows" else np.full(N, scale)
    D = np.ldexp(1.0, k)
    Ad = torch.as_tensor(D[:, None] * A * D, device="cuda").t().contiguous()
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    logd = torch.empty(N, dtype=torch.float64, device="cuda")
    dinv = torch.empty(N * 64, dtype=torch.float64, device="cuda")
    rc = _lib.lib().pgp_potrf(0, Ad.data_ptr(), N, N, dinv.data_ptr(), logd.data_ptr(),
                              info.data_ptr(), _lib.stream_handle())
    _lib.check(rc, "pgp_potrf")
    torch.cuda.synchronize()
    assert int(info.item()) == 0
    L = np.tril(Ad.t().cpu().numpy()) / D[:, None]
    ref = np.linalg.cholesky(A)
    assert rel_err(L, ref) < 1e-12
    assert rel_err(logd.cpu().numpy() - k * np.log(2.0), np.log(np.diag(ref))) < 1e-12
    Dv = dinv.cpu().numpy().reshape(N // 64, 64, 64)
    for b in range(N // 64):
        r = slice(64 * b, 64 * b + 64)
        assert np.max(np.abs((Dv[b].T * D[r]) @ ref[r, r] - np.eye(64))) < 1e-12
