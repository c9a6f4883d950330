"""Mixed-precision LU of matrices that FP32 factors cannot be made of: a NaN, entries beyond FP32's range,
entries that are FP32 denormals.  ReturnCode.Failure and nothing written to u, as for a singular matrix, at the
panel's shapes (one workgroup of 256, 512, 1024 and 2048 rows, several workgroups)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 64, 300, 700, 1500, 3300])
@pytest.mark.parametrize("what", ["nan", "nancol", "over", "denormal", "zerocol"])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_failure(lsx, n, what, precision):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    if what == "nan":
        A[n // 3, n // 2] = np.nan  # spreads to every later row: some column has only NaN candidates
    elif what == "nancol":
        A[:, n // 2] = np.nan
    elif what == "zerocol":
        A[:, n // 2] = 0.0
    else:
        A *= {"over": 1e39, "denormal": 1e-40}[what]
    cache = lsx.init(lsx.LinearProblem(A, np.ones(n)), lsx.MI355XMixedLUFactorization(precision=precision))
    cache.u[:] = 7.0
    sol = lsx.solve_(cache)
    assert sol.retcode == lsx.ReturnCode.Failure
    np.testing.assert_array_equal(sol.u, np.full(n, 7.0))
