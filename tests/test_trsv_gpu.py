"""Triangular solves at the edges of their shapes: orders around multiples of the 64-row blocks, 1, 2, 15,
16, 17 and 33 right-hand sides, forward and adjoint, on the same factors."""
import numpy as np
import pytest
import scipy.linalg.lapack as lapack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 130, 1000])
@pytest.mark.parametrize("nrhs", [1, 2, 15, 16, 17, 33])
@pytest.mark.parametrize("adjoint", [False, True])
def test_solves_match_lapack(lsx, n, nrhs, adjoint):
    # A = 2 I + N(0,1) / sqrt(n): condition number below 10, so both solves are within a small multiple of
    # n eps of the exact one; bound 20 n eps in the max norm, by column.
    print(f"trsv n={n} nrhs={nrhs} adjoint={adjoint}", flush=True)
    rng = np.random.default_rng(n * 100 + nrhs)
    A = rng.standard_normal((n, n)) / np.sqrt(n)
    A[rng.permutation(n), np.arange(n)] += 2.0
    B = np.asfortranarray(rng.standard_normal((n, nrhs)))
    h = lsx._LUHandle(lsx.Context.get(0), n, lsx.LSX_F64)
    assert h.factor(A) == 0
    F, ipiv = h.factors()
    X = np.empty((n, nrhs), order="F")
    (h.solve_adjoint if adjoint else h.solve)(B, X)
    ref, info = lapack.dgetrs(F, ipiv - 1, B, trans=int(adjoint))
    assert info == 0
    assert (np.abs(X - ref).max(axis=0) <= 20 * n * np.finfo(float).eps * np.abs(ref).max(axis=0)).all()
    # in place, and each column alone up to rounding (one right-hand side takes the other kernel)
    Y = B.copy(order="F")
    (h.solve_adjoint if adjoint else h.solve)(Y, Y)
    np.testing.assert_array_equal(Y, X)
    y = np.empty(n)
    (h.solve_adjoint if adjoint else h.solve)(B[:, -1].copy(), y)
    assert np.abs(y - X[:, -1]).max() <= 20 * n * np.finfo(float).eps * np.abs(y).max()
