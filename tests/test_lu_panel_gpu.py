"""The LU panel kernel at the edges of its shapes (one row per thread up to 256 and 512 rows, two up to
1024 rows per workgroup, several workgroups beyond, last panels of every width modulo 8) with what makes
a pivot search differ: ties across threads, waves and workgroups, zeros, rows of infinities and NaN."""
import numpy as np
import pytest
import scipy.linalg.lapack as lapack

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [31, 32, 33, 41, 255, 257, 300, 511, 513, 519, 1023, 1025, 1030, 2049, 2055])
def test_pivots_and_factors(lsx, n):
    print(f"panel n={n}", flush=True)
    A = np.random.default_rng(n).standard_normal((n, n))
    h = lsx._LUHandle(lsx.Context.get(0), n, lsx.LSX_F64)
    assert h.factor(A) == 0
    F, ipiv = h.factors()
    np.testing.assert_array_equal(ipiv, lapack.dgetrf(A)[1] + 1)
    np.testing.assert_array_equal(ipiv, O.dgetrf(A)[1])
    # P A = L U to rounding: |PA - LU| <= n eps |L| |U| entrywise
    L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    PA = A.copy()
    for i, p in enumerate(ipiv - 1):
        PA[[i, p]] = PA[[p, i]]
    bound = 4 * n * np.finfo(float).eps * (np.abs(L) @ np.abs(U)).max()
    assert np.abs(PA - L @ U).max() <= bound


@pytest.mark.parametrize("n", [33, 256, 300, 512, 700, 1024, 1100, 2100])
def test_first_of_equal_magnitudes_wins(lsx, n):
    # A = L U with L unit lower from {-1, 0, 1} and U unit upper from {-1, 0, 1}: every step is exact in
    # integers, every column's largest magnitude is 1, on the diagonal and in about two thirds of the
    # rows below it, and the first (the diagonal) has to win, so that L and U come back exactly.
    rng = np.random.default_rng(n)
    L = np.tril(rng.integers(-1, 2, size=(n, n)), -1) + np.eye(n)
    U = np.triu(rng.integers(-1, 2, size=(n, n)), 1) + np.eye(n)
    h = lsx._LUHandle(lsx.Context.get(0), n, lsx.LSX_F64)
    assert h.factor(L @ U) == 0
    F, ipiv = h.factors()
    np.testing.assert_array_equal(ipiv, np.arange(1, n + 1))
    np.testing.assert_array_equal(F, L - np.eye(n) + U)


@pytest.mark.parametrize("n", [100, 700, 1500])
def test_infinite_row_reaches_only_the_rows_eliminated_with_it(lsx, n):
    # An infinite entry wins its column's search; rows finished before it keep their finite values (an
    # update with multiplier zero would make them NaN), as in LAPACK.
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A[:, :5] *= 10.0
    r = n - 3
    A[r, 7] = np.inf
    h = lsx._LUHandle(lsx.Context.get(0), n, lsx.LSX_F64)
    h.factor(A)
    F, ipiv = h.factors()
    with np.errstate(all="ignore"):
        lu, piv, _ = lapack.dgetrf(A)
    np.testing.assert_array_equal(ipiv[:8], piv[:8] + 1)
    np.testing.assert_array_equal(np.isfinite(F[:7]), np.isfinite(lu[:7]))
    assert np.isfinite(F[:7]).all()
