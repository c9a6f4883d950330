"""BF16 factors: the products inside a block are BF16 products too (two pieces per operand), at the edges of
the 64 x 64 tiles and of the block widths, and a refined solve is as accurate as its refinement steps make it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 64, 65, 96, 97, 161, 500, 3072, 3073, 3300])
def test_factors(lsx, n):
    # scaled residual ||PA - LU|| / (||L|| ||U|| n u) < 20 with the unit u = 2^-16 of two BF16 pieces, as for
    # LAPACK's factors with u = eps.  The factors are not the FP32 ones: every order with a second panel
    # has BF16 products.
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    f = {}
    for dt in (lsx.LSX_F32, lsx.LSX_BF16):
        h = lsx._LUHandle(lsx.Context.get(0), n, dt)
        assert h.factor(A) == 0
        F, ipiv = h.factors()
        f[dt] = F
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        p = np.arange(n)
        for k in range(n):
            j = ipiv[k] - 1
            p[k], p[j] = p[j], p[k]
        u = 2.0**-24 if dt == lsx.LSX_F32 else 2.0**-16
        R = np.abs(A[p] - L @ U).sum(0).max()
        assert R < 20 * n * u * np.abs(L).sum(0).max() * np.abs(U).sum(0).max()
    assert not np.array_equal(f[lsx.LSX_F32], f[lsx.LSX_BF16])


@pytest.mark.parametrize("n", [300, 1000, 3072, 4500])
def test_refined_error(lsx, n):
    # A = 1.25 P + G / sqrt(n) (condition number about 10, growth below 10).  BF16 factors have a relative
    # error of about 2^-16, so the first step leaves a backward error of about 2^-32 > tol and the second one
    # of a few eps; the forward error is then a few tens of eps.
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) / np.sqrt(n)
    A[rng.permutation(n), np.arange(n)] += 1.25
    b = rng.standard_normal(n)
    sol = lsx.solve(lsx.LinearProblem(A, b), lsx.MI355XMixedLUFactorization(precision="bf16"))
    x = np.linalg.solve(A, b)
    x += np.linalg.solve(A, b - A @ x)
    assert sol.retcode == lsx.ReturnCode.Success and sol.iters == 2
    assert np.linalg.norm(sol.u - x) <= 100 * 2.0**-52 * np.linalg.norm(x)
