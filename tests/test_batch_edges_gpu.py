"""Batched LU at the sizes where a panel's rows go from one wave to several, where a thread's second rows
begin, and where the last panel is narrow: LAPACK's pivots and info, and FP32 factors refined to the target,
with a zero column in some of the systems."""
import numpy as np
import pytest
import scipy.linalg.lapack as lapack

from conftest import backward_error

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 24, 25, 31, 32, 33, 40, 63, 64, 65, 72, 95, 96, 97, 127, 128, 129, 160, 161, 193, 255, 256, 257, 288,
         289, 319, 320, 321, 352, 353, 449, 481, 505]


def systems(seed):
    rng = np.random.default_rng(seed)
    blocks = [rng.standard_normal((n, n)) for n in SIZES for _ in range(2)]
    zero = {}
    for i, B in enumerate(blocks):
        if i % 2:  # every second one: a zero column (LAPACK's info is its number), the last for some
            c = B.shape[0] - 1 if i % 4 == 1 else int(rng.integers(0, B.shape[0]))
            B[:, c] = 0.0
            zero[i] = c + 1
    return blocks, rng.standard_normal(sum(B.shape[0] for B in blocks)), zero


def test_pivots_and_info(lsx):
    blocks, b, zero = systems(11)
    alg = lsx.MI355XBatchedLUFactorization()
    sol = lsx.solve(lsx.LinearProblem(lsx.BlockDiagonal(blocks), b), alg)
    off = 0
    for i, B in enumerate(blocks):
        n = B.shape[0]
        lu, piv, info = lapack.dgetrf(B)
        assert alg.last_info[i] == info == zero.get(i, 0), f"block {i} n={n}"
        # after a zero pivot the rows below it are exact zeros in that column on both sides; the other
        # columns' pivots agree
        np.testing.assert_array_equal(alg.last_ipiv[off:off + n], piv + 1, err_msg=f"block {i} n={n}")
        if info == 0:
            assert backward_error(B, sol.u[off:off + n], b[off:off + n]) <= 1e-13, f"block {i} n={n}"
        off += n


def test_fp32_refined_and_info(lsx):
    blocks, b, zero = systems(12)
    alg = lsx.MI355XBatchedLUFactorization(precision="fp32", tol=1e-14)
    sol = lsx.solve(lsx.LinearProblem(lsx.BlockDiagonal(blocks), b), alg)
    off = 0
    for i, B in enumerate(blocks):
        n = B.shape[0]
        assert alg.last_info[i] == zero.get(i, 0), f"block {i} n={n}"
        if i in zero:
            assert alg.last_iters[i] == 0, f"block {i} n={n}"  # no refinement of a singular system
        else:
            # the kernel's own residual met 1e-14; one summed in another order may differ in the last bits
            assert backward_error(B, sol.u[off:off + n], b[off:off + n]) <= 2e-14, f"block {i} n={n}"
        off += n
