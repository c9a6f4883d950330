"""The blocked LU where its outer blocks change width: one last block of up to 3072 rows, blocks of 128
columns above, of 256 above 8192 rows (512 above 10000, FP64); orders whose L interchanges are not deferred (above 18432); and FP32 panels of up
to 2048 rows in one workgroup."""
import numpy as np
import pytest
import scipy.linalg.lapack as lapack
import torch

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n", [3071, 3072, 3073, 3201, 4099, 8193, 8450, 10001])
def test_factors_across_block_widths(lsx, n):
    print(f"blocks n={n}", flush=True)
    A = np.random.default_rng(n).standard_normal((n, n))
    h = lsx._LUHandle(lsx.Context.get(0), n, lsx.LSX_F64)
    assert h.factor(A) == 0
    F, ipiv = h.factors()
    if n <= 4099:
        np.testing.assert_array_equal(ipiv, lapack.dgetrf(A)[1] + 1)
    rows = np.arange(n)
    for i, p in enumerate(ipiv - 1):
        rows[[i, p]] = rows[[p, i]]
    F = torch.from_numpy(np.ascontiguousarray(F)).cuda()
    L, U = torch.tril(F, -1) + torch.eye(n, dtype=F.dtype, device="cuda"), torch.triu(F)
    PA = torch.from_numpy(A[rows]).cuda()
    # |PA - LU| <= n eps |L| |U| entrywise, with the product's own rounding formed here
    assert (PA - L @ U).abs().max() <= 4 * n * EPS * (L.abs() @ U.abs()).max()


@pytest.mark.parametrize("n,dtype", [(1025, "f32"), (2048, "f32"), (2049, "f32"), (3073, "f32"), (8200, "f32"), (8200, "bf16"), (18560, "f64")])
def test_solves_across_block_widths(lsx, n, dtype):
    print(f"blocks solve n={n} {dtype}", flush=True)
    rng = np.random.default_rng(n)
    A = rng.random((n, n)) - 0.5
    A[np.arange(n), rng.permutation(n)] += 4.0 * np.sqrt(n)  # well conditioned, rows in random order
    b = rng.standard_normal(n)
    h = lsx._LUHandle(lsx.Context.get(0), n, {"f64": lsx.LSX_F64, "f32": lsx.LSX_F32, "bf16": lsx.LSX_BF16}[dtype])
    assert h.factor(A) == 0
    x = np.zeros(n)
    if dtype == "f64":
        h.solve(b, x)
    else:
        h.refine(b, x, 1e-13, 20, 0)
    r = np.abs(b - A @ x).max()
    assert r <= (4 * n * EPS if dtype == "f64" else 2e-13) * (np.abs(A).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max())
