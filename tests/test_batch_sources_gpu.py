"""Batches whose matrices come from device memory (read where they are) and from host memory (copied), of
sizes around the panels (32), the steps (64) and the staged columns (128), and rows interchanged or not."""
import numpy as np
import pytest
import scipy.linalg.lapack as lapack

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 191, 193, 255, 256, 257, 300, 321, 511, 512]


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("where", ["device", "host"])
def test_batch_sources(lsx, dtype, where):
    # Blocks P (1.5 I) + N(0,1) / sqrt(n), P a random permutation (every column interchanges): condition
    # numbers below 20, so x agrees with LAPACK's to 20 n eps * 20 in the max norm.  The matrices are not
    # modified, pivots are LAPACK's, and a second call on other matrices gives the other answers.
    import torch
    sizes = np.array(SIZES + SIZES[::-1], dtype=np.int64)
    h = lsx._BatchHandle(lsx.Context.get(0), sizes, lsx.LSX_F64 if dtype == "fp64" else lsx.LSX_F32)
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        blocks = []
        for n in sizes:
            B = rng.standard_normal((n, n)) / np.sqrt(n)
            B[rng.permutation(n), np.arange(n)] += 1.5 * np.sign(rng.standard_normal(n))
            blocks.append(B)
        packed = np.concatenate([B.ravel(order="F") for B in blocks])
        b = rng.standard_normal(int(sizes.sum()))
        if where == "device":
            A, bb = torch.from_numpy(packed).cuda(), torch.from_numpy(b).cuda()
            x = torch.empty_like(bb)
        else:
            A, bb, x = packed.copy(), b.copy(), np.empty_like(b)
        nfail, info, ipiv = h.factor_solve(A, bb, x, want_pivots=True)
        assert nfail == 0 and not info.any()
        np.testing.assert_array_equal(A.cpu().numpy() if where == "device" else A, packed)
        x = x.cpu().numpy() if where == "device" else x
        off = 0
        for n, B in zip(sizes, blocks):
            lu, piv, _ = lapack.dgetrf(B)
            ref = lapack.dgetrs(lu, piv, b[off:off + n])[0]
            if dtype == "fp64":
                np.testing.assert_array_equal(ipiv[off:off + n], piv + 1, err_msg=f"n={n}")
            assert np.abs(x[off:off + n] - ref).max() <= 400 * max(n, 10) * np.finfo(float).eps * np.abs(ref).max(), n
            off += int(n)
    if dtype == "fp32":
        it, be = h.stats()
        assert (be <= 1e-14).all() and (it <= 10).all()
