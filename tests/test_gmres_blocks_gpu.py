"""Block-diagonal SimpleGMRES with more blocks than CUs, where several blocks' workgroups share a CU: block
sizes around 256, 512 and 1024 rows, Krylov dimensions whose bookkeeping leaves room for three, two or one
workgroup to a CU."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,memory", [(3, 60), (256, 20), (257, 20), (512, 5), (512, 75), (512, 128), (513, 20), (1024, 60),
                                      (1024, 128), (1025, 10)])
def test_many_blocks(lsx, n, memory):
    # Four different right-hand sides in turn: equal blocks give equal bits, and the four are the
    # oracle's.  A fixed number of steps (tolerances zero) with a perturbed 1D Laplacian plus a shift
    # (condition number below 100): each of the at most 130 steps adds a few rounding errors of size eps to
    # vectors of norm 1, so the iterates agree to 100 * 130 * 10 eps = 3e-11 at the worst.
    print(f"many blocks n={n} memory={memory}", flush=True)
    nb = 600
    steps = min(memory + 2, n)
    rng = np.random.default_rng(1000 * n + memory)
    r = np.arange(n)
    cols = np.stack([r - 1, r, r + 1], 1)
    keep = (cols >= 0) & (cols < n)
    vals = np.stack([-rng.uniform(0.99, 1.0, n), np.full(n, 2.1), -rng.uniform(0.99, 1.0, n)], 1)
    rp = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int64)
    ci, v, nnz = cols[keep], np.ascontiguousarray(vals[keep]), int(rp[-1])
    b = rng.standard_normal((4, n))
    rowptr = np.concatenate([(rp[None, :-1] + nnz * np.arange(nb)[:, None]).ravel(), [nb * nnz]]).astype(np.int32)
    colind = (ci[None, :] + n * np.arange(nb)[:, None]).ravel().astype(np.int32)
    A = lsx.CSRMatrix(rowptr, colind, np.tile(v, nb), (n * nb, n * nb))
    sol = lsx.solve(lsx.LinearProblem(A, np.tile(b, (nb // 4, 1)).ravel()),
                    lsx.MI355XSimpleGMRES(restart=True, memory=memory, blocksize=n), abstol=0.0, reltol=1e-30, maxiters=steps)
    u = sol.u.reshape(nb // 4, 4, n)
    assert sol.iters == steps
    np.testing.assert_array_equal(u, np.broadcast_to(u[:1], u.shape))
    for i in range(4):
        ref = O.gmres(rp.astype(np.int32), ci.astype(np.int32), v, b[i], memory=memory, restart=True, abstol=0.0,
                      reltol=1e-30, maxiters=steps)
        assert np.linalg.norm(u[0, i] - ref["u"]) <= 3e-11 * np.linalg.norm(ref["u"])
