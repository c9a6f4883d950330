"""The GMRES kernel at the edges of its launch shapes: threads and rows per workgroup, number of
workgroups (each reading all partial products up to 32, one summing each value beyond), groups of 32
basis vectors, blocks of 64 unknowns of the Gram-Schmidt system, bookkeeping in LDS and HBM, rows with
more entries than the kernel keeps in registers, and both diagonal preconditioners."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def system(N, seed, diag=2.1):
    """A perturbed 1D Laplacian plus a shift (condition number about 4 / (diag - 2)), nonsymmetric:
    neighbours, a weak entry half the matrix away (another workgroup's row) and, on every 7th row, 8
    more weak ones.  Rows sorted by column, no duplicates."""
    rng = np.random.default_rng(seed)
    r = np.arange(N, dtype=np.int64)
    offs = [0, 1, N - 1, N // 2] + [3 * t + 5 for t in range(8)]
    cols = (r[:, None] + np.array(offs)[None, :]) % N
    keep = np.ones((N, len(offs)), dtype=bool)
    keep[:, 4:] = (r % 7 == 0)[:, None]
    vals = -rng.uniform(0.0, 0.002, size=cols.shape)
    vals[:, 0] = diag
    vals[:, 1] = -rng.uniform(0.99, 1.0, size=N)
    vals[:, 2] = -rng.uniform(0.99, 1.0, size=N)
    key = np.where(keep, cols, N + np.arange(len(offs))[None, :])
    order = np.argsort(key, axis=1, kind="stable")
    cols, vals, key = (np.take_along_axis(x, order, axis=1) for x in (cols, vals, key))
    keep = key < N
    keep[:, 1:] &= key[:, 1:] != key[:, :-1]  # small N: two offsets may meet
    rowptr = np.concatenate([[0], np.cumsum(keep.sum(axis=1))]).astype(np.int32)
    return rowptr, cols[keep].astype(np.int32), np.ascontiguousarray(vals[keep]), rng.standard_normal(N)


CASES = [
    # N, memory, restart, steps, right preconditioner
    (1, 5, True, 1, False), (255, 20, True, 30, False), (256, 40, True, 50, True), (257, 40, True, 50, False),
    (513, 70, False, 70, False), (1025, 130, False, 130, False), (16384, 33, True, 40, True),
    (16385, 34, True, 45, False), (65536, 12, True, 20, False), (65537, 12, True, 20, True),
    (262145, 8, True, 12, False), (524289, 7, True, 10, True),
]


@pytest.mark.parametrize("N,memory,restart,steps,right", CASES)
def test_shapes_match_oracle(lsx, N, memory, restart, steps, right):
    # A fixed number of steps (tolerances zero): the iterate, the step count and the estimate are the
    # oracle's.  Each of the at most 130 steps adds a few rounding errors of size eps to vectors of
    # norm 1, and the condition numbers are below 100, so the iterates agree to 100 * 130 * 10 eps
    # = 3e-11 at the worst.
    print(f"gmres shape N={N} memory={memory} restart={restart} right={right}", flush=True)
    rp, ci, v, b = system(N, N, 2.05 if N < 2000 else 2.1)
    S = lsx.CSRMatrix(rp, ci, v, (N, N))
    d = np.random.default_rng(N + 1).uniform(0.9, 1.1, size=N)
    pl, pr = np.sqrt(d), (np.sqrt(d) if right else None)
    steps = min(steps, N)
    sol = lsx.solve(lsx.LinearProblem(S, b.copy()), lsx.MI355XSimpleGMRES(restart=restart, memory=memory), Pl=pl, Pr=pr,
                    abstol=0.0, reltol=1e-13, maxiters=steps)
    ref = O.gmres(rp, ci, v, b, memory=memory, restart=restart, abstol=0.0, reltol=1e-13, maxiters=steps, pl=pl, pr=pr)
    assert sol.iters == ref["iters"] and int(sol.retcode) == ref["retcode"]
    assert np.linalg.norm(sol.u - ref["u"]) <= 3e-11 * np.linalg.norm(ref["u"])


def test_multi_launch_at_its_largest_dimension(lsx):
    # memory = 128 is the most a multi-solve launch takes: 17 workgroups of 512 rows keep the
    # bookkeeping of 128 vectors in LDS and leave no room for basis vectors.  Equal to the plain call.
    N, memory = 8300, 128
    rp, ci, v, b = system(N, 5, 2.05)
    S = lsx.CSRMatrix(rp, ci, v, (N, N))
    srv = lsx.Server(hbm_budget=1 << 30)
    t = srv.submit_gmres(S, b, memory=memory, abstol=0.0, reltol=1e-12, maxiters=140)
    srv.drain()
    r = srv.poll(t)
    srv.close()
    sol = lsx.solve(lsx.LinearProblem(S, b.copy()), lsx.MI355XSimpleGMRES(memory=memory), abstol=0.0, reltol=1e-12, maxiters=140)
    assert r["status"] == 0 and r["iters"] == sol.iters
    np.testing.assert_array_equal(r["x"], sol.u)
