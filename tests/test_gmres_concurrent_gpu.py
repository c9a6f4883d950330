"""Plain SimpleGMRES solves from several host threads at once, each on its own handle, alone and beside a
serving loop: together they ask for more workgroups than the GPU has CUs.  Every solve ends, with the
bits it has alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def grid(lsx, m, pe=5.0):
    """5-point convection-diffusion on an m x m grid, as the serving loop generates it."""
    N = m * m
    h = 1.0 / (m + 1)
    lo, hi = -1.0 - pe * h / 2, -1.0 + pe * h / 2
    r = np.arange(N)
    i, j = r % m, r // m
    cols = np.stack([r - m, r - 1, r, r + 1, r + m], 1)
    keep = np.stack([j > 0, i > 0, j >= 0, i < m - 1, j < m - 1], 1)
    vals = np.broadcast_to(np.array([lo, lo, 4.0, hi, hi]), (N, 5))
    rowptr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return lsx.CSRMatrix(rowptr, cols[keep].astype(np.int32), np.ascontiguousarray(vals[keep]), (N, N))


def run(lsx, cache, reps):
    out = None
    for _ in range(reps):
        out = lsx.solve_(cache)
    return out.u.copy(), out.iters


@pytest.mark.parametrize("sides", [(700, 700, 700), (1024, 512, 300, 90, 64, 700)])
def test_threads_get_the_bits_of_a_lone_solve(lsx, sides):
    rng = np.random.default_rng(len(sides))
    caches = []
    for m in sides:
        b = rng.standard_normal(m * m)
        caches.append(lsx.init(lsx.LinearProblem(grid(lsx, m), b), lsx.MI355XSimpleGMRES(restart=True, memory=20),
                               Pl=np.full(m * m, 4.0), abstol=0.0, reltol=1e-14, maxiters=60))
    alone = [run(lsx, c, 1) for c in caches]
    got = [None] * len(caches)

    def work(i):
        got[i] = run(lsx, caches[i], 4)

    print(f"concurrent solves {sides}", flush=True)
    th = [threading.Thread(target=work, args=(i,)) for i in range(len(caches))]
    [t.start() for t in th]
    [t.join() for t in th]
    for (u, it), (v, jt) in zip(alone, got):
        assert it == jt == 60
        np.testing.assert_array_equal(u, v)


def test_beside_a_serving_loop(lsx):
    m = 700
    b = np.random.default_rng(7).standard_normal(m * m)
    cache = lsx.init(lsx.LinearProblem(grid(lsx, m), b), lsx.MI355XSimpleGMRES(restart=True, memory=20),
                     Pl=np.full(m * m, 4.0), abstol=0.0, reltol=1e-14, maxiters=60)
    u, _ = run(lsx, cache, 1)
    srv = lsx.Server(hbm_budget=8 << 30)
    print("solves beside a serving loop", flush=True)
    tickets = [srv.submit_gmres_synth(s, 5.0, k + 1, memory=20, maxiters=60) for k, s in enumerate((700, 600, 700, 90, 500, 64) * 2)]
    dense = [srv.submit_dense_synth(n, n) for n in (1500, 700, 3000, 100)]
    got = [run(lsx, cache, 1)[0] for _ in range(8)]
    srv.drain()
    for t in tickets + dense:
        assert srv.poll(t)["status"] == 0
    srv.close()
    for v in got:
        np.testing.assert_array_equal(u, v)
