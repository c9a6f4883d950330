"""SimpleGMRES on a graded spectrum, where the basis visibly loses orthogonality and the Gram-Schmidt
corrections between basis vectors carry the solution: more than 64 vectors (unknowns of the second block
of the triangular Gram-Schmidt system) with 256, 512 and 1024 threads per workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graded(N, seed, large=65, top=9, width=0.27):
    """Eigenvalues: `large` of them from 1 to 10^top, the others in [1, 1 + width]; in random order.  The
    large ones have the same share of the right-hand side at every order from 4096 on."""
    rng = np.random.default_rng(seed)
    lam = np.concatenate([np.logspace(0, top, large), 1 + width * rng.random(N - large)])
    b = rng.standard_normal(N)
    b[:large] *= max(1.0, np.sqrt(N / 4096))
    p = rng.permutation(N)
    return lam[p], b[p]


def diagonal(lsx, lam):
    N = len(lam)
    return lsx.CSRMatrix(np.arange(N + 1, dtype=np.int32), np.arange(N, dtype=np.int32), lam, (N, N))


def check(lam, b, u):
    # GMRES with modified Gram-Schmidt is backward stable: after its convergence the residual is a few
    # eps ||A|| ||x||.  The same recurrences in numpy leave 0.1 to 2 eps for these spectra, and 50 to 300
    # eps without the terms i % 16 >= 8 of the earlier blocks' contributions.
    r = np.linalg.norm(b - lam * u)
    assert r <= 10 * 2.0**-52 * (lam.max() * np.linalg.norm(u) + np.linalg.norm(b))


@pytest.mark.parametrize("N,memory", [(250, 130), (3000, 130), (300000, 130), (524289, 130), (600001, 128)])
def test_one_solve(lsx, N, memory):
    print(f"graded spectrum N={N} memory={memory}", flush=True)
    lam, b = graded(N, N + memory, 90, 10, 0.1)
    sol = lsx.solve(lsx.LinearProblem(diagonal(lsx, lam), b.copy()), lsx.MI355XSimpleGMRES(restart=True, memory=memory),
                    abstol=0.0, reltol=1e-30, maxiters=memory)
    assert sol.iters == memory
    check(lam, b, sol.u)


@pytest.mark.parametrize("blocksize", [200, 511, 4096, 4097, 8192])
def test_block_diagonal(lsx, blocksize):
    print(f"graded spectrum, blocks of {blocksize}", flush=True)
    parts = [graded(blocksize, 7 * blocksize + i) for i in range(3)]
    lam, b = (np.concatenate([p[i] for p in parts]) for i in (0, 1))
    sol = lsx.solve(lsx.LinearProblem(diagonal(lsx, lam), b.copy()),
                    lsx.MI355XSimpleGMRES(restart=True, memory=70, blocksize=blocksize), abstol=0.0, reltol=1e-30, maxiters=70)
    assert sol.iters == 70
    for i, (lam_i, b_i) in enumerate(parts):
        check(lam_i, b_i, sol.u[i * blocksize:(i + 1) * blocksize])
