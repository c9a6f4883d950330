"""The workloads this framework's speed is measured on: dense LU solves, re-solves with resident
factors, mixed-precision solves, batches of small systems and SimpleGMRES, each
called as a program calls it (the LinearProblem / init / solve_ interface, or the C entry points
of include/lsx.h on device arrays) with the handles such a program keeps.

listed() are the cases, draw(rng) gives more of the same ranges, prepare/run/work/exact are what a
measurement calls.  The matrices have their rows in random order, so that partial pivoting
interchanges rows in almost every column, and are well conditioned, so that two correct solvers
agree to rounding.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def _package():
    name = "linearsolve_jl_amd"  # the folder's own name holds a dot
    if name not in sys.modules:
        d = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linearsolve.jl_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


DEV = "cuda:0"
ABSTOL = math.sqrt(np.finfo(np.float64).eps)  # the framework's default tolerance


def listed():
    return [
        # one small dense solve inside a larger program (an implicit step, a Newton solve): latency
        dict(name="lu_100", kind="lu", n=100, nrhs=1, order="C"),
        # the size of the repository's CPU comparison, a new matrix on every call
        dict(name="lu_1024", kind="lu", n=1024, nrhs=1, order="C"),
        # a ragged order in between, a few right-hand sides
        dict(name="lu_3001_5rhs", kind="lu", n=3001, nrhs=5, order="F"),
        # the headline benchmark: factor and solve 16 right-hand sides
        dict(name="lu_16384_16rhs", kind="lu", n=16384, nrhs=16, order="F"),
        # resident factors, a new right-hand side per call: one solve and one adjoint solve
        # (sensitivities, adjoint time stepping)
        dict(name="resolve_6000", kind="resolve", n=6000, nrhs=1),
        # low-precision factorization, refined to FP64 accuracy
        dict(name="mixed_fp32_9000", kind="mixed", n=9000, precision="fp32"),
        # the batched benchmark: 20,000 systems of n in [8, 512], FP64
        dict(name="batch_fp64_20000", kind="batch", count=20000, nmin=8, nmax=512, dtype="fp64", permuted=False),
        # a smaller batch, FP32 factors with FP64 refinement, interchanges in every column
        dict(name="batch_fp32_3000", kind="batch", count=3000, nmin=8, nmax=512, dtype="fp32", permuted=True),
        # SimpleGMRES on the convection-diffusion benchmark: a small grid run to its tolerance ...
        dict(name="gmres_100", kind="gmres", m=100, pe=5.0, memory=30, restart=True, maxiters=10000),
        # ... and the large grid for the benchmark's 300 Arnoldi steps
        dict(name="gmres_1024", kind="gmres", m=1024, pe=5.0, memory=30, restart=True, maxiters=300),
        # one GMRES per diagonal block
        dict(name="gmres_batched_4096", kind="gmres_batched", blocks=4096, m=16, memory=20),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lu", "lu", "lu", "resolve", "mixed", "batch", "batch", "gmres", "gmres", "gmres_batched"])
    if kind == "lu":
        return dict(kind=kind, n=_logint(rng, 16, 12000), nrhs=rng.choice([1, 1, 3, 16, 37]), order=rng.choice("CF"))
    if kind == "resolve":
        return dict(kind=kind, n=_logint(rng, 64, 12000), nrhs=rng.choice([1, 1, 2, 16]))
    if kind == "mixed":
        return dict(kind=kind, n=_logint(rng, 300, 14000), precision=rng.choice(["fp32", "fp32", "bf16"]))
    if kind == "batch":
        nmin, nmax = rng.choice([(8, 512), (8, 64), (8, 200), (100, 300), (256, 512)])
        return dict(kind=kind, count=_logint(rng, 50, 6000), nmin=nmin, nmax=nmax,
                    dtype=rng.choice(["fp64", "fp32"]), permuted=rng.random() < 0.5)
    if kind == "gmres":
        restart = rng.random() < 0.8
        m = _logint(rng, 16, 900 if restart else 300)
        return dict(kind=kind, m=m, pe=round(rng.uniform(0.0, 10.0), 2), memory=rng.choice([10, 20, 30, 50]),
                    restart=restart, maxiters=rng.choice([60, 150, 300] if restart else [40, 100, 150]))
    return dict(kind=kind, blocks=_logint(rng, 50, 5000), m=rng.randint(4, 20), memory=rng.choice([10, 20, 30]))


# ---- inputs --------------------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + salt)
    return g


def _dense(n, seed):
    """1.25 P + G / sqrt(n): G iid N(0,1), P a random permutation."""
    g = _gen(seed, 1)
    A = torch.randn(n, n, dtype=torch.float64, device=DEV, generator=g).div_(math.sqrt(n))
    p = torch.randperm(n, device=DEV, generator=g)
    A[p, torch.arange(n, device=DEV)] += 1.25
    return A


def _rhs(n, nrhs, seed, salt=2):
    b = torch.randn(nrhs, n, dtype=torch.float64, device=DEV, generator=_gen(seed, salt))
    return b[0].contiguous() if nrhs == 1 else b.t()


def _batch_sizes(case):
    # fixed by the case, as a program's batch structure is; the values change from seed to seed
    r = np.random.default_rng([case["count"], case["nmin"], case["nmax"]])
    return r.integers(case["nmin"], case["nmax"] + 1, size=case["count"]).astype(np.int64)


def _batch_inputs(case, seed):
    """Packed column-major blocks P_i - g_i J_i, J iid N(0,1)/sqrt(n_i), g_i ~ U[1e-3, 1e-1], P_i the
    identity or a random permutation, and their right-hand sides."""
    sizes = _batch_sizes(case)
    g = _gen(seed, 3)
    ns = torch.from_numpy(sizes).to(DEV)
    total = int((sizes * sizes).sum())
    A = torch.randn(total, dtype=torch.float64, device=DEV, generator=g)
    gam = torch.rand(len(sizes), dtype=torch.float64, device=DEV, generator=g) * (1e-1 - 1e-3) + 1e-3
    offs = torch.from_numpy(np.concatenate([[0], np.cumsum(sizes * sizes)[:-1]])).to(DEV)
    scale = -gam / ns.double().sqrt()
    A *= torch.repeat_interleave(scale, ns * ns, output_size=total)
    nv = int(sizes.sum())
    voff = torch.from_numpy(np.concatenate([[0], np.cumsum(sizes)[:-1]])).to(DEV)
    sysid = torch.repeat_interleave(torch.arange(len(sizes), device=DEV), ns, output_size=nv)
    col = torch.arange(nv, device=DEV) - voff[sysid]
    row = col
    if case["permuted"]:
        key = sysid.double() + torch.rand(nv, dtype=torch.float64, device=DEV, generator=g)
        row = torch.argsort(key) - voff[sysid]
    A[offs[sysid] + col * ns[sysid] + row] += 1.0
    b = torch.randn(nv, dtype=torch.float64, device=DEV, generator=g)
    return sizes, A, b


def _stencil(m, pe):
    """CSR of the 5-point convection-diffusion grid (row = i + m j, columns ascending), on the GPU."""
    N, h = m * m, 1.0 / (m + 1)
    lo, hi = -1.0 - pe * h / 2.0, -1.0 + pe * h / 2.0
    r = torch.arange(N, device=DEV)
    i, j = r % m, r // m
    cols = torch.stack([r - m, r - 1, r, r + 1, r + m], 1)
    keep = torch.stack([j > 0, i > 0, j >= 0, i < m - 1, j < m - 1], 1)
    vals = torch.tensor([lo, lo, 4.0, hi, hi], dtype=torch.float64, device=DEV).expand(N, 5)
    rowptr = torch.zeros(N + 1, dtype=torch.int32, device=DEV)
    rowptr[1:] = keep.sum(1).cumsum(0)
    return rowptr, cols[keep].to(torch.int32), vals[keep].contiguous()


def _block_pe(case):
    return [float(k % 10) for k in range(case["blocks"])]


def _blocks_csr(case):
    """Block-diagonal CSR of m x m grids, the Peclet number cycling through 0..9."""
    m, nb = case["m"], case["blocks"]
    n = m * m
    parts = [_stencil(m, float(p)) for p in range(10)]
    nnz = parts[0][1].numel()
    k = torch.arange(nb, device=DEV)
    vals = torch.stack([p[2] for p in parts])[k % 10].reshape(-1).contiguous()
    col = (parts[0][1].long()[None, :] + (k * n)[:, None]).reshape(-1).to(torch.int32)
    rowptr = torch.empty(nb * n + 1, dtype=torch.int32, device=DEV)
    rowptr[:-1] = (parts[0][0][:-1].long()[None, :] + (k * nnz)[:, None]).reshape(-1).to(torch.int32)
    rowptr[-1] = nb * nnz
    return rowptr, col, vals


# ---- the framework's handles ---------------------------------------------------------------------

class _Csr:
    """A lsx_csr handle of the C interface, made from device arrays."""

    def __init__(self, rowptr, col, vals):
        lsx = _package()
        self.ctx, self.L = lsx.Context.get(0), lsx._abi.lib()
        self.h = ctypes.c_void_p()
        torch.cuda.synchronize()
        self.ctx.check(self.L.lsx_csr_create(self.ctx.handle, rowptr.numel() - 1, vals.numel(), rowptr.data_ptr(),
                                             col.data_ptr(), vals.data_ptr(), ctypes.byref(self.h)), "lsx_csr_create")

    def __del__(self):
        if self.h.value:
            self.L.lsx_csr_destroy(self.h)


class _Batch:
    """A lsx_batch handle of the C interface, with the committed tile table."""

    def __init__(self, sizes, dtype):
        lsx = _package()
        self.ctx, self.L = lsx.Context.get(0), lsx._abi.lib()
        self.h = ctypes.c_void_p()
        dt = lsx._abi.LSX_F64 if dtype == "fp64" else lsx._abi.LSX_F32
        self.ctx.check(self.L.lsx_batch_create(self.ctx.handle, len(sizes), sizes.ctypes.data, dt,
                                               ctypes.byref(self.h)), "lsx_batch_create")
        table = lsx.load_tile_table(dtype=dt)
        if table:
            up = np.array([u for u, _ in table], dtype=np.int32)
            bw = np.array([w for _, w in table], dtype=np.int32)
            self.ctx.check(self.L.lsx_batch_set_tiles(self.h, len(up), up.ctypes.data, bw.ctypes.data),
                           "lsx_batch_set_tiles")

    def __del__(self):
        if self.h.value:
            self.L.lsx_batch_destroy(self.h)


def prepare(case, seed):
    lsx, kind = _package(), case["kind"]
    if kind in ("lu", "mixed", "resolve"):
        n, nrhs = case["n"], case.get("nrhs", 1)
        A = _dense(n, seed)
        if case.get("order", "F") == "F":
            A = A.t()  # column-major storage (the transpose of one draw is another)
        b = _rhs(n, nrhs, seed)
        alg = (lsx.MI355XMixedLUFactorization(precision=case["precision"]) if kind == "mixed"
               else lsx.MI355XLUFactorization())
        cache = lsx.init(lsx.LinearProblem(A, b), alg, alias_A=True, alias_b=True)
        if kind == "resolve":
            lsx.solve_(cache)
            b = _rhs(n, nrhs, seed, 4)
        return dict(kind=kind, cache=cache, A=A, b=b)
    if kind == "batch":
        sizes, A, b = _batch_inputs(case, seed)
        return dict(kind=kind, h=_Batch(sizes, case["dtype"]), A=A, b=b, x=torch.empty_like(b),
                    ipiv=torch.zeros(b.numel(), dtype=torch.int64, device=DEV),
                    info=np.zeros(len(sizes), dtype=np.int64))
    if kind == "gmres":
        rowptr, col, vals = _stencil(case["m"], case["pe"])
        N = case["m"] ** 2
        return dict(kind=kind, case=case, h=_Csr(rowptr, col, vals), b=_rhs(N, 1, seed),
                    x=torch.empty(N, dtype=torch.float64, device=DEV),
                    pl=torch.full((N,), 4.0, dtype=torch.float64, device=DEV), st=lsx._abi.GmresStats())
    N = case["m"] ** 2 * case["blocks"]
    return dict(kind=kind, case=case, h=_Csr(*_blocks_csr(case)), b=_rhs(N, 1, seed),
                x=torch.empty(N, dtype=torch.float64, device=DEV),
                pl=torch.full((N,), 4.0, dtype=torch.float64, device=DEV), st=lsx._abi.GmresStats())


def run(s):
    lsx, kind = _package(), s["kind"]
    if kind in ("lu", "mixed"):
        cache = s["cache"]
        cache.A = s["A"]
        cache.b = s["b"]
        sol = lsx.solve_(cache)
        return {"x": sol.u, "retcode": int(sol.retcode)}
    if kind == "resolve":
        cache = s["cache"]
        cache.b = s["b"]
        x = lsx.solve_(cache).u.clone()
        return {"x": x, "xt": lsx.solve_(cache, adjoint=True).u}
    h = s.get("h")
    if kind == "batch":
        torch.cuda.current_stream().synchronize()
        nfail = h.ctx.check(h.L.lsx_batch_factor_solve(h.h, s["A"].data_ptr(), s["b"].data_ptr(), s["x"].data_ptr(),
                                                       s["info"].ctypes.data, s["ipiv"].data_ptr()),
                            "lsx_batch_factor_solve")
        return {"x": s["x"], "ipiv": s["ipiv"], "info": s["info"], "failed": nfail}
    if kind == "gmres":
        c = s["case"]
        torch.cuda.current_stream().synchronize()
        h.ctx.check(h.L.lsx_gmres_solve(h.h, s["b"].data_ptr(), s["x"].data_ptr(), c["memory"], int(c["restart"]),
                                        ABSTOL, 1e-8, c["maxiters"], s["pl"].data_ptr(), None,
                                        ctypes.byref(s["st"])), "lsx_gmres_solve")
        return {"x": s["x"], "iters": int(s["st"].iters), "retcode": int(s["st"].retcode)}
    c = s["case"]
    torch.cuda.current_stream().synchronize()
    h.ctx.check(h.L.lsx_gmres_solve_batched(h.h, c["m"] ** 2, s["b"].data_ptr(), s["x"].data_ptr(), c["memory"], 1,
                                            ABSTOL, 1e-8, 1000, s["pl"].data_ptr(), None, ctypes.byref(s["st"])),
                "lsx_gmres_solve_batched")
    return {"x": s["x"], "iters": int(s["st"].iters), "retcode": int(s["st"].retcode)}


# ---- what a pass cannot do without ---------------------------------------------------------------

def _luflop(n):
    return n + n * (n - 1) / 2 + (n - 1) * n * (2 * n - 1) / 3


def _gmres_work(N, nnz, steps, memory):
    """Matrix and vectors once; per Arnoldi step the sparse product and k Gram-Schmidt projections."""
    kavg = (min(memory, steps) + 1) / 2
    return 12 * nnz + 4 * N + 8 * 3 * N, steps * (2 * nnz + N * (4 * kavg + 6))


def work(case):
    kind = case["kind"]
    if kind in ("lu", "mixed"):
        n, r = case["n"], case.get("nrhs", 1)
        return {"bytes": 8 * (n * n + 2 * n * r), "flops": _luflop(n) + 2.0 * n * n * r}
    if kind == "resolve":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 2 * 8 * (n * n + 2 * n * r), "flops": 2 * 2.0 * n * n * r}
    if kind == "batch":
        n = _batch_sizes(case).astype(np.float64)
        return {"bytes": float((8 * (n * n + 3 * n)).sum()), "flops": float((_luflop(n) + 2 * n * n).sum())}
    if kind == "gmres":
        N = case["m"] ** 2
        memory = case["memory"] if case["restart"] else case["maxiters"]
        steps = min(case["maxiters"], 8 * case["m"])  # small grids stop at their tolerance
        b, f = _gmres_work(N, 5 * N, steps, memory)
        return {"bytes": b, "flops": f}
    N = case["m"] ** 2 * case["blocks"]
    b, f = _gmres_work(N, 5 * N, 4 * case["m"], case["memory"])
    return {"bytes": b, "flops": f}


# ---- the same results in 64 bits by plain torch and numpy ----------------------------------------

def _plain_solve(A, b):
    A, b = A.cpu(), b.cpu()
    return torch.linalg.solve(A, b if b.dim() == 2 else b[:, None]).reshape(b.shape)


def _plain_gmres(b, m, pes, memory, restart, maxiters, eps=None):
    """Restarted GMRES with Jacobi on one grid per row of b (k x m^2), the grids independent;
    returns the iterates.  eps: the stopping bound of every grid (default: from its own norm)."""
    k, N = b.shape
    h = 1.0 / (m + 1)
    pe = torch.as_tensor(pes, dtype=torch.float64, device=b.device).reshape(k, 1, 1)
    lo, hi = -1.0 - pe * h / 2.0, -1.0 + pe * h / 2.0

    def mul(x):
        X = x.reshape(k, m, m)
        Y = 4.0 * X
        Y[:, 1:] += lo * X[:, :-1]
        Y[:, :, 1:] += lo * X[:, :, :-1]
        Y[:, :, :-1] += hi * X[:, :, 1:]
        Y[:, :-1] += hi * X[:, 1:]
        return Y.reshape(k, N)

    x = torch.zeros_like(b)
    beta = (b / 4.0).norm(dim=1)
    eps = ABSTOL + 1e-8 * beta if eps is None else torch.full_like(beta, eps)
    done, it = beta <= eps, 0
    cap = memory if restart else maxiters
    while it < maxiters and not bool(done.all()):
        r = (b - mul(x)) / 4.0
        beta = r.norm(dim=1)
        V = torch.zeros(cap + 1, k, N, dtype=torch.float64, device=b.device)
        V[0] = r / beta[:, None]
        R = torch.zeros(k, cap, cap, dtype=torch.float64, device=b.device)
        z = torch.zeros(k, cap + 1, dtype=torch.float64, device=b.device)
        z[:, 0] = beta
        cs, sn = [], []
        used = torch.zeros(k, dtype=torch.long, device=b.device)
        for j in range(cap):
            q = mul(V[j]) / 4.0
            col = []
            for i in range(j + 1):
                c = (V[i] * q).sum(1)
                q = q - c[:, None] * V[i]
                col.append(c)
            hb = q.norm(dim=1)
            for i in range(j):
                col[i], col[i + 1] = cs[i] * col[i] + sn[i] * col[i + 1], sn[i] * col[i] - cs[i] * col[i + 1]
            rho = torch.hypot(col[j], hb)
            cs.append(col[j] / rho)
            sn.append(hb / rho)
            col[j] = rho
            R[:, : j + 1, j] = torch.stack(col, 1)
            z[:, j + 1] = sn[j] * z[:, j]
            z[:, j] = cs[j] * z[:, j]
            used = torch.where(done, used, torch.full_like(used, j + 1))
            it += 1
            done = done | (z[:, j + 1].abs() <= eps)
            if it >= maxiters or bool(done.all()):
                break
            V[j + 1] = q / hb[:, None]
        n = j + 1
        on = torch.arange(n, device=b.device)[None, :] < used[:, None]
        Rn = torch.where(on[:, None, :] & on[:, :, None], R[:, :n, :n], torch.zeros_like(R[:, :n, :n]))
        Rn = Rn + torch.diag_embed((~on).double())
        y = torch.linalg.solve_triangular(Rn, torch.where(on, z[:, :n], torch.zeros_like(z[:, :n]))[:, :, None],
                                          upper=True)[:, :, 0]
        for i in range(n):
            x = x + y[:, i: i + 1] * V[i]
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lu", "mixed", "resolve"):
        A = _dense(case["n"], seed)
        if case.get("order", "F") == "F":
            A = A.t()
        b = _rhs(case["n"], case.get("nrhs", 1), seed, 4 if kind == "resolve" else 2)
        if kind == "resolve":
            return {"x": _plain_solve(A, b), "xt": _plain_solve(A.t(), b)}
        return {"x": _plain_solve(A, b), "retcode": None}
    if kind == "batch":
        sizes, A, b = _batch_inputs(case, seed)
        A, b = A.cpu().numpy(), b.cpu().numpy()
        ao = np.concatenate([[0], np.cumsum(sizes * sizes)])
        vo = np.concatenate([[0], np.cumsum(sizes)])
        x = np.empty_like(b)
        for i, n in enumerate(sizes):
            B = A[ao[i]: ao[i + 1]].reshape(n, n).T
            x[vo[i]: vo[i + 1]] = np.linalg.solve(B, b[vo[i]: vo[i + 1]])
        return {"x": x, "ipiv": None, "info": None, "failed": None}
    if kind == "gmres":
        b = _rhs(case["m"] ** 2, 1, seed)
        x = _plain_gmres(b[None, :], case["m"], [case["pe"]], case["memory"], case["restart"], case["maxiters"])
        return {"x": x[0], "iters": None, "retcode": None}
    n, nb = case["m"] ** 2, case["blocks"]
    b = _rhs(n * nb, 1, seed)
    eps = ABSTOL + 1e-8 * float((b / 4.0).norm())
    x = _plain_gmres(b.reshape(nb, n), case["m"], _block_pe(case), case["memory"], True, 1000, eps)
    return {"x": x.reshape(-1), "iters": None, "retcode": None}
