// gmres.hip — SimpleGMRES (restarted GMRES, modified Gram-Schmidt Arnoldi, symmetric Givens) on a
// CSR matrix: the launches of the persistent kernel (gmres_kernel.hpp) for one solve, for several
// solves at once and for block-diagonal matrices, and their C entry points.
#include <algorithm>
#include <new>
#include <vector>

#include "gmres_kernel.hpp"

namespace lsx {

template <int NT, int RPT, bool RG>
__global__ __launch_bounds__(NT, NT == 1024 ? 4 : (NT == 256 ? 3 : 2)) void k_gmres(GmresArgs a) {
    __shared__ GShared<NT> sh;
    extern __shared__ __align__(16) double dyn[];
    GmresWg<NT, RPT, RG> g(a, sh, (int)blockIdx.x, dyn);
    g.run();
}

// Several solves in one launch (gmres_launch_multi), on a pool of workgroups that may be smaller
// than the solves' total: a workgroup takes the next number from a counter, runs that rank of
// its solve, and takes another number when the solve ends.  Numbers go out in start order, so
// every solve but the one holding the highest number handed out so far has all its ranks
// running and finishes by itself; with at least as many workgroups as the widest solve, that
// last one fills up as the others end.
template <int NT, int RPT, bool MR = (RPT <= 4)>
__global__ __launch_bounds__(NT, NT == 256 ? 3 : NT == 1024 || (RPT == 2 && !MR) ? 4 : 2) void k_gmres_multi(const GmresArgs* __restrict items,
                                                                       const int* __restrict first, int nitems,
                                                                       uint32_t* ticket) {
    __shared__ GShared<NT> sh;
    __shared__ int s_id;
    extern __shared__ __align__(16) double dyn[];
    const int total = first[nitems];
    while (true) {
        __syncthreads();  // the previous solve's LDS is no longer read
        if (threadIdx.x == 0) s_id = (int)atomicAdd(ticket, 1u);
        __syncthreads();
        const int id = __builtin_amdgcn_readfirstlane(s_id);
        if (id >= total) return;
        int lo = 0, hi = nitems - 1;  // last solve with first[i] <= id
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (first[mid] <= id) lo = mid;
            else hi = mid - 1;
        }
        const int item = __builtin_amdgcn_readfirstlane(lo);
        const GmresArgs a = items[item];
        GmresWg<NT, RPT, false, MR> g(a, sh, id - first[item], dyn);
        g.run();
    }
}

// Zeroes the exchange area and result of every solve of a multi launch, and its ticket counter.
// (grid.x: the solves, grid.y: shares of an exchange area)
__global__ void k_gmres_clear(const GmresArgs* __restrict items, uint32_t* ticket) {
    const GmresArgs& a = items[blockIdx.x];
    const int64_t words = gmres_red_words(a.P, a.cap);
    for (int64_t i = (int64_t)blockIdx.y * blockDim.x + threadIdx.x; i < words; i += (int64_t)gridDim.y * blockDim.x)
        a.red[i] = 0ull;
    if (threadIdx.x == 0 && blockIdx.y == 0) {
        a.out->retcode = 0;
        a.out->pad = 0;
        a.out->iters = 0;
        a.out->resid = 0.0;
        a.out->err = 0ull;
        if (blockIdx.x == 0) *ticket = 0u;
    }
}

// ------------------------------------------------------------------------------------------
__global__ void k_spmv(int64_t N, const int32_t* __restrict rowptr, const int32_t* __restrict col,
                       const double* __restrict val, const double* __restrict xv, double* __restrict y) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= N) return;
    double s = 0.0;
    for (int32_t k = rowptr[r]; k < rowptr[r + 1]; ++k) s = __dadd_rn(s, __dmul_rn(val[k], xv[col[k]]));
    y[r] = s;
}

// Threads, rows per thread and workgroups of a solve of N rows.  A step's two exchanges cost about
// the same from a few workgroups to GMRES_WIDE of them, while everything else shrinks with the rows
// of a workgroup, so a solve takes the fewest rows per thread that keep it within a bound of
// workgroups.  The bounds grow with the rows: up to GALL workgroups the products take one message
// round instead of two.  GMRES(30), us a step: with 16 for the first bound 110^2 14.8 instead of 13.0;
// with 32 for the second 230^2 20.1 instead of 17.1; with 64 for the third 512^2 44.4 instead of 23.7, for
// the fourth 600^2 80.6 instead of 46.7.  Wider ones: 64 first 160^2 14.8 instead of 15.4 (and twice the CUs),
// 128 second 300^2 17.6 instead of 21.3.  GMRES_WIDE keeps every solve inside the serving lanes' share of
// the CUs, so a solve has the same shape, and the same bits, in every launch form.
constexpr int GMRES_WIDE = 128;
static void pick_shape(int64_t N, bool one_wg, GmresPlan* out) {
    out->nt = N <= 256 ? 256 : 1024;
    out->rpt = N <= 256 ? 1 : 8;
    const int bound[4] = {32, 64, GMRES_WIDE, GMRES_WIDE};
    for (int i = 0; i < 4 && N > 256; ++i)
        if (cdiv(N, 512 << i) <= (one_wg ? 1 : bound[i])) {
            out->nt = 512;
            out->rpt = 1 << i;
            break;
        }
    out->P = (int)cdiv(N, (int64_t)out->nt * out->rpt);
}

int csr_spmv_dev(lsx_csr* A, const double* dx, double* dy, hipStream_t st) {
    hipLaunchKernelGGL(k_spmv, dim3((unsigned)cdiv(A->N, 256)), dim3(256), 0, st, A->N, A->rowptr, A->col, A->val,
                       dx, dy);
    return hipGetLastError() == hipSuccess ? LSX_OK : LSX_EHIP;
}

constexpr size_t GMRES_LDS_MAX = 149 * 1024;  // dynamic LDS of a workgroup (160 KB less the static part)

// The largest Krylov dimension of one solve: GMRES_MAX_CAP_G (bookkeeping in HBM where the LDS does
// not hold it); with hbm false (the multi-solve launches) GMRES_MAX_CAP, and less above 2048 rows of a
// workgroup.  That second limit is what the entry points have always accepted; gmres_plan holds every
// dimension up to GMRES_MAX_CAP in LDS.
int gmres_cap_limit(int64_t N, bool hbm) {
    if (hbm) return GMRES_MAX_CAP_G;
    int64_t rows = 8192;  // rows of a workgroup, at two doubles each beside cap (cap + 1) / 2 + 3 cap + 1
    if (N <= 512) rows = 512;
    else if (N <= 2048 || (N > 8192 && cdiv(N, 2048) <= GMRES_WIDE)) rows = 2048;
    else if (N > 8192 && cdiv(N, 4096) <= GMRES_WIDE) rows = 4096;
    int64_t cap = GMRES_MAX_CAP;
    while (cap > 1 && 8 * (cap * (cap + 1) / 2 + 3 * cap + 1 + 2 * rows) > 150 * 1024) --cap;
    return (int)cap;
}

int gmres_plan(lsx_ctx* ctx, int64_t N, const GmresParams& p, GmresPlan* out, bool hbm, int64_t blocks) {
    pick_shape(N, blocks > 0, out);
    if (out->P > PMAX_G) return fail(ctx, LSX_EINVAL, "gmres: N = %lld exceeds %d rows", (long long)N, PMAX_G * 8192);
    const int64_t memory = std::max<int64_t>(1, std::min<int64_t>(p.memory, p.maxiters));
    const int64_t cap = p.restart ? memory : std::max<int64_t>(memory, p.maxiters);
    const int lim = gmres_cap_limit(N, hbm);
    if (cap > lim)
        return fail(ctx, LSX_EINVAL, "gmres: Krylov dimension %lld exceeds %d (restart = %d, N = %lld)", (long long)cap,
                    lim, p.restart, (long long)N);
    out->cap = (int)cap;
    // Solves of one workgroup, more of them than CUs: LDS for as many as the registers let a CU run at
    // once (they wait on their own barriers and not on each other), if the bookkeeping fits: three of 256
    // threads for up to 512 rows; two for 513 to 1024 rows, without the rows' entries in registers.  Against
    // one workgroup to a CU: 2000 blocks of 400 rows, memory 5 / 10 / 20: 8.4 / 5.7 / 5.6 -> 4.9 / 3.3 / 3.2 ms;
    // of 529 rows 13.8 / 8.6 / 7.8 -> 11.2 / 6.9 / 6.2.  Beyond 1024 rows a second workgroup's registers spill.
    auto lds_of = [](int64_t share) { return share == 1 ? GMRES_LDS_MAX : 160 * 1024 / (size_t)share - 8 * 1024; };
    int64_t share = std::max<int64_t>(1, std::min<int64_t>(N <= 512 ? 3 : N <= 1024 ? 2 : 1, cdiv(blocks, ctx->num_cus)));
    while (share > 1 && sizeof(double) * (size_t)gmres_book_words(cap) > lds_of(share)) --share;
    out->shared = share > 1;
    if (out->shared && N > 256 && N <= 512) {
        out->nt = 256;
        out->rpt = 2;
    }
    // LDS: the bookkeeping and the receive buffer first, then the current vector's own rows, then as
    // many basis vectors as fit.  The receive buffer holds the products of a 32-vector group from
    // all workgroups when there is room.
    const int64_t R = (int64_t)out->nt * out->rpt, words = (int64_t)(lds_of(share) / sizeof(double));
    int64_t left = words - gmres_book_words(cap);
    const int64_t rmin = out->P == 1 ? 0 : 512;
    out->rglob = left < rmin;
    if (out->rglob) left = words;
    out->own_lds = left - rmin >= R;
    const int64_t rwant = out->P == 1 || out->P > GALL ? rmin : 64 * (int64_t)GALL;
    out->rbuf_len = (int)std::max(rmin, std::min(rwant, left - (out->own_lds ? R : 0)) & ~(int64_t)1);
    left -= out->rbuf_len + (out->own_lds ? R : 0);
    out->ncache = (int)std::min<int64_t>(cap + 1, left / R);
    out->dynlds = sizeof(double) * (size_t)((out->rglob ? 0 : gmres_book_words(cap)) + out->rbuf_len +
                                            (out->own_lds ? R : 0) + out->ncache * R);
    return LSX_OK;
}

void gmres_plan_args(const GmresPlan& plan, GmresArgs* a) {
    a->cap = plan.cap;
    a->P = plan.P;
    a->ncache = plan.ncache;
    a->own_lds = plan.own_lds;
    a->rbuf_len = plan.rbuf_len;
    a->allread = plan.P > 1 && plan.P <= GALL;
}

int gmres_launch_multi(lsx_ctx* ctx, hipStream_t st, const GmresArgs* items, const int* first, int nitems,
                       int pool, int cls, size_t dynlds, uint32_t* ticket) {
    if (nitems < 1 || pool < 1) return fail(ctx, LSX_EINVAL, "gmres: empty multi launch");
    hipLaunchKernelGGL(k_gmres_clear, dim3((unsigned)nitems, nitems <= 64 ? 16 : 1), dim3(256), 0, st, items, ticket);
    auto go = [&](auto kern, int nt) {
        hipLaunchKernelGGL(kern, dim3(pool), dim3(nt), dynlds, st, items, first, nitems, ticket);
    };
    switch (cls) {
        case 0: go(k_gmres_multi<256, 1>, 256); break;
        case 1: go(k_gmres_multi<512, 1>, 512); break;
        case 2: go(k_gmres_multi<512, 2>, 512); break;
        case 3: go(k_gmres_multi<256, 2>, 256); break;
        case 5: go(k_gmres_multi<512, 2, false>, 512); break;
        case 4: go(k_gmres_multi<512, 4>, 512); break;
        case 8: go(k_gmres_multi<512, 8>, 512); break;
        default: go(k_gmres_multi<1024, 8>, 1024); break;
    }
    LSX_HIP(ctx, hipGetLastError());
    return LSX_OK;
}

// A device buffer of at least `need` bytes in *p (*have: its size), reallocated when it is smaller.
static int grow(lsx_ctx* ctx, void** p, size_t* have, size_t need, const char* what) {
    if (need <= *have) return LSX_OK;
    (void)hipFree(*p);
    *p = nullptr;
    *have = 0;
    if (hipMalloc(p, need) != hipSuccess)
        return fail(ctx, LSX_ENOMEM, "gmres: cannot allocate %zu bytes of %s", need, what);
    *have = need;
    return LSX_OK;
}

int gmres_launch(lsx_csr* A, const GmresParams& p, CoopHold& hold, const double* db, double* dx, const double* dpl,
                 const double* dpr, hipStream_t st) {
    lsx_ctx* ctx = A->ctx;
    const int64_t N = A->N;
    GmresPlan plan;
    int rc = gmres_plan(ctx, N, p, &plan, true);
    if (rc) return rc;
    const int P = plan.P;
    const int64_t cap = plan.cap, ldv = gmres_ldv(N);
    if ((rc = grow(ctx, (void**)&A->ws, &A->ws_bytes, sizeof(double) * (size_t)ldv * (size_t)(cap + 2), "Krylov workspace")))
        return rc;
    if (plan.rglob && (rc = grow(ctx, (void**)&A->rg, &A->rg_bytes, sizeof(double) * (size_t)P * (size_t)gmres_book_words(cap),
                                 "Krylov bookkeeping")))
        return rc;
    const size_t rb = sizeof(uint64_t) * (size_t)gmres_red_words(P, cap);
    if ((rc = grow(ctx, (void**)&A->red, &A->red_bytes, rb, "exchange words"))) return rc;
    if (rb) LSX_HIP(ctx, hipMemsetAsync(A->red, 0, rb, st));
    LSX_HIP(ctx, hipMemsetAsync(A->out, 0, sizeof(GmresOut), st));
    GmresArgs g;
    g.N = N;
    g.rowptr = A->rowptr;
    g.col = A->col;
    g.val = A->val;
    g.b = db;
    g.x = dx;
    g.pl = dpl;
    g.pr = dpr;
    g.V = A->ws;
    g.ldv = ldv;
    g.xp = A->ws + ldv * (cap + 1);
    g.memory = (int)std::max<int64_t>(1, std::min<int64_t>(p.memory, p.maxiters));
    g.restart = p.restart;
    gmres_plan_args(plan, &g);
    g.Rg = plan.rglob ? A->rg : nullptr;
    g.maxiters = p.maxiters;
    g.abstol = p.abstol;
    g.reltol = p.reltol;
    g.red = A->red;
    g.out = A->out;
    g.timeout = wait_ticks(ctx, 20.0);
    hold.take(ctx->device, ctx->num_cus, P);
    auto go = [&](auto lds, auto hbm) {
        if (plan.rglob) hipLaunchKernelGGL(hbm, dim3(P), dim3(plan.nt), plan.dynlds, st, g);
        else hipLaunchKernelGGL(lds, dim3(P), dim3(plan.nt), plan.dynlds, st, g);
    };
    switch (plan.cls()) {
        case 0: go(k_gmres<256, 1, false>, k_gmres<256, 1, true>); break;
        case 1: go(k_gmres<512, 1, false>, k_gmres<512, 1, true>); break;
        case 2: go(k_gmres<512, 2, false>, k_gmres<512, 2, true>); break;
        case 4: go(k_gmres<512, 4, false>, k_gmres<512, 4, true>); break;
        case 8: go(k_gmres<512, 8, false>, k_gmres<512, 8, true>); break;
        default: go(k_gmres<1024, 8, false>, k_gmres<1024, 8, true>); break;
    }
    LSX_HIP(ctx, hipGetLastError());
    return LSX_OK;
}

}  // namespace lsx

namespace lsx {
// CSR structure check: rowptr[0] = 0, rowptr[N] = nnz, rows non-decreasing within [0, nnz], column
// indices in [0, N); *bad is set otherwise.  A row's entries are read only once its bounds passed.
__global__ void k_csr_check(int64_t N, int64_t nnz, const int32_t* __restrict rowptr, const int32_t* __restrict col,
                            int* bad) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k0 = rowptr[r], k1 = rowptr[r + 1];
        if ((r == 0 && k0 != 0) || (r == N - 1 && k1 != nnz) || k0 < 0 || k1 < k0 || k1 > nnz) {
            *bad = 1;
            continue;
        }
        for (int64_t k = k0; k < k1; ++k)
            if (col[k] < 0 || col[k] >= N) *bad = 1;
    }
}

int csr_validate(hipStream_t st, int64_t N, int64_t nnz, const int32_t* rowptr, const int32_t* col, int* dflag) {
    if (hipMemsetAsync(dflag, 0, sizeof(int), st) != hipSuccess) return LSX_EHIP;
    hipLaunchKernelGGL(k_csr_check, dim3((unsigned)std::min<int64_t>(cdiv(N, 256), 4096)), dim3(256), 0, st, N, nnz,
                       rowptr, col, dflag);
    return hipGetLastError() == hipSuccess ? LSX_OK : LSX_EHIP;
}
}  // namespace lsx

// Column indices local to each row's block of `bs` rows (block-diagonal matrices); *bad is set
// when an entry lies outside its row's diagonal block.
__global__ void k_local_cols(int64_t N, int64_t bs, const int32_t* __restrict rowptr, const int32_t* __restrict col,
                             int32_t* __restrict cl, int* bad) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b0 = (r / bs) * bs;
        for (int32_t k = rowptr[r]; k < rowptr[r + 1]; ++k) {
            const int64_t c = col[k];
            if (c < b0 || c >= b0 + bs) *bad = 1;
            cl[k] = (int32_t)(c - b0);
        }
    }
}

// ------------------------------------------------------------------------------------------
// C-ABI
using namespace lsx;

static void csr_free(lsx_csr* A) {
    if (A->stream) (void)hipStreamSynchronize(A->stream);
    (void)hipFree(A->col_local);
    (void)hipFree(A->bitems);
    (void)hipFree(A->bfirst);
    (void)hipFree(A->bout);
    (void)hipFree(A->bticket);
    (void)hipFree(A->bflag);
    (void)hipFree(A->bpart);
    (void)hipFree(A->rowptr);
    (void)hipFree(A->col);
    (void)hipFree(A->val);
    (void)hipFree(A->ws);
    (void)hipFree(A->rg);
    (void)hipFree(A->red);
    (void)hipFree(A->out);
    if (A->hout) (void)hipHostFree(A->hout);
    (void)hipFree(A->db);
    (void)hipFree(A->dx);
    (void)hipFree(A->dpl);
    (void)hipFree(A->dpr);
    if (A->stream) (void)hipStreamDestroy(A->stream);
}

namespace lsx {

// Stopping tolerance of a batched solve, on the device: partial sums of (b / pl)^2 over a fixed
// grid of NPART blocks, then every block of k_batch_tol sums the partials in the same fixed order
// and writes eps = abstol + reltol sqrt(sum) into its share of the launch table (one value for all
// blocks, the same rounding on every call).
constexpr int NPART = 256;

__global__ __launch_bounds__(256) void k_sumsq_partial(const double* b, const double* pl, int64_t N, double* part) {
    __shared__ double s[256];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)NPART * 256) {
        const double r = pl ? b[i] / pl[i] : b[i];
        acc = fma(r, r, acc);
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(256) void k_batch_tol(const double* part, double abstol, double reltol, GmresArgs* items,
                                                   int64_t nitems) {
    __shared__ double s[NPART];
    s[threadIdx.x] = part[threadIdx.x];
    __syncthreads();
    for (int w = NPART / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    const double eps = abstol + reltol * sqrt(s[0]);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nitems; i += (int64_t)gridDim.x * 256)
        items[i].abstol = eps;
}

}  // namespace lsx

extern "C" {

int lsx_csr_create(lsx_ctx* ctx, int64_t N, int64_t nnz, const int32_t* rowptr, const int32_t* colind,
                   const double* vals, lsx_csr** out) {
    if (!ctx || !out || !rowptr || (nnz > 0 && (!colind || !vals))) return LSX_EINVAL;
    *out = nullptr;
    if (N < 1 || nnz < 0 || nnz > INT32_MAX)
        return fail(ctx, LSX_EINVAL, "lsx_csr_create: N = %lld, nnz = %lld out of range", (long long)N,
                    (long long)nnz);
    DeviceGuard g(ctx);
    lsx_csr* A = new (std::nothrow) lsx_csr();
    if (!A) return LSX_ENOMEM;
    A->ctx = ctx;
    A->N = N;
    A->nnz = nnz;
    auto bad = [&](int rc) {
        csr_free(A);
        delete A;
        return rc;
    };
    if (hipStreamCreateWithFlags(&A->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&A->rowptr, sizeof(int32_t) * (N + 1)) != hipSuccess ||
        hipMalloc(&A->col, sizeof(int32_t) * std::max<int64_t>(nnz, 1)) != hipSuccess ||
        hipMalloc(&A->val, sizeof(double) * std::max<int64_t>(nnz, 1)) != hipSuccess ||
        hipMalloc(&A->out, sizeof(GmresOut)) != hipSuccess ||
        hipHostMalloc(&A->hout, sizeof(GmresOut), hipHostMallocDefault) != hipSuccess ||
        hipMalloc(&A->db, sizeof(double) * N) != hipSuccess || hipMalloc(&A->dx, sizeof(double) * N) != hipSuccess ||
        hipMalloc(&A->dpl, sizeof(double) * N) != hipSuccess || hipMalloc(&A->dpr, sizeof(double) * N) != hipSuccess ||
        hipMalloc(&A->bflag, sizeof(int)) != hipSuccess)
        return bad(fail(ctx, LSX_ENOMEM, "lsx_csr_create: device allocation failed (N = %lld)", (long long)N));
    if (hipMemcpyAsync(A->rowptr, rowptr, sizeof(int32_t) * (N + 1), hipMemcpyDefault, A->stream) != hipSuccess ||
        (nnz > 0 && hipMemcpyAsync(A->col, colind, sizeof(int32_t) * nnz, hipMemcpyDefault, A->stream) != hipSuccess) ||
        (nnz > 0 && hipMemcpyAsync(A->val, vals, sizeof(double) * nnz, hipMemcpyDefault, A->stream) != hipSuccess) ||
        hipStreamSynchronize(A->stream) != hipSuccess)
        return bad(fail(ctx, LSX_EHIP, "lsx_csr_create: upload failed"));
    int badcsr = 0;
    if (csr_validate(A->stream, N, nnz, A->rowptr, A->col, A->bflag) != LSX_OK ||
        hipMemcpyAsync(&badcsr, A->bflag, sizeof(int), hipMemcpyDeviceToHost, A->stream) != hipSuccess ||
        hipStreamSynchronize(A->stream) != hipSuccess)
        return bad(fail(ctx, LSX_EHIP, "lsx_csr_create: structure check failed to run"));
    if (badcsr)
        return bad(fail(ctx, LSX_EINVAL, "lsx_csr_create: not a CSR matrix of order %lld with %lld entries (row pointers "
                        "or column indices out of range)", (long long)N, (long long)nnz));
    *out = A;
    return LSX_OK;
}

int lsx_csr_destroy(lsx_csr* A) {
    if (!A) return LSX_EINVAL;
    DeviceGuard g(A->ctx);
    csr_free(A);
    delete A;
    return LSX_OK;
}

int lsx_csr_spmv(lsx_csr* A, const double* x, double* y) {
    if (!A || !x || !y) return LSX_EINVAL;
    lsx_ctx* ctx = A->ctx;
    DeviceGuard g(ctx);
    LSX_HIP(ctx, hipMemcpyAsync(A->dx, x, sizeof(double) * A->N, hipMemcpyDefault, A->stream));
    int rc = csr_spmv_dev(A, A->dx, A->db, A->stream);
    if (rc) return fail(ctx, rc, "lsx_csr_spmv: launch failed");
    LSX_HIP(ctx, hipMemcpyAsync(y, A->db, sizeof(double) * A->N, hipMemcpyDefault, A->stream));
    LSX_HIP(ctx, hipStreamSynchronize(A->stream));
    return LSX_OK;
}

int lsx_gmres_solve(lsx_csr* A, const double* b, double* x, int32_t memory, int32_t restart, double abstol,
                    double reltol, int64_t maxiters, const double* pl_diag, const double* pr_diag,
                    lsx_gmres_stats* stats) {
    if (!A || !b || !x) return LSX_EINVAL;
    lsx_ctx* ctx = A->ctx;
    if (memory < 1 || maxiters < 0) return fail(ctx, LSX_EINVAL, "lsx_gmres_solve: memory >= 1, maxiters >= 0");
    DeviceGuard g(ctx);
    const size_t vb = sizeof(double) * A->N;
    LSX_HIP(ctx, hipMemcpyAsync(A->db, b, vb, hipMemcpyDefault, A->stream));
    if (pl_diag) LSX_HIP(ctx, hipMemcpyAsync(A->dpl, pl_diag, vb, hipMemcpyDefault, A->stream));
    if (pr_diag) LSX_HIP(ctx, hipMemcpyAsync(A->dpr, pr_diag, vb, hipMemcpyDefault, A->stream));
    GmresParams p{memory, restart ? 1 : 0, maxiters, abstol, reltol};
    CoopHold hold;
    int rc = gmres_launch(A, p, hold, A->db, A->dx, pl_diag ? A->dpl : nullptr, pr_diag ? A->dpr : nullptr, A->stream);
    if (rc) return rc;
    LSX_HIP(ctx, hipMemcpyAsync(x, A->dx, vb, hipMemcpyDefault, A->stream));
    LSX_HIP(ctx, hipMemcpyAsync(A->hout, A->out, sizeof(GmresOut), hipMemcpyDeviceToHost, A->stream));
    LSX_HIP(ctx, hipStreamSynchronize(A->stream));
    if (A->hout->err) return fail(ctx, LSX_ETIMEOUT, "lsx_gmres_solve: a device-side wait exceeded its bound");
    if (stats) {
        stats->retcode = A->hout->retcode;
        stats->pad = 0;
        stats->iters = A->hout->iters;
        stats->resid = A->hout->resid;
    }
    return LSX_OK;
}

int lsx_gmres_max_memory(lsx_csr* A, int32_t* memory) {
    if (!A || !memory) return LSX_EINVAL;
    *memory = gmres_cap_limit(A->N, true);
    return LSX_OK;
}

int lsx_gmres_solve_batched(lsx_csr* A, int64_t blocksize, const double* b, double* x, int32_t memory,
                            int32_t restart, double abstol, double reltol, int64_t maxiters, const double* pl_diag,
                            const double* pr_diag, lsx_gmres_stats* stats) {
    if (!A || !b || !x) return LSX_EINVAL;
    lsx_ctx* ctx = A->ctx;
    const int64_t N = A->N;
    if (blocksize < 1 || N % blocksize != 0)
        return fail(ctx, LSX_EINVAL, "lsx_gmres_solve_batched: blocksize %lld must divide N = %lld", (long long)blocksize,
                    (long long)N);
    if (memory < 1 || maxiters < 0)
        return fail(ctx, LSX_EINVAL, "lsx_gmres_solve_batched: memory >= 1, maxiters >= 0");
    DeviceGuard g(ctx);
    const int64_t nb = N / blocksize;
    GmresParams p{memory, restart ? 1 : 0, maxiters, 0.0, 0.0};
    GmresPlan plan;
    if (blocksize > 8192)
        return fail(ctx, LSX_EINVAL, "lsx_gmres_solve_batched: blocks of more than %d rows are not supported", 8192);
    int rc = gmres_plan(ctx, blocksize, p, &plan, false, nb);
    if (rc) return rc;
    const hipStream_t st = A->stream;
    // local columns (once per block size), after checking that A is block diagonal
    if (A->local_bs != blocksize) {
        if (!A->col_local) LSX_HIP(ctx, hipMalloc(&A->col_local, sizeof(int32_t) * std::max<int64_t>(A->nnz, 1)));
        LSX_HIP(ctx, hipMemsetAsync(A->bflag, 0, sizeof(int), st));
        hipLaunchKernelGGL(k_local_cols, dim3((unsigned)std::min<int64_t>(cdiv(N, 256), 4096)), dim3(256), 0, st, N,
                           blocksize, A->rowptr, A->col, A->col_local, A->bflag);
        int bad = 0;
        LSX_HIP(ctx, hipMemcpyAsync(&bad, A->bflag, sizeof(int), hipMemcpyDeviceToHost, st));
        LSX_HIP(ctx, hipStreamSynchronize(st));
        if (bad) return fail(ctx, LSX_EINVAL, "lsx_gmres_solve_batched: A has entries outside its %lld x %lld diagonal blocks",
                             (long long)blocksize, (long long)blocksize);
        A->local_bs = blocksize;
    }
    // buffers for nb blocks
    if (nb > A->bcap) {
        (void)hipFree(A->bitems);
        (void)hipFree(A->bfirst);
        (void)hipFree(A->bout);
        A->bitems = nullptr;
        A->bfirst = nullptr;
        A->bout = nullptr;
        A->bcap = 0;
        LSX_HIP(ctx, hipMalloc(&A->bitems, sizeof(GmresArgs) * nb));
        LSX_HIP(ctx, hipMalloc(&A->bfirst, sizeof(int) * (nb + 1)));
        LSX_HIP(ctx, hipMalloc(&A->bout, sizeof(GmresOut) * nb));
        A->bcap = nb;
        A->bkey[0] = 0;  // new table buffers: rebuild
    }
    if (!A->bticket) LSX_HIP(ctx, hipMalloc(&A->bticket, 256));
    const int64_t ldv = gmres_ldv(blocksize), vstride = ldv * (plan.cap + 2);
    if ((rc = grow(ctx, (void**)&A->ws, &A->ws_bytes, sizeof(double) * (size_t)(vstride * nb), "Krylov workspace"))) return rc;
    if (!A->bpart) LSX_HIP(ctx, hipMalloc(&A->bpart, sizeof(double) * NPART));
    const size_t vb = sizeof(double) * N;
    LSX_HIP(ctx, hipMemcpyAsync(A->db, b, vb, hipMemcpyDefault, st));
    if (pl_diag) LSX_HIP(ctx, hipMemcpyAsync(A->dpl, pl_diag, vb, hipMemcpyDefault, st));
    if (pr_diag) LSX_HIP(ctx, hipMemcpyAsync(A->dpr, pr_diag, vb, hipMemcpyDefault, st));
    // the launch table, rebuilt when what it holds changes; its tolerance is written on the device
    const int64_t memv = std::max<int64_t>(1, std::min<int64_t>(memory, maxiters));
    const int64_t wt = wait_ticks(ctx, 20.0);
    const int64_t key[9] = {blocksize, (pl_diag ? 1 : 0) | (pr_diag ? 2 : 0), memv, restart ? 1 : 0, maxiters,
                            (int64_t)(uintptr_t)A->ws, (int64_t)(uintptr_t)A->bitems, plan.cap, wt};
    if (!std::equal(key, key + 9, A->bkey)) {
        std::vector<GmresArgs> items(nb);
        std::vector<int> first(nb + 1);
        for (int64_t i = 0; i < nb; ++i) {
            GmresArgs& a = items[i];
            const int64_t r0 = i * blocksize;
            a.N = blocksize;
            a.rowptr = A->rowptr + r0;
            a.col = A->col_local;
            a.val = A->val;
            a.b = A->db + r0;
            a.x = A->dx + r0;
            a.pl = pl_diag ? A->dpl + r0 : nullptr;
            a.pr = pr_diag ? A->dpr + r0 : nullptr;
            a.V = A->ws + i * vstride;
            a.ldv = ldv;
            a.xp = a.V + ldv * (plan.cap + 1);
            a.memory = (int)memv;
            a.restart = restart ? 1 : 0;
            gmres_plan_args(plan, &a);
            a.maxiters = maxiters;
            a.abstol = 0.0;
            a.reltol = 0.0;
            a.red = nullptr;
            a.out = A->bout + i;
            a.timeout = wt;
            first[i] = (int)i;
        }
        first[nb] = (int)nb;
        LSX_HIP(ctx, hipMemcpyAsync(A->bitems, items.data(), sizeof(GmresArgs) * nb, hipMemcpyHostToDevice, st));
        LSX_HIP(ctx, hipMemcpyAsync(A->bfirst, first.data(), sizeof(int) * (nb + 1), hipMemcpyHostToDevice, st));
        LSX_HIP(ctx, hipStreamSynchronize(st));  // the host tables are freed on return
        std::copy(key, key + 9, A->bkey);
    }
    // the stopping tolerance of the whole batch: eps = abstol + reltol ||Pl \ b||_2
    // (src/simplegmres.jl:110-129: beta is the norm of the whole vector)
    hipLaunchKernelGGL(k_sumsq_partial, dim3(NPART), dim3(256), 0, st, A->db, pl_diag ? A->dpl : nullptr, N, A->bpart);
    hipLaunchKernelGGL(k_batch_tol, dim3((unsigned)std::min<int64_t>(cdiv(nb, 256), 64)), dim3(256), 0, st, A->bpart,
                       abstol, reltol, A->bitems, nb);
    const int pool = (int)std::min<int64_t>(nb, 4 * (int64_t)ctx->num_cus);
    rc = gmres_launch_multi(ctx, st, A->bitems, A->bfirst, (int)nb, pool, plan.cls(), plan.dynlds, A->bticket);
    if (rc) return rc;
    std::vector<GmresOut> outs(nb);
    LSX_HIP(ctx, hipMemcpyAsync(outs.data(), A->bout, sizeof(GmresOut) * nb, hipMemcpyDeviceToHost, st));
    LSX_HIP(ctx, hipMemcpyAsync(x, A->dx, vb, hipMemcpyDefault, st));
    LSX_HIP(ctx, hipStreamSynchronize(st));
    // the batch's result: iterations and rNorm of its slowest block; Infeasible if any block is,
    // else Success if every block is solved, else MaxIters (src/simplegmres.jl:603-606)
    int64_t iters = 0;
    double resid = 0.0;
    bool any_inf = false, all_ok = true;
    for (const GmresOut& o : outs) {
        if (o.err) return fail(ctx, LSX_ETIMEOUT, "lsx_gmres_solve_batched: a device-side wait exceeded its bound");
        iters = std::max<int64_t>(iters, o.iters);
        resid = std::max(resid, o.resid);
        any_inf = any_inf || o.retcode == LSX_RET_INFEASIBLE;
        all_ok = all_ok && o.retcode == LSX_RET_SUCCESS;
    }
    if (stats) {
        stats->retcode = any_inf ? LSX_RET_INFEASIBLE : (all_ok ? LSX_RET_SUCCESS : LSX_RET_MAXITERS);
        stats->pad = 0;
        stats->iters = iters;
        stats->resid = resid;
    }
    return LSX_OK;
}

}  // extern "C"
