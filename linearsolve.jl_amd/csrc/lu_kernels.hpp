// lu_kernels.hpp — LU building blocks templated on the working type (double for the plain
// FP64 path, float for the mixed-precision factorization): panel, row-interchange lists,
// interchange + TRSM, inverses of diagonal blocks, triangular solves.
//
// Pivot search: maximum |a| with NaN ignored, first (smallest) row on ties
// (src/blocked_lufact.jl:38-54); zero pivot -> info = first such column, factorization
// continues (src/generic_lufact.jl:71-141).  Scaling multiplies by the reciprocal of the pivot
// (blocked_lufact.jl:110-113) unless |pivot| < the smallest normal number (then divides, as
// LAPACK dgetf2).
#pragma once
#include <cfloat>
#include <climits>
#include <limits>

#include "lu.hpp"
#include "panel.hpp"

namespace lsx {

// ------------------------------------------------------------------------------------------
// Panel factorization: rows [j0, m) x columns [j0, j0+W), W <= PW.
template <typename T>
struct PanelArgs {
    T* A;
    int64_t ld;
    int64_t m;
    int64_t j0;
    int W;
    int P;
    int64_t* ipiv;
    int64_t* dinfo;
    uint64_t* slots;
    uint32_t seq;
    int64_t timeout;
    int64_t* list;   // the panel's row moves as (destination, source) pairs, in k_perm_build's form
    int* count;
};

// The panel on P workgroups covering rows [j0, m) (panel_columns does the columns).  With P > 1 every
// column exchanges one record per workgroup (its best candidate and that row's entries) as flag-in-word
// messages, one round trip through memory.  1024 rows per workgroup: panels of up to 1024 rows need no
// exchange at all, taller ones half the messages of 512.
template <typename T, int NT, int RPT>
__global__ __launch_bounds__(NT) void k_panel(PanelArgs<T> a) {
    constexpr int NW = NT / 64;
    constexpr int WPE = Words<T>::W;
    constexpr int HW = panel_head<T>();
    constexpr bool MULTI = NT * RPT == PROWS;    // the shape that several workgroups share a panel in
    const int tid = threadIdx.x, w = blockIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = (int)a.j0 + w * NT * RPT + tid;
    T* col0 = a.A + a.j0 * a.ld;
    T v[RPT][PW];
    int lr[RPT];
    bool live[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int r = r0 + k * NT;
        live[k] = r < (int)a.m;
        lr[k] = r;
#pragma unroll
        for (int q = 0; q < PW; ++q) v[k][q] = (live[k] && q < a.W) ? col0[q * a.ld + r] : T(0);
    }
    // pivots and the first zero pivot are kept here and written at the end: a store in the column loop
    // would be waited for by the next global access (or the next wait the compiler places)
    int info = 0;
    __shared__ PanelLds<T, NW> sh;
    __shared__ PanelRec<T> s_all[MULTI ? PMAX : 1];
    if (w == 0 && tid == 0) {
        __hip_atomic_store(a.count, a.W, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // in memory before any workgroup counts its moved rows (which all have seen a message, or
        // passed a barrier, of this one)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const int P = a.P;
    auto exchange = [&](const PanelRec<T>* own, int col, bool sender) -> const PanelRec<T>* {
        if (!MULTI || P == 1) {
            __syncthreads();
            return own;
        }
        const uint32_t seq = a.seq + (uint32_t)col + 1u;
        uint64_t* gs = a.slots + (size_t)(col & 1) * (PMAX + 1) * RECS;
        // the words of a record: the head, then the entries from column col & ~1 on; sent by the wave
        // that wrote the record (its own LDS writes need no barrier)
        const int q0 = col & ~1, nw = HW + WPE * (PW - q0);
        if (sender) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = lane + 64 * h;
                if (x < nw) {
                    uint32_t word;
                    if (x >= HW) word = reinterpret_cast<const uint32_t*>(own->v)[x - HW + WPE * q0];
                    else if (x >= 4) word = reinterpret_cast<const uint32_t*>(&own->inv)[x - 4];
                    else word = reinterpret_cast<const uint32_t*>(own)[x];
                    st_relaxed_u64(gs + (size_t)w * RECS + x, ll_pack(word, seq));
                }
            }
        }
        // wave i reads the records of workgroups i, i + NW, ..., four at a time, all words in
        // flight; words not yet current are read again together
#pragma unroll 1
        for (int p0 = wave; p0 < P; p0 += 4 * NW) {
            uint64_t x[8];
            uint32_t stale = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (p0 + (i >> 1) * NW < P && lane + 64 * (i & 1) < nw) stale |= 1u << i;
            const int64_t t0 = wall_clock64();
            for (unsigned spin = 1; stale; ++spin) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (stale & (1u << i))
                        x[i] = ld_relaxed_u64(gs + (size_t)(p0 + (i >> 1) * NW) * RECS + lane + 64 * (i & 1));
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if ((stale & (1u << i)) && (uint32_t)(x[i] >> 32) == seq) {
                        PanelRec<T>& d = s_all[p0 + (i >> 1) * NW];
                        const int xw = lane + 64 * (i & 1);
                        uint32_t* to = xw >= HW ? reinterpret_cast<uint32_t*>(d.v) + (xw - HW + WPE * q0)
                                       : xw >= 4 ? reinterpret_cast<uint32_t*>(&d.inv) + (xw - 4)
                                                 : reinterpret_cast<uint32_t*>(&d) + xw;
                        *to = (uint32_t)x[i];
                        stale &= ~(1u << i);
                    }
                }
                if (stale) {
                    // give up at the bound, or soon after another wait of this factorization has
                    // (its results are invalid anyway); the error word is read only every 16th
                    // round, since its load would double the period of the polling
                    if (wall_clock64() - t0 > a.timeout) {
                        atomicOr((unsigned long long*)&a.dinfo[1], 1ull);
                        break;
                    }
                    if (spin % 16 == 0 && ld_relaxed_u64((const uint64_t*)&a.dinfo[1]) != 0) break;
                }
            }
        }
        __syncthreads();
        const int wlane = wave_argmax32(lane < P ? s_all[lane & (PMAX - 1)].key : 0,
                                               lane < P ? s_all[lane & (PMAX - 1)].row : INT_MAX);
        return &s_all[wlane];
    };
    panel_columns<T, NT, RPT, false>(v, lr, live, a.W, (int)a.j0, (int)a.m, sh, info, exchange);
    __syncthreads();
    if (w == 0) {
        if (tid < a.W) a.ipiv[a.j0 + tid] = (int64_t)sh.piv[tid] + 1;
        if (tid == 0 && info != 0 && a.dinfo[0] == 0) a.dinfo[0] = info;
    }
    const int rot = 8 * ((a.W + 7) / 8);  // slot q holds column (q + rot) mod PW
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
        const int r = r0 + t * NT;
        if (r < (int)a.m) {
            T* dst = col0 + lr[t];
            const int top = lr[t] - (int)a.j0;
            if (top >= a.W) {
#pragma unroll
                for (int p = 0; p < PW; ++p) {
                    const int q = (p + rot) & (PW - 1);
                    if (q < a.W) dst[q * a.ld] = v[t][p];
                }
            } else {
#pragma unroll
                for (int q = 0; q < PW; ++q)
                    if (q < a.W) dst[q * a.ld] = sh.fin[top].v[q];
            }
            if (top < a.W || lr[t] != r) {
                const int pos = top < a.W ? top : atomicAdd(a.count, 1);
                if (pos < 2 * PW) {  // always, unless a wait gave up and the workgroups disagree
                    a.list[pos] = lr[t];
                    a.list[2 * NBO + pos] = r;
                }
            }
        }
    }
}

// Applies a panel's row moves to the other columns of its outer block, 16 columns per workgroup: nl
// columns left of the panel (from c0 on; nl a multiple of 32), then those from cr to cend, whose rows
// j0 .. j0 + PW - 1 are also replaced by L11^{-1} times them, L11 the panel's unit lower triangle
// (blocked_lufact.jl:126-178).  A row of 16 lanes solves one column, each lane two of its 32 rows, the
// solved entries broadcast by DPP moves: no barriers.  It is bound by the latency of three dependent
// accesses (list, rows, stores): 5 us; 32 columns per workgroup with a barrier per solved row took 10-14 us.
constexpr int ICW = 16;
template <typename T>
__global__ __launch_bounds__(256) void k_inner_swap(T* __restrict A, int64_t ld, int64_t n, int64_t j0, int W,
                                                    const int64_t* __restrict list, const int* __restrict count,
                                                    int64_t c0, int nl, int64_t cr, int64_t cend,
                                                    int* __restrict perm) {
    __shared__ int s_dst[2 * PW], s_src[2 * PW];
    __shared__ T s_buf[2 * PW][ICW + 1];
    __shared__ T s_L[PW][PW + 1];
    const int t = threadIdx.x;
    const int first = (int)blockIdx.x * ICW;
    const int64_t cb = first >= nl ? cr + (first - nl) : c0 + first;
    const int ncol = first >= nl ? (int)min((int64_t)ICW, cend - cb) : ICW;
    const bool right = first >= nl && ncol > 0;
    const int M = min(*count, 2 * PW);
    if (t < M) {
        // rows of [j0, n); clamped, since after a wait that gave up the list may hold anything
        s_dst[t] = (int)min(max(list[t], j0), n - 1);
        s_src[t] = (int)min(max(list[2 * NBO + t], j0), n - 1);
    }
    T lv[4];
    if (right) {
#pragma unroll
        for (int u = 0; u < 4; ++u) lv[u] = A[(j0 + (t >> 5) + 8 * u) * ld + j0 + (t & 31)];
    }
    __syncthreads();
    const bool map = blockIdx.x == 0 && t < M;  // the row map moves as one more column
    const int pv = map ? perm[s_src[t]] : 0;
    T v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = t & 63, cc = (t >> 6) + 4 * u;
        v[u] = (i < M && cc < ncol) ? A[(cb + cc) * ld + s_src[i]] : T(0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) s_buf[t & 63][(t >> 6) + 4 * u] = v[u];
    if (right) {
#pragma unroll
        for (int u = 0; u < 4; ++u) s_L[t & 31][(t >> 5) + 8 * u] = lv[u];
    }
    __syncthreads();  // every source row read before any row is written
    if (map) perm[s_dst[t]] = pv;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = t & 63, cc = (t >> 6) + 4 * u;
        if (i < M && cc < ncol && (i >= W || !right)) A[(cb + cc) * ld + s_dst[i]] = v[u];
    }
    if (!right) return;
    // here W == PW: columns right of a panel exist only if it is whole
    const int cc = t >> 4, i0 = t & 15, i1 = i0 + 16;
    T x0 = s_buf[i0][cc], x1 = s_buf[i1][cc];
    auto step0 = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const T b = row_bcast<k>(x0);
        const T y0 = fma(-s_L[i0][k], b, x0);
        x0 = i0 > k ? y0 : x0;
        x1 = fma(-s_L[i1][k], b, x1);
    };
    auto step1 = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const T b = row_bcast<k>(x1);
        const T y1 = fma(-s_L[i1][16 + k], b, x1);
        x1 = i0 > k ? y1 : x1;
    };
    static_for<0, 16>(step0);
    static_for<0, 16>(step1);
    if (cc < ncol) {
        A[(cb + cc) * ld + j0 + i0] = x0;
        A[(cb + cc) * ld + j0 + i1] = x1;
    }
}

// ------------------------------------------------------------------------------------------
// Row permutation of the LAPACK swap sequence ipiv[k0 .. k0+kb) (ipiv[k] >= k, 1-based) as a
// list of (destination row, source row) pairs: after the swaps, row dest[i] holds the former
// row src[i].
// One workgroup of 256 threads; kb <= 128.
// Positions 0..kb-1 stand for rows k0..k0+kb-1, positions kb..T-1 for the distinct pivot rows
// below the block (first occurrences, in order); swap u exchanges positions u and pos[u] >= u.
// Position q is last written by the last swap v with pos[v] = q, which moved there what
// position v held just before swap v, so every final label follows such links backwards in time
// independently of the others: no sequential replay of the swaps.
static __global__ __launch_bounds__(256) void k_perm_build(const int64_t* __restrict ipiv, int64_t k0, int kb,
                                                    int64_t* __restrict list, int* __restrict count) {
    __shared__ int64_t s_p[NBO];
    __shared__ int s_first[NBO];
    __shared__ int s_pos[NBO];
    __shared__ int s_prev[NBO];         // last earlier swap with the same target position
    __shared__ int s_last[2 * NBO];     // last swap targeting each position
    __shared__ int64_t s_rows[2 * NBO];
    const int t = threadIdx.x;
    const int64_t top = k0 + kb;
    if (t < kb) s_p[t] = ipiv[k0 + t] - 1;
    if (t < 2 * NBO) s_last[t] = -1;
    __syncthreads();
    // every loop below runs to its end (no early exit), so its LDS reads are independent
    int fidx = t;
    if (t < kb) {  // first swap with the same pivot row (below the block)
        const int64_t p = s_p[t];
        for (int u = t - 1; u >= 0; --u)
            if (s_p[u] == p) fidx = u;
        s_first[t] = (p >= top && fidx == t) ? 1 : 0;
        s_rows[t] = k0 + t;
    }
    __syncthreads();
    int extra = 0, before = 0;
    for (int u = 0; u < kb; ++u) {
        const int f = s_first[u];
        extra += f;
        before += (u < fidx) ? f : 0;
    }
    const int T = kb + extra;
    if (t < kb) {  // target position of swap t
        const int64_t p = s_p[t];
        const int pos = p >= top ? kb + before : (int)(p - k0);
        if (p >= top && fidx == t) s_rows[kb + before] = p;
        s_pos[t] = pos;
        atomicMax(&s_last[pos], t);
    }
    __syncthreads();
    if (t < kb) {
        const int pos = s_pos[t];
        int prev = -1;
        for (int u = 0; u < t; ++u)
            if (s_pos[u] == pos) prev = u;
        s_prev[t] = prev;
    }
    __syncthreads();
    int lab = t;
    if (t < T) {
        // label of position t: position q at time tm took, from the last swap v < tm targeting q,
        // what position v held just before swap v
        int q = t < kb ? s_pos[t] : t, tm = t < kb ? t : kb;
        while (true) {
            int v = s_last[q];
            while (v >= tm) v = s_prev[v];
            if (v < 0) break;
            q = v;
            tm = v;
        }
        lab = q;
        list[t] = s_rows[t];
        list[2 * NBO + t] = s_rows[lab];
    }
    if (t == 0) *count = T;
}

// Inverse of a row map, inv[perm[r]] = r, in each of nb consecutive maps of n.
static __global__ void k_inv_perm(const int* __restrict perm, int* __restrict inv, int nb, int64_t n) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int p = perm[r];
    for (int b = 0; b < nb; ++b) inv[b * n + p] = (int)r;
}

// Deferred row interchanges of the L columns.  While the matrix is factored, the interchanges of
// an outer block are applied to the columns right of it only; column c of outer block b keeps
// its rows [r0, n) (r0 = end of block b) in the row order the matrix had after block b.  At the
// end, row i of that segment takes the stored row inv_b[perm[i]]: perm is the final row map and
// inv_b the inverse of the row map after block b.  One workgroup per column, the segment staged
// in LDS (dynamic, (n - NBO) elements at most).
template <typename T>
__global__ __launch_bounds__(256) void k_left_gather(T* __restrict F, int64_t ld, int64_t n,
                                                     const int* __restrict perm, const int* __restrict pinv) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    T* s = reinterpret_cast<T*>(s_raw);
    const int64_t c = blockIdx.x;
    const int64_t b = c / NBO;
    const int64_t r0 = (b + 1) * NBO;
    if (r0 >= n) return;
    T* col = F + c * ld;
    // eight loads of a thread in flight before their LDS stores, and eight row indices (two
    // dependent loads each) before the gathers
    for (int64_t i0 = r0 + threadIdx.x; i0 < n; i0 += 8 * 256) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = i0 + u * 256 < n ? col[i0 + u * 256] : T(0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + u * 256 < n) s[i0 + u * 256 - r0] = v[u];
    }
    __syncthreads();
    const int* inv = pinv + b * n;
    for (int64_t i0 = r0 + threadIdx.x; i0 < n; i0 += 8 * 256) {
        int pr[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) pr[u] = i0 + u * 256 < n ? perm[i0 + u * 256] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) pr[u] = i0 + u * 256 < n ? inv[pr[u]] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + u * 256 < n) col[i0 + u * 256] = s[pr[u] - r0];
    }
}

static __global__ void k_iota(int* __restrict p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int)i;
}

// ------------------------------------------------------------------------------------------
// Applies a permutation list of rows to columns [c0, c1).  Each workgroup handles LCW columns.
constexpr int LCW = 32;
template <typename T>
__global__ __launch_bounds__(256) void k_laswp(T* __restrict A, int64_t ld, const int64_t* __restrict list,
                                               const int* __restrict count, int64_t c0, int64_t c1) {
    __shared__ int64_t s_dst[2 * NBO];
    __shared__ int64_t s_src[2 * NBO];
    __shared__ T s_buf[2 * NBO][LCW + 1];
    const int t = threadIdx.x;
    const int NT = *count;
    for (int i = t; i < NT; i += 256) {
        s_dst[i] = list[i];
        s_src[i] = list[2 * NBO + i];
    }
    __syncthreads();
    const int64_t cb = c0 + (int64_t)blockIdx.x * LCW;
    const int ncol = (int)min((int64_t)LCW, c1 - cb);
    // gather: consecutive threads walk consecutive list entries of one column; eight loads of a
    // thread in flight before their LDS stores (a store right after each load would wait for
    // the scattered rows one at a time)
    for (int base = t; base < NT * LCW; base += 8 * 256) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int idx = base + u * 256, cc = idx / NT, i = idx - cc * NT;
            v[u] = (idx < NT * LCW && cc < ncol) ? A[(cb + cc) * ld + s_src[i]] : T(0);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int idx = base + u * 256, cc = idx / NT, i = idx - cc * NT;
            if (idx < NT * LCW && cc < ncol) s_buf[i][cc] = v[u];
        }
    }
    __syncthreads();
    for (int idx = t; idx < NT * LCW; idx += 256) {
        const int cc = idx / NT, i = idx - cc * NT;
        if (cc < ncol) A[(cb + cc) * ld + s_dst[i]] = s_buf[i][cc];
    }
}

// ------------------------------------------------------------------------------------------
// Inverses of the 64 x 64 diagonal blocks of L (unit lower) and U (upper) of the factored
// matrix, used by the blocked TRSM of the outer update and by the triangular solves.
// grid = (number of blocks, 2): y = 0 inverts L blocks, y = 1 U blocks.  Four threads per
// column c of the inverse (columns are independent): thread p of the quad keeps the entries
// x[4 m + p] in registers and forms the substitution sum over them; the quad's four partial sums
// are added by two lane exchanges, so every step of the substitution is a chain of at most 16
// products instead of 64.  The block is staged in LDS.
template <typename T>
__global__ __launch_bounds__(256) void k_diag_inv(const T* __restrict F, int64_t ld, int64_t n,
                                                  int64_t b0, T* __restrict DL, T* __restrict DU) {
    const int64_t blk = b0 + blockIdx.x;
    const int64_t r0 = blk * DB;
    const int nb = (int)min((int64_t)DB, n - r0);
    const int t = threadIdx.x, c = t >> 2, p = t & 3;
    __shared__ T D[DB][DB + 1];   // D[i][k]
    {
        // all sixteen loads of a thread issued before any LDS store
        T v[DB * DB / 256];
#pragma unroll
        for (int u = 0; u < DB * DB / 256; ++u) {
            const int idx = t + 256 * u, i = idx & (DB - 1), k = idx / DB;
            v[u] = (i < nb && k < nb) ? F[(r0 + k) * ld + r0 + i] : (i == k ? T(1) : T(0));
        }
#pragma unroll
        for (int u = 0; u < DB * DB / 256; ++u) {
            const int idx = t + 256 * u;
            D[idx & (DB - 1)][idx / DB] = v[u];
        }
    }
    __syncthreads();
    T xk[DB / 4];  // x[4 m + p]
#pragma unroll
    for (int m = 0; m < DB / 4; ++m) xk[m] = T(0);
    auto quad_sum = [&](T v) {
        v += __shfl_xor(v, 1);
        v += __shfl_xor(v, 2);
        return v;
    };
    if (blockIdx.y == 0) {
        // column c of L^{-1}: x_c = 1, x_i = -sum_{k=c}^{i-1} L[i,k] x_k (i > c); x_k = 0 for k < c
#pragma unroll
        for (int i = 0; i < DB; ++i) {
            T a0 = T(0), a1 = T(0);
#pragma unroll
            for (int m = 0; 4 * m < i; ++m) {
                const T u = fma(D[i][4 * m + p], xk[m], (m & 1) ? a1 : a0);
                if (m & 1) a1 = (4 * m + p < i) ? u : a1;
                else a0 = (4 * m + p < i) ? u : a0;
            }
            const T sum = quad_sum(a0 + a1);
            const T xi = (i < c) ? T(0) : (i == c ? T(1) : -sum);
            if (p == (i & 3)) xk[i >> 2] = xi;
        }
    } else {
        // column c of U^{-1}: x_c = 1/U[c,c], x_i = -(sum_{k=i+1}^{c} U[i,k] x_k) / U[i,i] (i < c);
        // x_k = 0 for k > c
#pragma unroll
        for (int i = DB - 1; i >= 0; --i) {
            T a0 = T(0), a1 = T(0);
#pragma unroll
            for (int m = (i + 1) / 4; m < DB / 4; ++m) {
                const T u = fma(D[i][4 * m + p], xk[m], (m & 1) ? a1 : a0);
                if (m & 1) a1 = (4 * m + p > i) ? u : a1;
                else a0 = (4 * m + p > i) ? u : a0;
            }
            const T sum = quad_sum(a0 + a1);
            const T xi = (i > c) ? T(0) : (i == c ? T(1) / D[c][c] : -sum / D[i][i]);
            if (p == (i & 3)) xk[i >> 2] = xi;
        }
    }
    T* out = (blockIdx.y == 0 ? DL : DU) + blk * DB * DB;
#pragma unroll
    for (int m = 0; m < DB / 4; ++m) out[c * DB + 4 * m + p] = xk[m];  // column-major 64 x 64
}

// ------------------------------------------------------------------------------------------
// Triangular solves (getrs), one workgroup per DB-row block.
//   LOWER, not TR: Out = L^{-1} (P In)  (unit lower; the permutation gathers In by perm)
//   not LOWER, not TR: Out = U^{-1} In
// and with the transposed factors (trans = 'T': A^T x = b with P A = L U is U^T w = b, L^T v = w,
// x = P^T v):
//   LOWER, TR: Out = U^{-T} In  (U^T is lower triangular: blocks in forward order)
//   not LOWER, TR: Out[perm[i]] = (L^{-T} In)[i]  (blocks in backward order)
// Each block publishes its solution (DB x nrhs FP64 values) as flag-in-word messages: two
// 64-bit words per value, its 32-bit halves each with the launch's sequence number.  The blocks
// after it read those words directly, so a dependency costs one memory round trip (no flags, no
// fences).  A block accumulates the contributions of the blocks before it in solve order (four
// k-quarters of partial sums per row), the message reads of the next block issued before the
// current one is used, then applies the inverse of its diagonal block.
constexpr int TMW = 2 * DB * TRHS;  // message words of one block

// Words x[0 .. K) of block message m (word tid + 256 i) until they carry sequence number seq (mask:
// which of them the thread reads; they were loaded once before).  A wait that gives up sets err.
template <int K>
__device__ __forceinline__ void trsv_wait(uint64_t (&x)[K], uint32_t mask, const uint64_t* m, uint32_t seq,
                                          int64_t timeout, int64_t* err) {
    uint32_t stale = 0;
#pragma unroll
    for (int i = 0; i < K; ++i)
        if ((mask >> i & 1) && (uint32_t)(x[i] >> 32) != seq) stale |= 1u << i;
    if (!stale) return;
    const int64_t t0 = wall_clock64();
    for (unsigned spin = 1; stale; ++spin) {
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int i = 0; i < K; ++i)
            if (stale & (1u << i)) x[i] = ld_relaxed_u64(m + threadIdx.x + 256 * i);
#pragma unroll
        for (int i = 0; i < K; ++i)
            if ((stale & (1u << i)) && (uint32_t)(x[i] >> 32) == seq) stale &= ~(1u << i);
        if (stale && wall_clock64() - t0 > timeout) {
            atomicOr((unsigned long long*)err, 2ull);
            break;
        }
        // an earlier wait gave up (read every 16th round: its load would double the polling period)
        if (stale && spin % 16 == 0 && ld_relaxed_u64((const uint64_t*)err) != 0) break;
    }
}

// One right-hand side.  The block's right-hand side is read before the chain reaches the block.  The
// chain is bound by one memory round trip per block; the tiles are loaded one block ahead.  TR: the
// tile (j, b) of F is loaded down its columns (coalesced) and turned through LDS.  n = 6000, per
// triangle: 138 us forward, 140 us transposed (385-409 us with each transposed tile loaded where it was
// used and its row sums left to wave reductions).
template <typename T, bool LOWER, bool TR>
__global__ __launch_bounds__(256) void k_trsv(const T* __restrict F, int64_t ld, int64_t n,
                                              const int* __restrict perm, const T* __restrict Dinv,
                                              const double* In, double* Out, uint64_t* msg, uint32_t seq,
                                              int64_t timeout, int64_t* err) {
    const int nblk = (int)((n + DB - 1) / DB);
    const int bw = LOWER ? (int)blockIdx.x : nblk - 1 - (int)blockIdx.x;
    const int64_t r0 = (int64_t)bw * DB;
    const int tid = threadIdx.x, rr = tid & 63, g = tid >> 6;
    const int64_t row = r0 + rr;
    __shared__ double Ds[DB][DB + 1];
    __shared__ double Ys[2][DB];
    __shared__ double Ps[4][DB];
    __shared__ T Ts[TR ? 2 : 1][TR ? DB : 1][DB + 1];  // TR: the tile, Ts[.][r][c] = F[j DB + r, r0 + c]
    double bin = 0.0;
    if (tid < DB && row < n) bin = In[LOWER && !TR ? (int64_t)perm[row] : row];
    {
        T dv[DB * DB / 256];  // all loads in flight before the LDS stores
#pragma unroll
        for (int u = 0; u < DB * DB / 256; ++u) dv[u] = Dinv[(int64_t)bw * DB * DB + tid + 256 * u];
#pragma unroll
        for (int u = 0; u < DB * DB / 256; ++u) {
            const int idx = tid + 256 * u, i = idx & (DB - 1), k = idx >> 6;
            if (TR) Ds[k][i] = (double)dv[u];
            else Ds[i][k] = (double)dv[u];
        }
    }
    double acc = 0.0;
    // word w of a block's message: row w / 2, half w & 1
    const int nj = LOWER ? bw : nblk - 1 - bw;  // blocks before this one in solve order
    auto jblk = [&](int t) { return LOWER ? t : nblk - 1 - t; };
    uint64_t x[1] = {0};
    const uint32_t mask = tid < 2 * DB;
    auto issue = [&](int t) {
        if (mask) x[0] = ld_relaxed_u64(msg + (size_t)jblk(t) * TMW + tid);
    };
    // the 64 x 64 tile of block j: lane rr of group g holds F[row, j DB + 16 g + q] (TR:
    // F[j DB + rr, r0 + 16 g + q]), q < 16, in the factor's own type (converted where it is used, so
    // that no wait for the load is placed early)
    auto tload = [&](int t, T (&lv)[16]) {
        const int j = jblk(t);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t fr = TR ? (int64_t)j * DB + rr : row;
            const int64_t col = (TR ? r0 : (int64_t)j * DB) + 16 * g + q;
            lv[q] = (fr < n && col < n) ? F[col * ld + fr] : T(0);
        }
    };
    // block t of the solve order: its message (issued earlier) until current, into Ys, the next
    // block's message issued, then acc += tile * x_j
    auto step = [&](int t, const T (&lv)[16]) {
        const int buf = t & 1;
        if constexpr (TR) {
#pragma unroll
            for (int q = 0; q < 16; ++q) Ts[buf][rr][16 * g + q] = lv[q];
        }
        trsv_wait<1>(x, mask, msg + (size_t)jblk(t) * TMW, seq, timeout, err);
        // the two halves of a value sit in words w, w + 1 of threads tid, tid ^ 1
        const uint32_t mine = (uint32_t)x[0];
        const uint32_t other = (uint32_t)__shfl_xor((int)mine, 1);
        if (mask && !(tid & 1)) Ys[buf][tid >> 1] = __hiloint2double((int)other, (int)mine);
        if (t + 1 < nj) issue(t + 1);  // the next block's words travel while this one is used
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const double f = TR ? (double)Ts[buf][16 * g + q][rr] : (double)lv[q];
            acc = fma(f, Ys[buf][16 * g + q], acc);
        }
        // Ys and Ts are double-buffered: buffer buf is written again two blocks on, after the next
        // barrier
    };
    if (nj > 0) {
        issue(0);
        T la[16], lb[16];
        tload(0, la);
        for (int t = 0; t < nj; t += 2) {
            if (t + 1 < nj) tload(t + 1, lb);
            step(t, la);
            if (t + 1 >= nj) break;
            if (t + 2 < nj) tload(t + 2, la);
            step(t + 1, lb);
        }
    }
    Ps[g][rr] = acc;
    __syncthreads();
    double* Yb = Ys[nj & 1];
    if (tid < DB) Yb[tid] = bin - (Ps[0][tid] + Ps[1][tid] + Ps[2][tid] + Ps[3][tid]);
    __syncthreads();
    // y = Dinv Yb: group g forms the partial products over k in [16 g, 16 g + 16) (four short
    // chains instead of one of 64), reduced through Ps
    double y = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) y = fma(Ds[rr][16 * g + q], Yb[16 * g + q], y);
    Ps[g][rr] = y;
    __syncthreads();
    if (g == 0) {
        y = (Ps[0][rr] + Ps[1][rr]) + (Ps[2][rr] + Ps[3][rr]);
        uint64_t* mine = msg + (size_t)bw * TMW;
        st_relaxed_u64(mine + 2 * rr, ll_pack((uint32_t)__double2loint(y), seq));
        st_relaxed_u64(mine + 2 * rr + 1, ll_pack((uint32_t)__double2hiint(y), seq));
        if (row < n) Out[TR && !LOWER ? (int64_t)perm[row] : row] = y;
    }
}

// Up to TRHS right-hand sides: the same chain with the products on MFMA (v_mfma_f64_16x16x4f64), wave w
// forming rows 16 w .. of the block for all right-hand sides.  Lane l gives the tile's entry (row l & 15,
// column 4 s + l / 16) and x_j's (row 4 s + l / 16, right-hand side l & 15) at k-step s and holds rows
// l / 16 + 4 q, right-hand side l & 15 of the sums.  The message word of (row k, right-hand side s, half
// h) is 2 (16 k + s) + h.  With the products as vector arithmetic (an LDS read per term) a block took
// 6-8 us; factor + solve of 16 right-hand sides at n = 16384 went from 115.3 to 112.2 ms, of 5 at
// n = 3001 from 11.0 to 10.5 ms.
template <typename T, bool LOWER, bool TR>
__global__ __launch_bounds__(256) void k_trsv_mrhs(const T* __restrict F, int64_t ld, int64_t n,
                                                   const int* __restrict perm, const T* __restrict Dinv,
                                                   const double* In, int64_t ldin, double* Out, int64_t ldout,
                                                   int nrhs, uint64_t* msg, uint32_t seq, int64_t timeout,
                                                   int64_t* err) {
    typedef double v4d __attribute__((ext_vector_type(4)));
    static_assert(TRHS == 16, "one MFMA column block of right-hand sides");
    constexpr int WPT = TMW / 256;  // message words per thread
    const int nblk = (int)((n + DB - 1) / DB);
    const int bw = LOWER ? (int)blockIdx.x : nblk - 1 - (int)blockIdx.x;
    const int64_t r0 = (int64_t)bw * DB;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lo = lane & 15, hi = lane >> 4;
    const int64_t frow = r0 + 16 * w + lo;  // the row whose tile entries this lane gives
    __shared__ double Ys[2][DB][TRHS + 1];
    __shared__ T Ts[TR ? 2 : 1][TR ? DB : 1][DB + 1];  // TR: the tile, Ts[.][r][c] = F[j DB + r, r0 + c]
    for (int i = tid; i < 2 * DB * (TRHS + 1); i += 256) (&Ys[0][0][0])[i] = 0.0;  // unused right-hand sides
    double bin[4];
    T dv[16];  // the diagonal block's inverse, as tile entries
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t gr = r0 + 16 * w + hi + 4 * q;
        bin[q] = (gr < n && lo < nrhs) ? In[(int64_t)lo * ldin + (LOWER && !TR ? (int64_t)perm[gr] : gr)] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int i = 16 * w + lo, k = 4 * s + hi;
        dv[s] = Dinv[(int64_t)bw * DB * DB + (TR ? i * DB + k : k * DB + i)];
    }
    const int nj = LOWER ? bw : nblk - 1 - bw;  // blocks before this one in solve order
    auto jblk = [&](int t) { return LOWER ? t : nblk - 1 - t; };
    uint64_t x[WPT];
    uint32_t mask = 0;
#pragma unroll
    for (int i = 0; i < WPT; ++i)
        if (((tid + 256 * i) >> 1 & 15) < nrhs) mask |= 1u << i;
    auto issue = [&](int t) {
#pragma unroll
        for (int i = 0; i < WPT; ++i)
            x[i] = (mask >> i & 1) ? ld_relaxed_u64(msg + (size_t)jblk(t) * TMW + tid + 256 * i) : 0;
    };
    auto tload = [&](int t, T (&lv)[16]) {
        const int64_t j0 = (int64_t)jblk(t) * DB;
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const int64_t fr = TR ? j0 + lane : frow;
            const int64_t col = TR ? r0 + 16 * w + s : j0 + 4 * s + hi;
            lv[s] = (fr < n && col < n) ? F[col * ld + fr] : T(0);
        }
    };
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    auto step = [&](int t, const T (&lv)[16]) {
        const int buf = t & 1;
        if constexpr (TR) {
#pragma unroll
            for (int s = 0; s < 16; ++s) Ts[buf][lane][16 * w + s] = lv[s];
        }
        trsv_wait<WPT>(x, mask, msg + (size_t)jblk(t) * TMW, seq, timeout, err);
#pragma unroll
        for (int i = 0; i < WPT; ++i) {
            const int v = (tid + 256 * i) >> 1;
            const uint32_t mine = (uint32_t)x[i];
            const uint32_t other = (uint32_t)__shfl_xor((int)mine, 1);
            if (!(tid & 1) && (mask >> i & 1)) Ys[buf][v >> 4][v & 15] = __hiloint2double((int)other, (int)mine);
        }
        if (t + 1 < nj) issue(t + 1);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const double f = TR ? (double)Ts[buf][4 * s + hi][16 * w + lo] : (double)lv[s];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(f, Ys[buf][4 * s + hi][lo], acc, 0, 0, 0);
        }
    };
    __syncthreads();
    if (nj > 0) {
        issue(0);
        T la[16], lb[16];
        tload(0, la);
        for (int t = 0; t < nj; t += 2) {
            if (t + 1 < nj) tload(t + 1, lb);
            step(t, la);
            if (t + 1 >= nj) break;
            if (t + 2 < nj) tload(t + 2, la);
            step(t + 1, lb);
        }
    }
    double (*Yb)[TRHS + 1] = Ys[nj & 1];
#pragma unroll
    for (int q = 0; q < 4; ++q) Yb[16 * w + hi + 4 * q][lo] = bin[q] - acc[q];
    __syncthreads();
    v4d y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 16; ++s)
        y = __builtin_amdgcn_mfma_f64_16x16x4f64((double)dv[s], Yb[4 * s + hi][lo], y, 0, 0, 0);
    uint64_t* mine = msg + (size_t)bw * TMW;
    if (lo < nrhs) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = 16 * w + hi + 4 * q;
            st_relaxed_u64(mine + 2 * (16 * k + lo), ll_pack((uint32_t)__double2loint(y[q]), seq));
            st_relaxed_u64(mine + 2 * (16 * k + lo) + 1, ll_pack((uint32_t)__double2hiint(y[q]), seq));
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t row = r0 + 16 * w + hi + 4 * q;
            if (row < n) Out[(int64_t)lo * ldout + (TR && !LOWER ? (int64_t)perm[row] : row)] = y[q];
        }
    }
}

}  // namespace lsx
