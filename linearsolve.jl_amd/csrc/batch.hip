// batch.hip — thousands of independent small dense systems (n <= 512), each factored with
// partial pivoting and solved, in one persistent launch.
//
// Reference: the blockwise factorization of BlockDiagonalFactorization
// (ext/LinearSolveBlockDiagonalsExt.jl:101-114: lu!(B_i, pivot; check = false) per block,
// success = all(issuccess); :123-185 per-block ldiv!).  Per system the arithmetic of the FP64
// path is that of LAPACK dgetrf/dgetrs (pivot = first index of max |a|, NaN ignored; info = first
// zero pivot).  The FP32 path factors in FP32 and refines the solution in FP64
// (r = b - A x with the FP64 matrix, d = U \ L \ P r, x += d) until the normwise backward error
// ||r||_inf / (||A||_inf ||x||_inf + ||b||_inf) reaches the tolerance.
//
// Scheduling: systems are sorted by decreasing size on the host (longest first); a persistent
// grid of workgroups takes them from an atomic counter, one workgroup per system.
// Per system (BT threads): right-looking blocked LU, panels of 32 columns factored by the blocked LU's panel
// code (panel.hpp), two of them per step: the second panel's columns take the first's interchanges and
// update, then the columns right of both take the interchanges, U12 and one trailing update
// A22 -= L21 U12 of 64 columns on MFMA, so A22 is read and written once per 64 columns.  Row
// interchanges are applied in memory to the columns right of the panels as U12 is formed, so the
// trailing updates read and write contiguous rows; the L columns
// take the interchanges of later panels in one gather after the last panel (like dlaswp on the
// left, but once).  Triangular solves go by
// blocks of 64 (FP32: 32) rows: the diagonal block is staged in LDS and solved by one wave with
// shuffles, the rows beyond it are updated by all threads, sixteen loads in flight per row.
// The launch sequence of a handle (counter reset + persistent kernel) is captured once in a HIP
// graph and replayed by every factor_solve call (LSX_BATCH_NO_GRAPH=1 launches it directly).
#include <algorithm>
#include <cfloat>
#include <cstdlib>
#include <limits>
#include <new>
#include <numeric>
#include <vector>

#include "batch.hpp"
#include "panel.hpp"

namespace lsx {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int BT = 256;            // threads per system
constexpr int BNMAX = 512;         // largest system
constexpr int RPT = (BNMAX + BT - 1) / BT;  // panel rows per thread
static_assert(RPT <= 2, "a pivot row is held by the first or the last of a thread's panel rows");

// Per factor type: systems (workgroups) per CU and the row block SB of the triangular solves.  FP64: two
// systems per CU (up to 256 registers, 80 KB of LDS each).  FP32: three (168 registers, 53 KB), which
// hide the latency of its refinement passes.
template <typename T> struct BatchCfg;
template <> struct BatchCfg<double> { static constexpr int WG = 2, SB = 64; };
template <> struct BatchCfg<float> { static constexpr int WG = 3, SB = 32; };
constexpr int SW = 2 * PW;  // columns of a step of factor_sys (two panels)
constexpr int UCH = 128;    // columns of U12 staged in LDS at a time
// Stride of a staged column of U12, such that the 16 columns and the k entries that a wave (FP64: half a
// wave) reads at once fall into different LDS banks.
template <typename T> constexpr int ust() { return sizeof(T) == 8 ? SW + 2 : SW + 4; }

struct BatchArgs {
    int64_t count;
    const int32_t* order;     // systems by decreasing n
    const int32_t* n;
    const int64_t* aoff;      // offset of A_i (n_i^2 elements)
    const int64_t* voff;      // offset of b_i / x_i / ipiv_i
    void* A;                  // workspace of the factor type: factored in place
    const double* const* src; // device word holding the matrices' address: they are read there and factored
                              // in A (null, or a null address: A holds them; FP32 needs an address)
    const double* b;
    double* x;
    int64_t* ipiv;            // LAPACK swap sequence (1-based), packed like b
    int32_t* perm;            // row i of P A is row perm[i] of A, packed like b
    int64_t* info;
    int32_t* iters;           // refinement steps per system (nullable)
    double* berr;             // FP32 path: final backward error per system (nullable)
    int maxref;
    double tol;
    uint32_t* counter;
};

template <typename T>
struct BatchShared {
    static constexpr int SB = BatchCfg<T>::SB;
    static_assert(BNMAX <= SB * (SB + 1), "the FP32 residual is kept in the solve staging block");
    union {
        // factor_sys: the panel's LDS and, behind it, the second panel's U12 / L11 of both panels / staged U12
        __align__(16) T wide[UCH * ust<T>()];
        double dblk[SB][SB + 1];   // staged diagonal block of the solves / FP32 path: the residual
    };
    double red[2][BT / 64];
    int info;                  // 1 + the first column whose pivot is zero
    int chg[SW];               // rows below the panel(s) that the interchanges move
    int nchg;
    double xs[BNMAX];          // solve vector
    union {
        double xr[BNMAX];      // FP32 path: the refined solution (after the factorization)
        int piv[BNMAX];        // 0-based swap sequence (during the factorization)
    };
    int perm[BNMAX];
};

__device__ __forceinline__ int64_t uniform64(int64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Entry i of a system's matrix (at most 2 MB): a 32-bit byte offset from a uniform base, one register per
// address (and no scalar pair per column, which spill).
template <typename T> __device__ __forceinline__ T& el(T* A, int i) {
    typedef typename std::conditional<std::is_const<T>::value, const char, char>::type C;
    return *reinterpret_cast<T*>(reinterpret_cast<C*>(A) + (uint32_t)i * (uint32_t)sizeof(T));
}

// MFMA of the factor type: the transposed 16 x 16 tile D = X Y (X(i, k) = -U12(k, col i),
// Y(k, j) = L21(row j, k)); lane l / slot q holds C(row rb + (l & 15), col cb + ccol(l, q)).
template <typename T> struct BMma;
template <> struct BMma<double> {
    typedef v4d acc_t;
    __device__ static acc_t mma(double x, double y, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0); }
    __device__ static int ccol(int lane, int q) { return 4 * q + (lane >> 4); }
};
template <> struct BMma<float> {
    typedef v4f acc_t;
    __device__ static acc_t mma(float x, float y, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
    __device__ static int ccol(int lane, int q) { return 4 * (lane >> 4) + q; }
};

// Block-wide max of two non-negative values (all threads get both).
template <typename T>
__device__ __forceinline__ void block_max2(BatchShared<T>& sh, double& a, double& b) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a = fmax(a, __shfl_xor(a, off));
        b = fmax(b, __shfl_xor(b, off));
    }
    if (lane == 0) { sh.red[0][wave] = a; sh.red[1][wave] = b; }
    __syncthreads();
    a = sh.red[0][0];
    b = sh.red[1][0];
#pragma unroll
    for (int i = 1; i < BT / 64; ++i) { a = fmax(a, sh.red[0][i]); b = fmax(b, sh.red[1][i]); }
    __syncthreads();
}

// The columns of panel p (BW columns) hold their rows below the panel in the order after panel p; later
// panels swapped those rows.  S (kept in sh.perm, which ends as the system's permutation) is the
// composition of the swaps after panel p, built from the last panel back (row i of the final order is row
// S(i) of that order).
template <typename T, int BW>
__device__ __forceinline__ void gather_left(BatchShared<T>& sh, T* A, int n) {
    const int tid = threadIdx.x;
    for (int i = tid; i < n; i += BT) sh.perm[i] = i;
    __syncthreads();
    bool moved = false;  // some later swap exchanges two different rows
    for (int p = (n - 1) / BW; p >= 0; --p) {
        const int j0 = p * BW, jb = min(BW, n - j0), c1 = j0 + jb, m2 = n - c1;
        if (moved) {
            // thread tid moves rows c1 + tid + k BT, k < RPT (m2 < RPT BT), of the panel's columns,
            // through registers, GC columns at a time: in each group every source is read before
            // any row is written
            constexpr int GC = BW < 16 ? BW : 16;
#pragma unroll
            for (int cg = 0; cg < BW; cg += GC) {
                T g[RPT][GC];
#pragma unroll
                for (int k = 0; k < RPT; ++k) {
                    const int r = tid + k * BT;
#pragma unroll
                    for (int c = 0; c < GC; ++c)
                        g[k][c] = (r < m2 && cg + c < jb) ? el(A, (j0 + cg + c) * n + sh.perm[c1 + r]) : T(0);
                }
                __syncthreads();
#pragma unroll
                for (int k = 0; k < RPT; ++k) {
                    const int r = tid + k * BT;
#pragma unroll
                    for (int c = 0; c < GC; ++c)
                        if (r < m2 && cg + c < jb) el(A, (j0 + cg + c) * n + c1 + r) = g[k][c];
                }
            }
        }
        // S := tau(j0) o ... o tau(c1 - 1) o S, tau(k) exchanging rows k and piv[k]
        int pk[BW];
#pragma unroll
        for (int k = 0; k < BW; ++k) pk[k] = sh.piv[min(j0 + k, c1 - 1)];
        for (int i = j0 + tid; i < n; i += BT) {
            int x = sh.perm[i];
#pragma unroll
            for (int k = BW - 1; k >= 0; --k)
                if (k < jb) x = (x == j0 + k) ? pk[k] : (x == pk[k] ? j0 + k : x);
            sh.perm[i] = x;
        }
        for (int k = j0; k < c1; ++k) moved = moved || sh.piv[k] != k;
        __syncthreads();
    }
}

// MFMA tiles of the trailing updates: a C tile (R x C 16 x 16 blocks at rows rb, columns cb of the mr x nc
// matrix at A, leading dimension ld).  S (nullable): the tile's entries are read from there instead, row
// rb + 16 a2 + l of the tile being row sr[a2] of S (lane l's).
template <typename T, int R, int C>
__device__ __forceinline__ void tile_load(typename BMma<T>::acc_t (&c)[R][C], const T* A, const double* S, const int (&sr)[R],
                                          int ld, int mr, int nc, int rb, int cb, int lane) {
    if (S) {
#pragma unroll
        for (int a2 = 0; a2 < R; ++a2)
#pragma unroll
            for (int b2 = 0; b2 < C; ++b2)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int lr = rb + 16 * a2 + (lane & 15), lc = cb + 16 * b2 + BMma<T>::ccol(lane, q);
                    c[a2][b2][q] = (lr < mr && lc < nc) ? (T)el(S, lc * ld + sr[a2]) : T(0);
                }
        return;
    }
#pragma unroll
    for (int a2 = 0; a2 < R; ++a2)
#pragma unroll
        for (int b2 = 0; b2 < C; ++b2)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int lr = rb + 16 * a2 + (lane & 15), lc = cb + 16 * b2 + BMma<T>::ccol(lane, q);
                c[a2][b2][q] = (lr < mr && lc < nc) ? el(A, lc * ld + lr) : T(0);
            }
}
template <typename T, int R, int C>
__device__ __forceinline__ void tile_store(const typename BMma<T>::acc_t (&c)[R][C], T* A, int ld, int mr, int nc, int rb, int cb, int lane) {
#pragma unroll
    for (int a2 = 0; a2 < R; ++a2)
#pragma unroll
        for (int b2 = 0; b2 < C; ++b2)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int lr = rb + 16 * a2 + (lane & 15), lc = cb + 16 * b2 + BMma<T>::ccol(lane, q);
                if (lr < mr && lc < nc) el(A, lc * ld + lr) = c[a2][b2][q];
            }
}
// C (mr x nc at A22) -= L21 U12 for KB columns of L21 (at L21), U12 staged negated in LDS (column c's KB
// entries at Us + c us), by the waves in turn: a wave keeps a block of 32 rows of L21 in registers and
// sweeps the 32-column blocks of its segment of the columns, the next tile of C loaded while the
// current one is formed.  S (nullable): C is read from there, its row r being row map[r] (LDS) of S, and
// written to A22.
template <typename T, int KB>
__device__ __forceinline__ void tiles_update(T* A22, const double* S, const int* map, const T* L21, const T* Us, int us, int ld,
                                             int mr, int nc) {
    constexpr int R2 = 2, C2 = 2, KS = KB / 4, NW = BT / 64;
    using acc_t = typename BMma<T>::acc_t;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // (addresses are formed here, not before the loop over the steps)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tbr = (mr + 16 * R2 - 1) / (16 * R2), tbc = (nc + 16 * C2 - 1) / (16 * C2);
    const int nseg = min(tbc, (NW + tbr - 1) / tbr), segw = (tbc + nseg - 1) / nseg;
    for (int u = wave; u < tbr * nseg; u += NW) {
        const int rb = (u % tbr) * (16 * R2), sg = u / tbr;
        const int cbs = sg * segw, cbe = min(tbc, (sg + 1) * segw);
        if (cbs >= cbe) continue;
        acc_t acc[R2][C2];
        int sr[R2];
#pragma unroll
        for (int a2 = 0; a2 < R2; ++a2) sr[a2] = S ? map[min(rb + 16 * a2 + (lane & 15), mr - 1)] : 0;
        tile_load<T, R2, C2>(acc, A22, S, sr, ld, mr, nc, rb, cbs * (16 * C2), lane);
        T yl[R2][KS];
#pragma unroll
        for (int a2 = 0; a2 < R2; ++a2) {
            const int lr = rb + 16 * a2 + (lane & 15);
#pragma unroll
            for (int k4 = 0; k4 < KS; ++k4) yl[a2][k4] = lr < mr ? el(L21, (k4 * 4 + (lane >> 4)) * ld + lr) : T(0);
        }
        for (int cbi = cbs; cbi < cbe; ++cbi) {
            const int cb = cbi * (16 * C2);
            acc_t nxt[R2][C2];
            if (cbi + 1 < cbe) tile_load<T, R2, C2>(nxt, A22, S, sr, ld, mr, nc, rb, cb + 16 * C2, lane);
            const T* x0 = Us + (cb + (lane & 15)) * us + (lane >> 4);
#pragma unroll
            for (int k4 = 0; k4 < KS; ++k4) {
                T xv[C2];
#pragma unroll
                for (int b2 = 0; b2 < C2; ++b2) xv[b2] = x0[16 * b2 * us + 4 * k4];
#pragma unroll
                for (int a2 = 0; a2 < R2; ++a2)
#pragma unroll
                    for (int b2 = 0; b2 < C2; ++b2) acc[a2][b2] = BMma<T>::mma(xv[b2], yl[a2][k4], acc[a2][b2]);
            }
            tile_store<T, R2, C2>(acc, A22, ld, mr, nc, rb, cb, lane);
#pragma unroll
            for (int a2 = 0; a2 < R2; ++a2)
#pragma unroll
                for (int b2 = 0; b2 < C2; ++b2) acc[a2][b2] = nxt[a2][b2];
        }
    }
}

// The interchanges (sh.perm: row i of the new order is row sh.perm[i] of the old one; sh.chg: the rows below
// the panels that change) of columns [c0, c1), and U12 = L11^{-1} A12 in their rows j0 .. j0 + 32 NB - 1,
// L11's strictly lower part given by lf(i, k).  A row of 16 lanes takes one column (two with NB = 2, which
// share the reads of L11), each lane every 16th of its rows, the solved entries broadcast by DPP.  A row
// below the panels only ever receives what a swap brings from the panels' own rows, and every row is
// read before any is written.  S (nullable): the columns are read from there and only the U12 rows are
// written (the update that follows reads the other rows there too).  neg: also stores -U12 there (entry k of column c at neg[(c - c0) ns + k]).
template <typename T, int NB, typename LF>
__device__ __forceinline__ void swap_solve(BatchShared<T>& sh, T* A, const double* S, int n, int j0, int c0, int c1, LF&& lf, T* neg, int ns) {
    constexpr int NR = 2 * NB, NC = NB, CP = BT / 16;  // rows and columns per lane, columns per round
    int tid = threadIdx.x;
    const int nchg = S ? 0 : sh.nchg;
    for (int b = c0; b < c1; b += CP * NC) {
        // (hides the thread's number and the LDS contents, or L11's entries would be read before the loop
        // and spilled)
        asm volatile("" : "+v"(tid) : : "memory");
        const int l16 = tid & 15, grp = tid >> 4;
        T x[NC][NR], w[NC][NR];
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const int c = b + u * CP + grp, co = c * n;
            if (S) {
#pragma unroll
                for (int t = 0; t < NR; ++t) x[u][t] = c < c1 ? (T)el(S, co + sh.perm[j0 + l16 + 16 * t]) : T(0);
            } else {
#pragma unroll
                for (int t = 0; t < NR; ++t) {
                    x[u][t] = c < c1 ? el(A, co + sh.perm[j0 + l16 + 16 * t]) : T(0);
                    const int i = l16 + 16 * t;
                    w[u][t] = (c < c1 && i < nchg) ? el(A, co + sh.perm[sh.chg[i]]) : T(0);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const int c = b + u * CP + grp, co = c * n;
#pragma unroll
            for (int t = 0; t < NR; ++t) {
                const int i = l16 + 16 * t;
                if (c < c1 && i < nchg) el(A, co + sh.chg[i]) = w[u][t];
            }
        }
        static_for<0, 16 * NR>([&](auto kc) {
            constexpr int k = decltype(kc)::value, t0 = k / 16;
            T bx[NC];
#pragma unroll
            for (int u = 0; u < NC; ++u) bx[u] = row_bcast<(k & 15)>(x[u][t0]);
#pragma unroll
            for (int t = t0; t < NR; ++t) {
                const T l = lf(l16 + 16 * t, k);
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const T y = fma(-l, bx[u], x[u][t]);
                    x[u][t] = (t > t0 || l16 > (k & 15)) ? y : x[u][t];
                }
            }
            if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // L11 read a few columns ahead, not all
        });
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const int c = b + u * CP + grp;
#pragma unroll
            for (int t = 0; t < NR; ++t)
                if (c < c1) {
                    el(A, c * n + j0 + l16 + 16 * t) = x[u][t];
                    if (neg) neg[(c - c0) * ns + l16 + 16 * t] = -x[u][t];
                }
        }
    }
}

// LU with partial pivoting of one n x n system, panels of 32 columns, two per step (column-major, in
// place; on return A holds L and U in LAPACK's row order and sh.perm the system's permutation).
// What bounds a large system is its traffic on A22 (16 n^3 / (3 * 64) bytes at FP64; once per 32
// columns it was twice that) and the panel's chain (about 1.2 us a column, two systems to a CU).
// src: the matrix where the caller has it, read by the first step (so no copy is made first).
// 20,000 systems of n in [8, 512], FP64: 58.2 -> 39.1 ms against one update per 32-column panel (8
// or 16 columns below n = 192), panels with two barriers and two rows through LDS per column, and a
// copy of the matrices first.  3,000 systems, FP32 factors: 11.2 -> 8.9 ms.
// Small systems leave most of a panel's waves without rows, and a branch per column between the loads of
// a panel (with a spilled address each) made every load wait for the one before it.  With those waves
// waiting at the barriers only, no barriers in panels of one wave, and branch-free loads by 32-bit offsets
// (el): 20,000 FP64 systems of n = 1 0.65 -> 0.45 ms, of 8 to 16 1.25 -> 0.83; FP32 of 33 to 64 5.3 -> 3.3,
// 3,000 FP32 systems of 8 to 512 8.9 -> 6.7, 20,000 50.6 -> 36.8; FP64 of 8 to 512 39.2 -> 38.8.  Of the
// time of 20,000 systems, FP64 (FP32): panels 30 (23) %, trailing updates 29 (27), solves 21 (9), U12 16
// (11), the L columns' gather 3 (2), FP32's refinement 28.
template <typename T>
__device__ __forceinline__ void factor_sys(BatchShared<T>& sh, T* A, const double* src, int n, int64_t vo, int64_t* ipiv,
                                           int64_t& info) {
    int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    PanelLds<T, BT / 64>& pl = *reinterpret_cast<PanelLds<T, BT / 64>*>(sh.wide);
    constexpr int POFF = (int)((sizeof(PanelLds<T, BT / 64>) + 15) / 16 * 16 / sizeof(T));  // LDS after the panel's
    constexpr int BST = PW + 2;                                                          // stride of panel B's U12 there
    static_assert(POFF + PW * BST <= UCH * ust<T>() && SW * (SW + 1) <= UCH * ust<T>(), "LDS of factor_sys");
    int zero = (int)info;
    for (int j0 = 0; j0 < n; j0 += SW) {
        const int c1 = min(j0 + PW, n), c2 = min(j0 + SW, n);
        const double* S = j0 == 0 ? src : nullptr;  // the first step reads the matrix where the caller has it
        for (int i = j0 + tid; i < n; i += BT) sh.perm[i] = i;
        __syncthreads();
#pragma unroll 1
        for (int j = j0; j < c2; j += PW) {
            asm volatile("" : "+v"(tid));  // (as in tiles_update)
            // the panel of columns [j, j + w), rows j .. n - 1: to A in logical order, its interchanges
            // composed into sh.perm and applied to the step's first panel when this is the second
            const int w = min(PW, n - j);
            int lr[RPT];
            {
                T v[RPT][PW];
                bool live[RPT];
                int old[RPT];
#pragma unroll
                for (int t = 0; t < RPT; ++t) {
                    const int r = j + tid + t * BT;
                    live[t] = r < n;
                    lr[t] = r;
                    old[t] = r < n ? sh.perm[r] : 0;
                    // (eight columns at a time without branches: rows past the end take the last one's
                    // values, which nothing uses, columns past the end zeros)
                    const int rc = min(r, n - 1);
                    const bool none = j + 64 * wave + t * BT >= n;  // a wave without such rows
#pragma unroll
                    for (int q0 = 0; q0 < PW; q0 += 8) {
                        if (none || q0 >= w) {
#pragma unroll
                            for (int q = q0; q < q0 + 8; ++q) v[t][q] = T(0);
                        } else if (S && j == 0) {
#pragma unroll
                            for (int q = q0; q < q0 + 8; ++q) v[t][q] = (T)el(S, min(q, w - 1) * n + rc);
                        } else {
#pragma unroll
                            for (int q = q0; q < q0 + 8; ++q) v[t][q] = el(A, (j + min(q, w - 1)) * n + rc);
                        }
                    }
                    if (w < PW) {
#pragma unroll
                        for (int q = 0; q < PW; ++q) v[t][q] = q < w ? v[t][q] : T(0);
                    }
                }
                panel_columns<T, BT, RPT, true>(v, lr, live, w, j, n, pl, zero, [](const PanelRec<T>* r, int, bool) {
                    __syncthreads();
                    return r;
                });
                if (tid == 0) sh.info = zero;
                __syncthreads();
                zero = sh.info;
                if (tid == 0) sh.nchg = 0;
                if (tid < w) {
                    sh.piv[j + tid] = pl.piv[tid];
                    if (ipiv) ipiv[vo + j + tid] = (int64_t)pl.piv[tid] + 1;
                }
#pragma unroll
                for (int t = 0; t < RPT; ++t) {
                    if (j + tid + t * BT >= n) continue;
                    const int top = lr[t] - j;
                    sh.perm[lr[t]] = old[t];
                    const int dst = j * n + lr[t];
                    if (top >= w) {  // a whole panel: after its four rotations slot q holds column q again
#pragma unroll
                        for (int q = 0; q < PW; ++q) el(A, dst + q * n) = v[t][q];
                    } else if (w == PW) {
#pragma unroll
                        for (int q = 0; q < PW; ++q) el(A, dst + q * n) = pl.fin[top].v[q];
                    } else {
                        for (int q = 0; q < w; ++q) el(A, dst + q * n) = pl.fin[top].v[q];
                    }
                }
            }
            if (j > j0) {
                T g[RPT][PW];
#pragma unroll
                for (int t = 0; t < RPT; ++t) {
                    const int r = j + tid + t * BT;
                    if (r < n && lr[t] != r) {
#pragma unroll
                        for (int q = 0; q < PW; ++q) g[t][q] = el(A, (j0 + q) * n + r);
                    }
                }
                __syncthreads();
#pragma unroll
                for (int t = 0; t < RPT; ++t) {
                    const int r = j + tid + t * BT;
                    if (r < n && lr[t] != r) {
#pragma unroll
                        for (int q = 0; q < PW; ++q) el(A, (j0 + q) * n + lr[t]) = g[t][q];
                    }
                }
            }
            __syncthreads();
            if (j + w >= n) continue;  // the last panel
            // the rows below the panel that are not in their places of the step's start
            for (int i = j + w + tid; i < n; i += BT)
                if (sh.perm[i] != i) sh.chg[atomicAdd(&sh.nchg, 1)] = i;
            __syncthreads();
            if (j > j0 || c1 >= n) continue;
            // the second panel's columns: interchanges, U12 and update of the first
            T* Ub = sh.wide + POFF;
            swap_solve<T, 1>(sh, A, S, n, j0, c1, c2, [&](int i, int k) { return pl.fin[i].v[k]; }, Ub, BST);
            __syncthreads();
            tiles_update<T, PW>(A + c1 * n + c1, S ? S + c1 * n : nullptr, sh.perm + c1, A + j0 * n + c1, Ub, BST, n, n - c1, c2 - c1);
            __syncthreads();
        }
        if (c2 >= n) break;
        // the columns right of both panels
        T* L11 = sh.wide;  // L11[i (SW + 1) + k]
        for (int i = tid; i < SW * SW; i += BT) {
            const int r = i & (SW - 1), k = i / SW;
            L11[r * (SW + 1) + k] = el(A, (j0 + k) * n + j0 + r);
        }
        __syncthreads();
        swap_solve<T, 2>(sh, A, S, n, j0, c2, n, [&](int i, int k) { return L11[i * (SW + 1) + k]; }, (T*)nullptr, 0);
        for (int cc = c2; cc < n; cc += UCH) {
            const int nc = min(UCH, n - cc);
            __syncthreads();  // L11, or the previous columns' U12, is no longer read; U12 is in memory
            for (int b0 = tid; b0 < nc * SW; b0 += 8 * BT) {
                T t8[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int i = b0 + u * BT;
                    t8[u] = i < nc * SW ? el(A, (cc + i / SW) * n + j0 + (i & (SW - 1))) : T(0);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int i = b0 + u * BT;
                    if (i < nc * SW) sh.wide[(i / SW) * ust<T>() + (i & (SW - 1))] = -t8[u];
                }
            }
            __syncthreads();
            tiles_update<T, SW>(A + cc * n + c2, S ? S + cc * n : nullptr, sh.perm + c2, A + j0 * n + c2, sh.wide, ust<T>(), n, n - c2, nc);
        }
        __syncthreads();
    }
    info = zero;
    if (n > SW) gather_left<T, SW>(sh, A, n);  // (one step: nothing to its left, and sh.perm is its interchanges)
}

// s - sum_{k0 <= k < k1} a[k * n] x[k] in the order of k (FP64), sixteen loads in flight; ABS: ra += the
// sum of |a[k * n]| too.
template <bool ABS, typename T>
__device__ __forceinline__ double row_dot_sub(double s, const T* a, int n, const double* x, int k0, int k1, double& ra) {
    int k = k0;
    for (; k + 16 <= k1; k += 16) {
        T av[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) av[u] = a[(int64_t)(k + u) * n];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            s = fma(-(double)av[u], x[k + u], s);
            if (ABS) ra += fabs((double)av[u]);
        }
    }
    for (; k < k1; ++k) {
        const double av = (double)a[(int64_t)k * n];
        s = fma(-av, x[k], s);
        if (ABS) ra += fabs(av);
    }
    return s;
}

// The kb x kb diagonal block at (k0, k0) into D (FP64); a full block with all of a thread's
// loads in flight before its LDS stores.
template <typename T, int SB>
__device__ __forceinline__ void stage_block(double (*D)[SB + 1], const T* A, int n, int k0, int kb) {
    const int tid = threadIdx.x;
    if (kb == SB) {
        T v[SB * SB / BT];
#pragma unroll
        for (int u = 0; u < SB * SB / BT; ++u) {
            const int idx = tid + u * BT, r = idx % SB, c = idx / SB;
            v[u] = A[(int64_t)(k0 + c) * n + k0 + r];
        }
#pragma unroll
        for (int u = 0; u < SB * SB / BT; ++u) {
            const int idx = tid + u * BT;
            D[idx % SB][idx / SB] = (double)v[u];
        }
    } else {
        for (int idx = tid; idx < kb * kb; idx += BT) {
            const int r = idx % kb, c = idx / kb;
            D[r][c] = (double)A[(int64_t)(k0 + c) * n + k0 + r];
        }
    }
}

// sh.xs := U^{-1} L^{-1} sh.xs (sh.xs already holds P b), arithmetic in FP64.
template <typename T>
__device__ __forceinline__ void solve_sys(BatchShared<T>& sh, const T* A, int n) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int SB = BatchCfg<T>::SB;
    double dummy = 0.0;
    static_assert((SB * SB) % BT == 0, "a full diagonal block is whole loads per thread");
    double (*D)[SB + 1] = sh.dblk;
    // forward: unit lower L
    for (int k0 = 0; k0 < n; k0 += SB) {
        const int kb = min(SB, n - k0);
        stage_block<T, SB>(D, A, n, k0, kb);
        __syncthreads();
        if (wave == 0) {
            double xv = lane < kb ? sh.xs[k0 + lane] : 0.0;
            for (int c = 0; c < kb; ++c) {
                const double xc = __shfl(xv, c);
                if (lane > c && lane < kb) xv = fma(-D[lane][c], xc, xv);
            }
            if (lane < kb) sh.xs[k0 + lane] = xv;
        }
        __syncthreads();
        for (int i = k0 + kb + tid; i < n; i += BT) sh.xs[i] = row_dot_sub<false>(sh.xs[i], A + i, n, sh.xs, k0, k0 + kb, dummy);
        __syncthreads();
    }
    // backward: U
    for (int k1 = n; k1 > 0; k1 -= SB) {
        const int k0 = max(0, k1 - SB), kb = k1 - k0;
        stage_block<T, SB>(D, A, n, k0, kb);
        __syncthreads();
        if (wave == 0) {
            double xv = lane < kb ? sh.xs[k0 + lane] : 0.0;
            for (int c = kb - 1; c >= 0; --c) {
                if (lane == c) xv = xv / D[c][c];
                const double xc = __shfl(xv, c);
                if (lane < c) xv = fma(-D[lane][c], xc, xv);
            }
            if (lane < kb) sh.xs[k0 + lane] = xv;
        }
        __syncthreads();
        for (int i = tid; i < k0; i += BT) sh.xs[i] = row_dot_sub<false>(sh.xs[i], A + i, n, sh.xs, k0, k1, dummy);
        __syncthreads();
    }
}

template <typename T>
__global__ __launch_bounds__(BT, BatchCfg<T>::WG * BT / 256) void k_batch_lu(BatchArgs a) {  // min waves per SIMD
    __shared__ BatchShared<T> sh;
    __shared__ int s_item;
    const int tid = threadIdx.x;
    while (true) {
        if (tid == 0) s_item = (int)atomicAdd(a.counter, 1u);
        __syncthreads();
        // the system's scalars are wave-uniform (held in scalar registers)
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        if (item >= a.count) break;
        const int sys = __builtin_amdgcn_readfirstlane(a.order[item]);
        const int n = __builtin_amdgcn_readfirstlane(a.n[sys]);
        const int64_t ao = uniform64(a.aoff[sys]);
        T* A = reinterpret_cast<T*>(a.A) + ao;
        const int64_t vo = uniform64(a.voff[sys]);
        int64_t info = 0;
        const double* src = a.src ? *a.src : nullptr;
        if (src) src += ao;
        factor_sys<T>(sh, A, src, n, vo, a.ipiv, info);
        // solve: x = U^{-1} L^{-1} P b
        for (int i = tid; i < n; i += BT) sh.xs[i] = a.b[vo + sh.perm[i]];
        __syncthreads();
        solve_sys<T>(sh, A, n);
        if constexpr (sizeof(T) == 4) {
            // FP64 refinement
            double an = 0.0, bn = 0.0;  // ||A||_inf (summed during the first residual), ||b||_inf
            for (int i = tid; i < n; i += BT) sh.xr[i] = sh.xs[i];
            __syncthreads();
            double* rr = &sh.dblk[0][0];  // residual by original row (n <= (SB + 1) SB)
            int it = 0;
            double be = 0.0;
            while (true) {
                double rn = 0.0, xn = 0.0;
                for (int i = tid; i < n; i += BT) {
                    double s, ra = 0.0;
                    if (it == 0) {
                        s = row_dot_sub<true>(a.b[vo + i], src + i, n, sh.xr, 0, n, ra);
                        an = fmax(an, ra);
                        bn = fmax(bn, fabs(a.b[vo + i]));
                    } else {
                        s = row_dot_sub<false>(a.b[vo + i], src + i, n, sh.xr, 0, n, ra);
                    }
                    rr[i] = s;
                    rn = fmax(rn, fabs(s));
                    xn = fmax(xn, fabs(sh.xr[i]));
                }
                block_max2(sh, rn, xn);
                if (it == 0) block_max2(sh, an, bn);
                const double den = an * xn + bn;
                be = den > 0.0 ? rn / den : 0.0;
                if (!(be > a.tol) || it >= a.maxref || info != 0) break;
                for (int i = tid; i < n; i += BT) sh.xs[i] = rr[sh.perm[i]];
                __syncthreads();
                solve_sys<T>(sh, A, n);
                for (int i = tid; i < n; i += BT) sh.xr[i] += sh.xs[i];
                __syncthreads();
                ++it;
            }
            for (int i = tid; i < n; i += BT) a.x[vo + i] = sh.xr[i];
            if (tid == 0) {
                if (a.iters) a.iters[sys] = it;
                if (a.berr) a.berr[sys] = be;
            }
        } else {
            for (int i = tid; i < n; i += BT) a.x[vo + i] = sh.xs[i];
            if (tid == 0) {
                if (a.iters) a.iters[sys] = 0;
                if (a.berr) a.berr[sys] = -1.0;
            }
        }
        for (int i = tid; i < n; i += BT) a.perm[vo + i] = sh.perm[i];
        if (tid == 0) a.info[sys] = info;
        __syncthreads();
    }
}

__global__ void k_reset_counter(uint32_t* c) { *c = 0u; }

int batch_launch_raw(lsx_ctx* ctx, hipStream_t st, int64_t count, const int32_t* order, const int32_t* n,
                     const int64_t* aoff, const int64_t* voff, double* A, const double* b, double* x, int64_t* ipiv,
                     int32_t* perm, int64_t* info, uint32_t* counter) {
    hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(1), 0, st, counter);
    BatchArgs a{};
    a.count = count;
    a.order = order;
    a.n = n;
    a.aoff = aoff;
    a.voff = voff;
    a.A = A;
    a.b = b;
    a.x = x;
    a.ipiv = ipiv;
    a.perm = perm;
    a.info = info;
    a.counter = counter;
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(count, (int64_t)ctx->num_cus * BatchCfg<double>::WG));
    hipLaunchKernelGGL(k_batch_lu<double>, dim3(grid), dim3(BT), 0, st, a);
    LSX_HIP(ctx, hipGetLastError());
    return LSX_OK;
}

// The launch sequence of a handle: counter reset + the persistent kernel on the handle's buffers.
static void batch_enqueue(lsx_batch* B) {
    hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(1), 0, B->stream, B->counter);
    BatchArgs a{};
    a.count = B->count;
    a.order = B->order;
    a.n = B->n;
    a.aoff = B->aoff;
    a.voff = B->voff;
    a.b = B->b;
    a.x = B->x;
    a.ipiv = B->ipiv;
    a.perm = B->perm;
    a.info = B->info;
    a.iters = B->iters;
    a.berr = B->berr;
    a.maxref = B->maxref;
    a.tol = B->tol;
    a.counter = B->counter;
    a.src = B->dsrc;
    auto grid = [&](int wg) { return (int)std::max<int64_t>(1, std::min<int64_t>(B->count, (int64_t)B->ctx->num_cus * wg)); };
    if (B->dtype == LSX_F64) {
        a.A = B->A;
        hipLaunchKernelGGL(k_batch_lu<double>, dim3(grid(BatchCfg<double>::WG)), dim3(BT), 0, B->stream, a);
    } else {
        a.A = B->A32;
        hipLaunchKernelGGL(k_batch_lu<float>, dim3(grid(BatchCfg<float>::WG)), dim3(BT), 0, B->stream, a);
    }
}

int batch_run(lsx_batch* B, const double* A, const double* db, double* dx) {
    lsx_ctx* ctx = B->ctx;
    // matrices in this GPU's memory are read where they are (a copy of them took a ninth of a call's
    // time); others are copied into the handle, where FP64 batches factor them in place
    const double* src = A;
    if (!is_device_ptr(ctx->device, A)) {
        if (!B->A && hipMalloc(&B->A, sizeof(double) * B->total_a) != hipSuccess) {
            B->A = nullptr;
            return fail(ctx, LSX_ENOMEM, "lsx_batch_factor_solve: cannot stage the matrices");
        }
        LSX_HIP(ctx, hipMemcpyAsync(B->A, A, sizeof(double) * B->total_a, hipMemcpyDefault, B->stream));
        src = B->dtype == LSX_F64 ? nullptr : B->A;
    }
    *B->hsrc = src;
    LSX_HIP(ctx, hipMemcpyAsync(B->dsrc, B->hsrc, sizeof(src), hipMemcpyHostToDevice, B->stream));
    if (db != B->b) LSX_HIP(ctx, hipMemcpyAsync(B->b, db, sizeof(double) * B->total_v, hipMemcpyDefault, B->stream));
    const int pi = B->prof.begin(B->stream, PK_OTHER, B->flops, sizeof(double) * 2.0 * (double)B->total_a);
    if (B->use_graph) {
        if (!B->graph_exec) {
            hipGraph_t g = nullptr;
            LSX_HIP(ctx, hipStreamBeginCapture(B->stream, hipStreamCaptureModeThreadLocal));
            batch_enqueue(B);
            LSX_HIP(ctx, hipStreamEndCapture(B->stream, &g));
            const hipError_t e = hipGraphInstantiate(&B->graph_exec, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            LSX_HIP(ctx, e);
        }
        LSX_HIP(ctx, hipGraphLaunch(B->graph_exec, B->stream));
    } else {
        batch_enqueue(B);
    }
    B->prof.end(B->stream, pi);
    LSX_HIP(ctx, hipGetLastError());
    if (dx != B->x) LSX_HIP(ctx, hipMemcpyAsync(dx, B->x, sizeof(double) * B->total_v, hipMemcpyDefault, B->stream));
    return LSX_OK;
}

}  // namespace lsx

using namespace lsx;

static void batch_free(lsx_batch* B) {
    if (B->stream) (void)hipStreamSynchronize(B->stream);
    if (B->graph_exec) (void)hipGraphExecDestroy(B->graph_exec);
    (void)hipFree(B->order);
    (void)hipFree(B->n);
    (void)hipFree(B->aoff);
    (void)hipFree(B->voff);
    (void)hipFree(B->A);
    (void)hipFree(B->dsrc);
    if (B->hsrc) (void)hipHostFree((void*)B->hsrc);
    (void)hipFree(B->A32);
    (void)hipFree(B->b);
    (void)hipFree(B->x);
    (void)hipFree(B->ipiv);
    (void)hipFree(B->perm);
    (void)hipFree(B->info);
    (void)hipFree(B->iters);
    (void)hipFree(B->berr);
    (void)hipFree(B->counter);
    if (B->hinfo) (void)hipHostFree(B->hinfo);
    if (B->stream) (void)hipStreamDestroy(B->stream);
}

extern "C" {

int lsx_batch_create(lsx_ctx* ctx, int64_t count, const int64_t* n, int dtype, lsx_batch** out) {
    if (!ctx || !out || !n || count < 1) return LSX_EINVAL;
    *out = nullptr;
    if (dtype != LSX_F64 && dtype != LSX_F32)
        return fail(ctx, LSX_EINVAL, "lsx_batch_create: dtype must be LSX_F64 or LSX_F32");
    std::vector<int32_t> hn(count);
    std::vector<int64_t> aoff(count), voff(count);
    int64_t ta = 0, tv = 0;
    double flops = 0.0;
    for (int64_t i = 0; i < count; ++i) {
        if (n[i] < 1 || n[i] > BNMAX)
            return fail(ctx, LSX_EINVAL, "lsx_batch_create: n[%lld] = %lld outside [1, %d]", (long long)i,
                        (long long)n[i], BNMAX);
        hn[i] = (int32_t)n[i];
        aoff[i] = ta;
        voff[i] = tv;
        ta += n[i] * n[i];
        tv += n[i];
        const double nn = (double)n[i];
        flops += nn + nn * (nn - 1) / 2 + (nn - 1) * nn * (2 * nn - 1) / 3 + 2 * nn * nn;
    }
    std::vector<int32_t> order(count);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) { return hn[x] > hn[y]; });
    DeviceGuard g(ctx);
    lsx_batch* B = new (std::nothrow) lsx_batch();
    if (!B) return LSX_ENOMEM;
    B->ctx = ctx;
    B->dtype = dtype;
    B->count = count;
    B->total_a = ta;
    B->total_v = tv;
    B->flops = flops;
    const char* ng = std::getenv("LSX_BATCH_NO_GRAPH");
    B->use_graph = !(ng && ng[0] == '1');
    auto bad = [&](int rc) {
        batch_free(B);
        delete B;
        return rc;
    };
    if (hipStreamCreateWithFlags(&B->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&B->order, sizeof(int32_t) * count) != hipSuccess ||
        hipMalloc(&B->n, sizeof(int32_t) * count) != hipSuccess ||
        hipMalloc(&B->aoff, sizeof(int64_t) * count) != hipSuccess ||
        hipMalloc(&B->voff, sizeof(int64_t) * count) != hipSuccess ||
        (dtype == LSX_F64 && hipMalloc(&B->A, sizeof(double) * ta) != hipSuccess) ||
        hipMalloc(&B->dsrc, sizeof(double*)) != hipSuccess ||
        hipHostMalloc(&B->hsrc, sizeof(double*), hipHostMallocDefault) != hipSuccess ||
        (dtype == LSX_F32 && hipMalloc(&B->A32, sizeof(float) * ta) != hipSuccess) ||
        hipMalloc(&B->b, sizeof(double) * tv) != hipSuccess ||
        hipMalloc(&B->x, sizeof(double) * tv) != hipSuccess || hipMalloc(&B->ipiv, sizeof(int64_t) * tv) != hipSuccess ||
        hipMalloc(&B->perm, sizeof(int32_t) * tv) != hipSuccess ||
        hipMalloc(&B->info, sizeof(int64_t) * count) != hipSuccess ||
        hipMalloc(&B->iters, sizeof(int32_t) * count) != hipSuccess ||
        hipMalloc(&B->berr, sizeof(double) * count) != hipSuccess ||
        hipMalloc(&B->counter, 256) != hipSuccess ||
        hipHostMalloc(&B->hinfo, sizeof(int64_t) * count, hipHostMallocDefault) != hipSuccess)
        return bad(fail(ctx, LSX_ENOMEM, "lsx_batch_create: device allocation failed"));
    if (hipMemcpy(B->order, order.data(), sizeof(int32_t) * count, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(B->n, hn.data(), sizeof(int32_t) * count, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(B->aoff, aoff.data(), sizeof(int64_t) * count, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(B->voff, voff.data(), sizeof(int64_t) * count, hipMemcpyHostToDevice) != hipSuccess)
        return bad(fail(ctx, LSX_EHIP, "lsx_batch_create: upload failed"));
    *out = B;
    return LSX_OK;
}

int lsx_batch_destroy(lsx_batch* B) {
    if (!B) return LSX_EINVAL;
    DeviceGuard g(B->ctx);
    batch_free(B);
    delete B;
    return LSX_OK;
}

// (for callers of earlier versions: checks the table, which chooses nothing any more)
int lsx_batch_set_tiles(lsx_batch* B, int32_t nbins, const int32_t* upper, const int32_t* bw) {
    if (!B || nbins < 0 || (nbins > 0 && (!upper || !bw))) return LSX_EINVAL;
    lsx_ctx* ctx = B->ctx;
    for (int k = 0; k < nbins; ++k)
        if (bw[k] != 8 && bw[k] != 16 && bw[k] != PW)
            return fail(ctx, LSX_EINVAL, "lsx_batch_set_tiles: panel width %d is not 8, 16 or 32", bw[k]);
    return LSX_OK;
}

int lsx_batch_set_refinement(lsx_batch* B, double tol, int32_t max_iters) {
    if (!B || !(tol >= 0.0) || max_iters < 0) return LSX_EINVAL;
    B->tol = tol;
    B->maxref = max_iters;
    if (B->graph_exec) {  // the values are kernel arguments of the captured launch
        (void)hipGraphExecDestroy(B->graph_exec);
        B->graph_exec = nullptr;
    }
    return LSX_OK;
}

int lsx_batch_factor_solve(lsx_batch* B, const double* A, const double* b, double* x, int64_t* info,
                           int64_t* ipiv) {
    if (!B || !A || !b || !x) return LSX_EINVAL;
    lsx_ctx* ctx = B->ctx;
    DeviceGuard g(ctx);
    int rc = batch_run(B, A, b, x);
    if (rc) return rc;
    LSX_HIP(ctx, hipMemcpyAsync(B->hinfo, B->info, sizeof(int64_t) * B->count, hipMemcpyDeviceToHost, B->stream));
    if (info) LSX_HIP(ctx, hipMemcpyAsync(info, B->info, sizeof(int64_t) * B->count, hipMemcpyDefault, B->stream));
    if (ipiv) LSX_HIP(ctx, hipMemcpyAsync(ipiv, B->ipiv, sizeof(int64_t) * B->total_v, hipMemcpyDefault, B->stream));
    LSX_HIP(ctx, hipStreamSynchronize(B->stream));
    B->prof.collect();
    int nfail = 0;
    for (int64_t i = 0; i < B->count; ++i) nfail += B->hinfo[i] > 0;
    return nfail;
}

int lsx_batch_stats(lsx_batch* B, int32_t* iters, double* backward_error) {
    if (!B) return LSX_EINVAL;
    lsx_ctx* ctx = B->ctx;
    DeviceGuard g(ctx);
    if (iters) LSX_HIP(ctx, hipMemcpyAsync(iters, B->iters, sizeof(int32_t) * B->count, hipMemcpyDefault, B->stream));
    if (backward_error)
        LSX_HIP(ctx, hipMemcpyAsync(backward_error, B->berr, sizeof(double) * B->count, hipMemcpyDefault, B->stream));
    LSX_HIP(ctx, hipStreamSynchronize(B->stream));
    return LSX_OK;
}

}  // extern "C"
