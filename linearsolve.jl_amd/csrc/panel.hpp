// panel.hpp — one panel of partial-pivot LU held in the registers of a workgroup: the columns' chain
// shared by the blocked LU (lu_kernels.hpp) and the batched LU (batch.hip).
//
// Pivot search: maximum |a| with NaN ignored, first (smallest) row on ties
// (src/blocked_lufact.jl:38-54); zero pivot -> info = first such column, factorization
// continues (src/generic_lufact.jl:71-141).  Scaling multiplies by the reciprocal of the pivot
// (blocked_lufact.jl:110-113) unless |pivot| < the smallest normal number (then divides, as
// LAPACK dgetf2).
#pragma once
#include <climits>
#include <limits>

#include "wave.hpp"

namespace lsx {
constexpr int PW = 32;        // panel width held in registers

// Words (32-bit) per element of an exchange record, and word i of an element.
template <typename T> struct Words;
template <> struct Words<double> {
    static constexpr int W = 2;
    __device__ static uint32_t word(double x, int i) { return (uint32_t)(i ? __double2hiint(x) : __double2loint(x)); }
};
template <> struct Words<float> {
    static constexpr int W = 1;
    __device__ static uint32_t word(float x, int) { return __float_as_uint(x); }
};
// Candidate record: key, logical row, 1 / candidate, and the candidate row in the panel's register
// layout.
template <typename T>
struct __align__(16) PanelRec {
    uint64_t key;
    int row;
    int pad;
    T inv;
    T pad2[16 / sizeof(T) - 1];
    T v[PW];
};
// Message words ahead of the row's entries: key (2), row, pad, inverse.
template <typename T> constexpr int panel_head() { return 4 + Words<T>::W; }

// Each thread holds RPT rows of the panel in registers.  Columns go by groups of eight: within a
// group the code of column c is unrolled and its slot is v[.][c]; after a group the slots rotate by
// eight, so the loop body is one group's code (it stays in the instruction cache) and every register
// index is static.  Rows do not move while the panel is factored: each carries the logical row index
// lr of the row it holds.  The interchange of column k relabels two rows (the pivot row's becomes k,
// the one labelled k takes the pivot row's old label) and marks the pivot row finished; at the end
// every row is written to its logical position, and the rows that moved are listed for the
// interchanges of the other columns.  Ties of the pivot search are broken by the logical index, as an
// explicit row interchange would.
// A column is a chain of latencies: the pivot search in the wave (32-bit steps), the waves' keys through
// LDS, the winner's row written to LDS by its own thread, and read back as one value per lane of a row of
// 16 lanes, from where the update broadcasts it by DPP (an LDS read per entry and wave would be bound by
// LDS bandwidth).  About 1 us a column, of which 40 % are waits and none dominates: writing every wave's
// candidate row ahead of a single barrier, or the broadcast as moves of its own, measured the same
// within 5 %.
// Measured per 32-column panel against a rotating layout (one slot per column, selects instead of
// static slots, 64-bit search steps, an LDS read per pivot-row entry, 512 rows per workgroup): 256
// rows 59 -> 32 us, 512 rows 70 -> 38 us, 1024 rows 105 -> 47 us, 16384 rows 124 -> 105 us.

// v[S + q] += nl * (lane (S & 15) + q of the row of 16 lanes' pr), q = FROM .. 7, with the broadcast as the
// fused multiply-add's own DPP operand (one instruction per entry; the compiler makes two).  The DPP
// operand must not have been written by the two instructions before: s_nop 1 keeps that true whatever
// the compiler places there.  All lanes active.
template <int S, int FROM>
__device__ __forceinline__ void fmac_row(double (&v)[PW], double pr, double nl) {
#define LSX_FM(i) "v_fmac_f64_dpp %" #i ", %8, %9 row_newbcast:%1" #i " row_mask:0xf bank_mask:0xf\n\t"
    if constexpr (FROM == 0) {
        asm("s_nop 1\n\t" LSX_FM(0) LSX_FM(1) LSX_FM(2) LSX_FM(3) LSX_FM(4) LSX_FM(5) LSX_FM(6) LSX_FM(7)
            : "+v"(v[S]), "+v"(v[S + 1]), "+v"(v[S + 2]), "+v"(v[S + 3]), "+v"(v[S + 4]), "+v"(v[S + 5]), "+v"(v[S + 6]),
              "+v"(v[S + 7])
            : "v"(pr), "v"(nl), "n"((S & 15) + 0), "n"((S & 15) + 1), "n"((S & 15) + 2), "n"((S & 15) + 3),
              "n"((S & 15) + 4), "n"((S & 15) + 5), "n"((S & 15) + 6), "n"((S & 15) + 7));
    } else if constexpr (FROM < 8) {
        asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
            : "+v"(v[S + FROM])
            : "v"(pr), "v"(nl), "n"((S & 15) + FROM));
        fmac_row<S, FROM + 1>(v, pr, nl);
    }
#undef LSX_FM
}
template <int S, int FROM>
__device__ __forceinline__ void fmac_row(float (&v)[PW], float pr, float nl) {
    if constexpr (FROM < 8) {
        asm("s_nop 1\n\tv_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
            : "+v"(v[S + FROM])
            : "v"(pr), "v"(nl), "n"((S & 15) + FROM));
        fmac_row<S, FROM + 1>(v, pr, nl);
    }
}

struct PanelCand {
    uint64_t key;
    int row, pad;
};
template <typename T, int NW>
struct PanelLds {
    PanelCand cand[NW];     // each wave's best key and row
    PanelRec<T> fin[PW];    // per column: the workgroup's best row (with one workgroup, the pivot row)
    int piv[PW];
};

// v: the rows (panel column q in slot q); lr, live: their labels (logical rows, j0 ..) and whether they
// may still become a pivot; W columns; labels lie in [j0, m).  exchange(rec, column, sender) turns the
// workgroup's winning record (written by the wave whose sender is true) into the panel's, past a barrier.
// piv[c] (LDS): the logical row interchanged with row j0 + c; info: 1 + the first column (from 0, in the
// matrix) whose pivot is zero (FP32 without FEW: zero, NaN or without a reciprocal), if it was 0.  On return row lr is row j0 + i (i < W): its columns are
// fin[i] (LDS, after a barrier); of the other rows slot q holds column (q + 8 ceil(W / 8)) mod PW.
// FEW (one workgroup): panels may have far fewer rows than NT RPT and fewer than PW columns, and other
// workgroups of the CU use what the waves without rows leave: those only take part in the barriers, a
// thread's second row and the groups of slots past the last column are skipped where there are none, and a
// panel of one wave needs no barriers.  info is then valid in the waves with rows (the first among them).
template <typename T, int NT, int RPT, bool FEW, typename EX>
__device__ __forceinline__ void panel_columns(T (&v)[RPT][PW], int (&lr)[RPT], bool (&live)[RPT], int W, int j0, int m,
                                              PanelLds<T, NT / 64>& sh, int& info, EX&& exchange) {
    constexpr int NW = NT / 64;
    static_assert(NW == 2 || NW == 4 || NW == 8 || NW == 16, "the search among the waves takes up to sixteen candidates");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool one = FEW && m - j0 <= 64;                           // one wave has all the rows
    const bool two = RPT > 1 && (!FEW || j0 + NT + 64 * wave < m);  // this wave has second rows
    if (FEW && j0 + 64 * wave >= m) {
        if (one) return;
        if (lane == 0) {
            sh.cand[wave].key = 0;
            sh.cand[wave].row = INT_MAX;
        }
        for (int c = 0; c < 2 * W; ++c) __syncthreads();  // two per column
        return;
    }
#pragma unroll 1
    for (int g = 0; g < PW / 8; ++g) {
        if (8 * g >= W) break;
        const int nb = (FEW ? (W + 7) / 8 : 4) - g;  // groups of eight slots that hold columns not yet finished
        // columns of slots lane & 15 and 16 + (lane & 15)
        const int ca = ((lane & 15) + 8 * g) & (PW - 1), cb = ca ^ 16;
        static_for<0, 8>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            const int col = 8 * g + c;
            if (col >= W) return;  // uniform: only the last panel is narrower
            const int k = j0 + col;
            // the workgroup's candidate
            uint64_t key = live[0] ? pivot_key(v[0][c]) : 0;
            int krow = lr[0];
            T best = v[0][c];
            bool second = false;
            if (RPT > 1 && two) {
                const uint64_t k1 = live[RPT - 1] ? pivot_key(v[RPT - 1][c]) : 0;
                second = k1 > key || (k1 == key && lr[RPT - 1] < krow);
                key = second ? k1 : key;
                krow = second ? lr[RPT - 1] : krow;
                best = second ? v[RPT - 1][c] : best;
            }
            const T binv = T(1) / best;  // formed in the shadow of the search
            const int wl = wave_argmax32(key, krow);
            int wi = 0;
            if (!one) {
                if (lane == wl) {
                    sh.cand[wave].key = key;
                    sh.cand[wave].row = krow;
                }
                __syncthreads();
                const PanelCand cd = sh.cand[lane & (NW - 1)];
                wi = wave_argmax_rep<NW>(cd.key, cd.row);
            }
            PanelRec<T>& rec = sh.fin[col];
            if (wave == wi && lane == wl) {
                rec.key = key;
                rec.row = krow;
                rec.inv = binv;
                // (the asm statements keep the two branches from being merged into one that indexes v)
                auto put = [&](const T (&r)[PW]) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        T* to = rec.v + 8 * ((b + g) & 3);
#pragma unroll
                        for (int q = 0; q < 8; ++q) to[q] = r[8 * b + q];
                    }
                };
                if (RPT > 1 && second) {
                    put(v[RPT - 1]);
                    asm volatile("; second row" ::: "memory");
                } else {
                    put(v[0]);
                    asm volatile("; first row" ::: "memory");
                }
            }
            const PanelRec<T>* win = &rec;
            if (one) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            else win = exchange(&rec, col, wave == wi);
            int grow = win->row;
            const T pv = win->v[col], inv = win->inv;
            const T pa = win->v[ca], pb = win->v[cb];
            // interchange of column k with pivot row grow (relabelling), pivots and info.  A live row
            // always wins the pivot search, so grow lies in [k, m); only a record left stale by a wait
            // that gave up (the factorization then reports LSX_ETIMEOUT) could hold another label, and
            // it is replaced by k so that every later row index stays inside the matrix.
            if (grow < k || grow >= m) grow = k;
            if (tid == 0) sh.piv[col] = grow;
            // FP32 factors to be refined (not FEW): neither a NaN pivot nor one without an FP32 reciprocal
            // (the matrix is not finite, or out of FP32's range) gives factors to refine with
            const bool bad = sizeof(T) == 4 && !FEW ? !(fabs(inv) <= std::numeric_limits<T>::max()) : pv == T(0);
            if (bad && info == 0) info = k + 1;
            const bool normal = fabs(pv) >= std::numeric_limits<T>::min();
            T nl[RPT];
#pragma unroll
            for (int t = 0; t < RPT; ++t) {
                if (t > 0 && !two) continue;
                live[t] = live[t] && lr[t] != grow;
                lr[t] = lr[t] == grow ? k : (lr[t] == k ? grow : lr[t]);
                T l = v[t][c] * inv;
                if (!normal) l = pv != T(0) ? v[t][c] / pv : v[t][c];
                v[t][c] = l;
                nl[t] = live[t] ? -l : T(0);  // a finished row's registers do not matter any more
            }
#pragma unroll
            for (int t = 0; t < RPT; ++t)
                if (t == 0 || two) fmac_row<0, c + 1>(v[t], pa, nl[t]);
#pragma unroll
            for (int b = 1; b < 4; ++b)
                if (b < nb) {
#pragma unroll
                    for (int t = 0; t < RPT; ++t) {
                        if (t > 0 && !two) continue;
                        if (b == 1) fmac_row<8, 0>(v[t], pa, nl[t]);
                        else if (b == 2) fmac_row<16, 0>(v[t], pb, nl[t]);
                        else fmac_row<24, 0>(v[t], pb, nl[t]);
                    }
                }
        });
        // the next group's columns to slots 0 .. 7
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            if (t > 0 && !two) continue;
            T done[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) done[q] = v[t][q];
#pragma unroll
            for (int q = 0; q < PW - 8; ++q) v[t][q] = v[t][q + 8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[t][PW - 8 + q] = done[q];
        }
    }
}

}  // namespace lsx
