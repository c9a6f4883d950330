// gmres_kernel.hpp — the persistent SimpleGMRES kernel: one workgroup's share of a solve.
//
// Follows src/simplegmres.jl (scalar layout):
//   reinit / _init_cacheval (:110-129, :420-462): x = 0, r0 = Pl \ b, beta = ||r0||,
//     eps = abstol + reltol * beta;
//   outer restart loop (:500-601): on passes >= 2, w = b - A x, r0 = Pl \ w;
//   Arnoldi step (:521-574): q = Pl \ (A (Pr \ v_k)); MGS h_i = <v_i, q>, q -= h_i v_i (i = 1..k);
//     Hbis = ||q||; previous Givens applied to the new column, new Givens (_sym_givens
//     :140-162); zeta update; stopping tests rNorm <= eps, rNorm + 1 <= 1, Hbis <= eps^(3/4);
//     v_{k+1} = q / Hbis;
//   back-substitution R y = z with zero for |R_ii| <= btol (:576-585), x_r += sum y_i v_i,
//     x_r = Pr \ x_r, x += x_r (:587-595); retcodes (:603-606).
//
// The modified Gram-Schmidt recurrence h_i = <v_i, q - sum_{j<i} h_j v_j> is the triangular system
// (I + L) h = V^T q with L[i][j] = <v_i, v_j>, j < i (the compact form of Gram-Schmidt, Swirydowicz
// et al., Numer. Linear Algebra Appl. 28, 2021).  So a step takes all its products <v_i, q>, and row
// k of L, in one pass over the basis and one exchange between the workgroups, solves the system
// redundantly in every workgroup, and takes its projections off q in a second pass: two exchanges
// per step instead of one per basis vector and two more.
// What bounds it: below about 2^17 rows the two exchanges (a store and a polled load through the
// memory side, each a few hundred ns) and the dependent loads of the sparse product; above that, the two
// passes over the basis.  So the rows are spread over as many workgroups as the exchange carries
// cheaply, and the first basis vectors live in LDS.  Measured against one exchange per basis vector
// (GMRES(30), 5-point grids): 100^2 to 1e-8, 27.0 -> 7.7 ms (5 -> 20 workgroups); 1024^2, 300 steps,
// 52.3 -> 30.3 ms (101 us a step); 4096 blocks of 16^2 at once, 6.23 -> 3.32 ms.
//
// Layout: workgroup w of P owns rows [w R, (w+1) R), R = NT * RPT, each thread RPT of them in
// registers (in pairs of neighbours from RPT = 2 on, for 16-byte loads).  Basis vectors are kept
// unnormalized, u_k with scale 1 / ||u_k||, so that one exchange of the norm also publishes the
// vector: the rows are written through to memory, and each workgroup adds its partial sum to the
// exchange only after its own writes have completed.  Every workgroup keeps its own copy of the
// Hessenberg/Givens scalars and computes them identically from identically summed values, so all
// workgroups take the same branches and a solve is bitwise reproducible.
#pragma once
#include <cfloat>
#include <cmath>

#include "gmres.hpp"
#include "wave.hpp"

namespace lsx {

constexpr int GSC = 32;             // basis vectors per exchange group
constexpr int GSV = 2 * GSC + 2;    // values of a group: two per vector, one for the current vector

template <int NT>
struct GShared {
    double part[NT / 64][GSV];  // wave sums of a group's products
    double wsum[2][NT / 64];    // wave sums of a norm
    uint32_t nbuf[2 * PMAX_G];  // received partial norms
    double cur;                 // last entry of the new Hessenberg column after the earlier rotations
    int inc;
    int abort;                  // a wait of this solve gave up: leave the solve
};

// ---- wave reductions
__device__ __forceinline__ double f64_of(uint32_t lo, uint32_t hi) { return __hiloint2double((int)hi, (int)lo); }
template <int CTRL> __device__ __forceinline__ double dpp_f64(double x) {
    return f64_of(dpp32<CTRL>((uint32_t)__double2loint(x)), dpp32<CTRL>((uint32_t)__double2hiint(x)));
}
// a + b with halves exchanged: lanes of the lower half (even rows of 16) get a's sum over the pair of
// halves (rows), the others b's.
__device__ __forceinline__ double fold32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(a), (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b), false, false);
    return f64_of(lo[0], hi[0]) + f64_of(lo[1], hi[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(a), (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b), false, false);
    return f64_of(lo[0], hi[0]) + f64_of(lo[1], hi[1]);
}
// M sums over the wave at once (M a power of two <= 16): at each exchange a lane gives away half
// of its values, so M sums cost about M exchanges instead of 6 M.  Lane l returns the sum of value
// l / (64 / M).  r is overwritten.
template <int M>
__device__ __forceinline__ double wave_sums(double (&r)[M]) {
    static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16, "a power of two up to 16");
    const int lane = threadIdx.x & 63;
    double t8[M >= 4 ? M / 4 : 1];
    if constexpr (M >= 4) {
#pragma unroll
        for (int j = 0; j < M / 2; ++j) r[j] = fold32(r[j], r[j + M / 2]);
#pragma unroll
        for (int j = 0; j < M / 4; ++j) t8[j] = fold16(r[j], r[j + M / 4]);
    } else {
        const double h = M == 2 ? fold32(r[0], r[M - 1]) : fold32(r[0], r[0]);
        t8[0] = fold16(h, h);
    }
    double s;
    if constexpr (M >= 8) {
        double t4[M / 8];
#pragma unroll
        for (int j = 0; j < M / 8; ++j) {
            const double a = t8[j], b = t8[j + M / 8];
            t4[j] = ((lane & 8) ? b : a) + dpp_f64<0x128>((lane & 8) ? a : b);  // row_ror:8: lane ^ 8
        }
        if constexpr (M == 16) {
            const double a = t4[0], b = t4[1];
            s = ((lane & 4) ? b : a) + dpp_f64<0x141>((lane & 4) ? a : b);  // row_half_mirror: lane ^ 7
        } else {
            s = t4[0] + dpp_f64<0x141>(t4[0]);
        }
    } else {
        s = t8[0] + dpp_f64<0x128>(t8[0]);
        s += dpp_f64<0x141>(s);
    }
    s += dpp_f64<0x4E>(s);  // quad_perm [2,3,0,1]: lane ^ 2
    s += dpp_f64<0xB1>(s);  // quad_perm [1,0,3,2]: lane ^ 1
    return s;
}
__device__ __forceinline__ double wave_sum(double v) {
    double r[1] = {v};
    return wave_sums<1>(r);
}
__device__ __forceinline__ double readlane_f64(double x, int l) {
    return f64_of((uint32_t)__builtin_amdgcn_readlane(__double2loint(x), l),
                  (uint32_t)__builtin_amdgcn_readlane(__double2hiint(x), l));
}

// Symmetric Givens rotation (src/simplegmres.jl:140-162).
__device__ __forceinline__ void sym_givens(double a, double b, double& c, double& s, double& rho) {
    auto sgn = [](double t) { return t > 0.0 ? 1.0 : (t < 0.0 ? -1.0 : 0.0); };
    if (b == 0.0) {
        c = (a == 0.0) ? 1.0 : sgn(a);
        s = 0.0;
        rho = fabs(a);
    } else if (a == 0.0) {
        c = 0.0;
        s = sgn(b);
        rho = fabs(b);
    } else if (fabs(b) > fabs(a)) {
        const double t = a / b;
        s = sgn(b) / sqrt(1.0 + t * t);
        c = s * t;
        rho = b / s;
    } else {
        const double t = b / a;
        c = sgn(a) / sqrt(1.0 + t * t);
        s = c * t;
        rho = a / c;
    }
}

// The solve on workgroup w of a.P (sh, dyn: the workgroup's static and dynamic LDS).  RG: the
// bookkeeping is in HBM (a.Rg) instead of LDS; a compile-time choice, so that each pointer below
// is known to be LDS or global memory and gets that memory's instructions.
template <int NT, int RPT, bool RG, bool MR = (RPT <= 4)>
struct GmresWg {
    static constexpr int R = NT * RPT;             // rows of the workgroup
    static constexpr int VW = RPT >= 2 ? 2 : 1;    // neighbouring rows per load
    static constexpr int NP = RPT / VW;            // loads per thread and vector
    static constexpr int NW = NT / 64;
    static constexpr int MAXE = 8;                 // entries of a row held in registers
    static constexpr bool MREG = MR;               // whether they are (else read on each product)
    typedef double dvec __attribute__((ext_vector_type(VW)));

    const GmresArgs& a;
    GShared<NT>& sh;
    int tid;                   // refreshed (below) once per pass of a loop
    const int w;
    const int row0;            // first row of this workgroup
    const int N;
    const int64_t ldv;
    uint32_t nred = 0;         // exchanges so far (sequence number of the messages)
    bool dead = false;         // a wait gave up (uniform in the workgroup): every loop ends
    double *Rm, *L, *cs, *sn, *z, *sc, *hs;  // bookkeeping
    double* us;                // own rows of the vector the sparse product reads (null: not kept)
    uint32_t* rbuf;            // received products
    double* Vc;                // the first a.ncache basis vectors' own rows
    int32_t ecol[MREG ? RPT : 1][MAXE];
    double eval[MREG ? RPT : 1][MAXE];
    int32_t ek0[MREG ? RPT : 1], ecnt[MREG ? RPT : 1];

    __device__ __forceinline__ GmresWg(const GmresArgs& a_, GShared<NT>& sh_, int w_, double* dyn)
        : a(a_), sh(sh_), tid((int)threadIdx.x), w(w_),
          row0(w_ * R), N((int)a_.N), ldv(a_.ldv) {
        const int64_t cap = a.cap;
        double* book = RG ? a.Rg + (size_t)w * (size_t)gmres_book_words(cap) : dyn;
        Rm = book;                          // packed columns, cap (cap + 1) / 2
        L = Rm + cap * (cap + 1) / 2;       // packed rows, cap (cap - 1) / 2
        cs = L + cap * (cap - 1) / 2;
        sn = cs + cap;
        z = sn + cap;                       // cap + 1
        sc = z + cap + 1;                   // cap + 1
        hs = sc + cap + 1;                  // cap + 1
        double* p = dyn + (RG ? 0 : gmres_book_words(cap));
        rbuf = reinterpret_cast<uint32_t*>(p);
        p += a.rbuf_len;
        us = a.own_lds ? p : nullptr;
        p += a.own_lds ? R : 0;
        Vc = p;
    }

    // Hides the thread's number from the compiler, which would otherwise compute the addresses of every
    // pass over the basis before the step loop, and spill them.
    __device__ __forceinline__ void refresh() { asm volatile("" : "+v"(tid)); }
    __device__ __forceinline__ int lane() const { return tid & 63; }
    __device__ __forceinline__ int wave() const { return __builtin_amdgcn_readfirstlane(tid >> 6); }
    __device__ __forceinline__ int loc(int i) const {  // own row of slot i, relative to row0
        return VW == 2 ? 2 * (tid + (i >> 1) * NT) + (i & 1) : tid + i * NT;
    }
    __device__ __forceinline__ int row(int i) const { return row0 + loc(i); }

    // ---- messages
    __device__ __forceinline__ uint64_t* slot(int v, int p) const {  // value v of workgroup p
        return a.red + 2 * (a.allread ? (int64_t)p * 2 * a.cap + v : (int64_t)v * a.P + p);
    }
    __device__ __forceinline__ uint64_t* total_slot(int v) const { return a.red + 4 * (int64_t)a.cap * a.P + 2 * v; }
    __device__ __forceinline__ uint64_t* norm_slot(int par, int p) const {
        return a.red + 4 * (int64_t)a.cap * (a.P + 1) + 2 * ((int64_t)par * a.P + p);
    }
    __device__ __forceinline__ void send(uint64_t* s, double v, uint32_t seq) const {
        st_relaxed_u64(s, ll_pack((uint32_t)__double2loint(v), seq));
        st_relaxed_u64(s + 1, ll_pack((uint32_t)__double2hiint(v), seq));
    }
    // Payloads of K flag-in-word messages (null: none) once they carry sequence number seq, all
    // reads in flight together.  The wait ends at the bound, or at once when any wait of this solve
    // has given up (the solve's error word is set); either way the workgroup's abort flag is raised,
    // read after the caller's barrier.
    template <int K>
    __device__ __forceinline__ void poll(const uint64_t* const (&word)[K], uint32_t (&out)[K], uint32_t seq) const {
        uint64_t x[K];
#pragma unroll
        for (int i = 0; i < K; ++i) x[i] = word[i] ? ld_relaxed_u64(word[i]) : ((uint64_t)seq << 32);
        bool stale = false;
#pragma unroll
        for (int i = 0; i < K; ++i) stale = stale || (uint32_t)(x[i] >> 32) != seq;
        if (stale) {
            const int64_t t0 = wall_clock64();
            for (unsigned spin = 0;; ++spin) {
                __builtin_amdgcn_s_sleep(1);  // back off: many workgroups poll the same words
#pragma unroll
                for (int i = 0; i < K; ++i)
                    if ((uint32_t)(x[i] >> 32) != seq) x[i] = ld_relaxed_u64(word[i]);
                stale = false;
#pragma unroll
                for (int i = 0; i < K; ++i) stale = stale || (uint32_t)(x[i] >> 32) != seq;
                if (!stale) break;
                if (wall_clock64() - t0 > a.timeout) {
                    atomicOr((unsigned long long*)&a.out->err, 1ull);
                    sh.abort = 1;
                    break;
                }
                if ((spin & 15) == 15 && ld_relaxed_u64(&a.out->err) != 0) {
                    sh.abort = 1;
                    break;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < K; ++i) out[i] = (uint32_t)x[i];
    }

    // Sum of v over all threads of all workgroups, the same bits in every thread.  Writes to global
    // memory made by agent-scope atomic stores before the call are complete in memory before any
    // workgroup returns from it.
    __device__ __forceinline__ double allreduce(double v) {
        const int par = (int)(nred & 1);
        const uint32_t seq = ++nred;
        v = wave_sum(v);
        if (lane() == 0) sh.wsum[par][wave()] = v;
        if (a.P > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NW; ++i) s += sh.wsum[par][i];
        if (a.P == 1) return s;
        if (tid == 0) send(norm_slot(par, w), s, seq);
        if (tid < 2 * a.P) {
            const uint64_t* const word[1] = {norm_slot(par, 0) + tid};
            uint32_t got[1];
            poll<1>(word, got, seq);
            sh.nbuf[tid] = got[0];
        }
        __syncthreads();
        dead = sh.abort != 0;
        // lane p adds partials p, p + 64, ...; then the wave sum: the same tree in every wave
        double t = 0.0;
        for (int p = lane(); p < a.P; p += 64) t += f64_of(sh.nbuf[2 * p], sh.nbuf[2 * p + 1]);
        return wave_sum(t);
    }

    // ---- the sparse product
    __device__ __forceinline__ void load_rows() {
        if constexpr (MREG) {
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                const int r = row(i);
                ek0[i] = r < N ? a.rowptr[r] : 0;
                ecnt[i] = r < N ? a.rowptr[r + 1] - ek0[i] : 0;
#pragma unroll
                for (int e = 0; e < MAXE; ++e) {
                    ecol[i][e] = e < ecnt[i] ? a.col[ek0[i] + e] : row0;
                    eval[i][e] = e < ecnt[i] ? a.val[ek0[i] + e] : 0.0;
                }
            }
        }
    }
    // entry j of the vector at src (own rows in us when kept)
    __device__ __forceinline__ double gather(int j, const double* src) const {
        const unsigned lj = (unsigned)(j - row0);
        const bool own = lj < (unsigned)R;
        double x = us ? us[own ? lj : 0u] : src[own ? j : row0];
        if (!own) x = ld_coherent_f64(src + j);
        return x;
    }
    // y_i = (A x)_r / pl_r, x the vector at src times s, for the rows of every slot i inside the
    // matrix (0 elsewhere); RES: (b - A x)_r / pl_r.  The terms of a row are added in ascending
    // column order without fusion (the order in which SparseArrays' CSC mul! accumulates a row); the
    // entries of SR rows are read together.
    template <bool RES>
    __device__ __forceinline__ void spmv(const double* src, double s, double (&y)[RPT]) const {
        constexpr int SR = (RPT < 2 || NT == 1024) ? 1 : 2;
#pragma unroll
        for (int i0 = 0; i0 < RPT; i0 += SR) {
            int k0[SR], cnt[SR];
            int32_t c[SR][MAXE];
            double v[SR][MAXE];
#pragma unroll
            for (int t = 0; t < SR; ++t) {
                if constexpr (MREG) {
                    k0[t] = ek0[i0 + t];
                    cnt[t] = ecnt[i0 + t];
                } else {
                    const int r = row(i0 + t);
                    k0[t] = r < N ? a.rowptr[r] : 0;
                    cnt[t] = r < N ? a.rowptr[r + 1] - k0[t] : 0;
                }
            }
#pragma unroll
            for (int t = 0; t < SR; ++t)
#pragma unroll
                for (int e = 0; e < MAXE; ++e) {
                    if constexpr (MREG) {
                        c[t][e] = ecol[i0 + t][e];
                        asm volatile("" : "+v"(c[t][e]));  // as refresh()
                        v[t][e] = eval[i0 + t][e];
                    } else {
                        c[t][e] = e < cnt[t] ? a.col[k0[t] + e] : row0;
                        v[t][e] = e < cnt[t] ? a.val[k0[t] + e] : 0.0;
                    }
                }
#pragma unroll
            for (int t = 0; t < SR; ++t) {
                double x[MAXE];
#pragma unroll
                for (int e = 0; e < MAXE; ++e) x[e] = gather(c[t][e], src);
                double acc = 0.0;
#pragma unroll
                for (int e = 0; e < MAXE; ++e) {
                    const double n = __dadd_rn(acc, __dmul_rn(v[t][e], RES ? x[e] : x[e] * s));
                    acc = e < cnt[t] ? n : acc;
                }
                for (int e = MAXE; e < cnt[t]; ++e) {
                    const double xe = gather(a.col[k0[t] + e], src);
                    acc = __dadd_rn(acc, __dmul_rn(a.val[k0[t] + e], RES ? xe : xe * s));
                }
                const int r = row(i0 + t);
                y[i0 + t] = 0.0;
                if (r < N) {
                    if (RES) acc = a.b[r] - acc;
                    y[i0 + t] = a.pl ? acc / a.pl[r] : acc;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- basis vectors
    // own entries of vector c that load p brings in: from LDS, or from memory with the rows past the
    // end replaced by the last ones inside (their q is zero, and what they give is not kept)
    template <bool LDS>
    __device__ __forceinline__ dvec vload(int c, int p) const {
        const int l = VW * (tid + p * NT);
        if constexpr (LDS) return *reinterpret_cast<const dvec*>(Vc + c * R + l);
        const int last = (int)ldv - VW;
        const int r = row0 + l;
        return *reinterpret_cast<const dvec*>(a.V + (int64_t)c * ldv + (r < last ? r : last));
    }
    // stores own rows u of vector c (zero past the end) where the passes read them, and u / pr where
    // the sparse products read it
    __device__ __forceinline__ void vstore(int c, const double (&u)[RPT]) {
        const bool cached = c < a.ncache;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int l = loc(i), r = row0 + l;
            double g = u[i];
            if (a.pr && r < N) g /= a.pr[r];
            if (us) us[l] = g;
            if (cached) Vc[c * R + l] = u[i];
            if (r < ldv) {
                double* dst = a.V + (int64_t)c * ldv + r;
                double* pub = a.pr ? a.xp + r : dst;
                if (a.pr || a.P == 1) {
                    if (!cached) *dst = u[i];
                }
                if (a.P > 1) st_relaxed_u64((uint64_t*)pub, (uint64_t)__double_as_longlong(g));
                else if (!us) *pub = g;
            }
            if (i & 1) __builtin_amdgcn_sched_barrier(0);  // not every row's division at once
        }
    }
    // Products of vectors c0 .. c1 - 1 with q and u, summed over the wave into sh.part (slots
    // 2 (c - g0) + 0 / 1), CH vectors at a time.  The last group repeats its last vector (read again
    // from the nearest cache); with up to two rows per thread the last one to four vectors have a body of
    // their own (memory 5: blocks of 64 to 529 rows 3 to 5 % faster), beyond that another body means
    // another copy of q and u, which spill.
    static constexpr int CH = RPT >= 8 ? 4 : 8, TAIL = 4;
    template <bool LDS>
    __device__ __forceinline__ void dots(int c0, int c1, int g0, const double (&q)[RPT], const double (&u)[RPT]) {
        if constexpr (RPT > 2) {
            dots_by<LDS, CH, false>(c0, c1, g0, q, u);
        } else {
            int c = c0;
            for (; c1 - c > TAIL; c += CH) dots_by<LDS, CH, true>(c, c1, g0, q, u);
            if (c < c1) dots_by<LDS, TAIL, true>(c, c1, g0, q, u);
        }
    }
    // (ONE: the first group alone)
    template <bool LDS, int M, bool ONE>
    __device__ __forceinline__ void dots_by(int c0, int c1, int g0, const double (&q)[RPT], const double (&u)[RPT]) {
        for (int c = c0; c < c1; c += M) {
            double r[2 * M];
#pragma unroll
            for (int j = 0; j < 2 * M; ++j) r[j] = 0.0;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                dvec v[M];
#pragma unroll
                for (int j = 0; j < M; ++j) v[j] = vload<LDS>(min(c + j, c1 - 1), p);
#pragma unroll
                for (int j = 0; j < M; ++j)
#pragma unroll
                    for (int t = 0; t < VW; ++t) {
                        r[2 * j] = fma(v[j][t], q[VW * p + t], r[2 * j]);
                        r[2 * j + 1] = fma(v[j][t], u[VW * p + t], r[2 * j + 1]);
                    }
            }
            constexpr int G = 64 / (2 * M);  // lanes that hold the same sum
            const double s = wave_sums<2 * M>(r);
            const int x = lane() / G;
            if ((lane() & (G - 1)) == 0 && c + (x >> 1) < c1) sh.part[wave()][2 * (c - g0) + x] = s;
            if constexpr (ONE) break;
        }
    }
    // q += sum over vectors c0 .. c1 - 1 of f_c u_c, f_c = sign coef[c] sc[c]
    template <bool LDS>
    __device__ __forceinline__ void axpys(int c0, int c1, double sign, const double* coef, double (&q)[RPT]) const {
        if constexpr (RPT > 2) {
            axpys_by<LDS, CH, false>(c0, c1, sign, coef, q);
        } else {
            int c = c0;
            for (; c1 - c > TAIL; c += CH) axpys_by<LDS, CH, true>(c, c1, sign, coef, q);
            if (c < c1) axpys_by<LDS, TAIL, true>(c, c1, sign, coef, q);
        }
    }
    template <bool LDS, int M, bool ONE>
    __device__ __forceinline__ void axpys_by(int c0, int c1, double sign, const double* coef, double (&q)[RPT]) const {
        for (int c = c0; c < c1; c += M) {
            double f[M];
#pragma unroll
            for (int j = 0; j < M; ++j) {
                const int cj = min(c + j, c1 - 1);
                f[j] = c + j < c1 ? sign * (coef[cj] * sc[cj]) : 0.0;
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                dvec v[M];
#pragma unroll
                for (int j = 0; j < M; ++j) v[j] = vload<LDS>(min(c + j, c1 - 1), p);
#pragma unroll
                for (int j = 0; j < M; ++j)
#pragma unroll
                    for (int t = 0; t < VW; ++t) q[VW * p + t] = fma(f[j], v[j][t], q[VW * p + t]);
            }
            if constexpr (ONE) break;
        }
    }

    // value v of the step (even: <u_{v/2}, q>, odd: <u_{v/2}, u_k>), summed over all workgroups
    __device__ __forceinline__ void put(int v, double t, int k) {
        const int i = v >> 1;
        if (v & 1) L[(int64_t)(k - 1) * (k - 2) / 2 + i] = t * sc[i] * sc[k - 1];
        else hs[i] = t * sc[i];
    }
    // All products of step k into hs (<v_i, q>, i < k) and row k of L.
    __device__ __forceinline__ void products(int k, const double (&q)[RPT], const double (&u)[RPT]) {
        const uint32_t seq = ++nred;
        const int P = a.P;
        for (int g0 = 0;; g0 += GSC) {
            const int g1 = min(k - 1, g0 + GSC);
            const bool last = g1 == k - 1;
            const int nc = max(g0, min(g1, a.ncache));
            dots<true>(g0, nc, g0, q, u);
            dots<false>(nc, g1, g0, q, u);
            if (last) {
                double own = 0.0;
#pragma unroll
                for (int i = 0; i < RPT; ++i) own = fma(u[i], q[i], own);
                own = wave_sum(own);
                if (lane() == 0) sh.part[wave()][2 * (g1 - g0)] = own;
            }
            __syncthreads();
            const int nv = 2 * (g1 - g0) + (last ? 1 : 0), v0 = 2 * g0;
            if (tid < nv) {
                double s = 0.0;
#pragma unroll
                for (int i = 0; i < NW; ++i) s += sh.part[i][tid];
                if (P == 1) put(v0 + tid, s, k);
                else send(slot(v0 + tid, w), s, seq);
            }
            if (P > 1) exchange(nv, v0, k, seq);
            if (last) break;
            __syncthreads();
            if (dead) return;
        }
        __syncthreads();
    }
    // Sums values v0 .. v0 + nv - 1 of the step over the workgroups.  Up to GALL workgroups, each
    // reads all partial values; beyond, workgroup (v - v0) mod P sums value v and publishes the
    // total (the reads would grow as P^2).  Every sum has one fixed order.
    __device__ __forceinline__ void exchange(int nv, int v0, int k, uint32_t seq) {
        const int P = a.P;
        if (a.allread) {
            // rounds of as many values as the receive buffer holds: wave i reads the words of
            // workgroups i, i + NW, ...
            constexpr int KP = (GALL + NW - 1) / NW;
            const int chunk = min(64, (int)(a.rbuf_len / P));
            for (int c0 = 0; c0 < nv; c0 += chunk) {
                const int nw = 2 * min(chunk, nv - c0);
                const uint64_t* word[2 * KP];
                uint32_t got[2 * KP];
#pragma unroll
                for (int j = 0; j < KP; ++j)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int p = wave() + j * NW, x = lane() + 64 * h;
                        word[2 * j + h] = (p < P && x < nw) ? slot(v0 + c0, p) + x : nullptr;
                    }
                poll<2 * KP>(word, got, seq);
#pragma unroll
                for (int j = 0; j < KP; ++j)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int p = wave() + j * NW, x = lane() + 64 * h;
                        if (p < P && x < nw) rbuf[p * nw + x] = got[2 * j + h];
                    }
                __syncthreads();
                dead = sh.abort != 0;
                // four threads per value, each every fourth workgroup
                const int v = tid >> 2, sub = tid & 3;
                for (int vv = v; 2 * vv < nw; vv += NT / 4) {
                    double s = 0.0;
                    for (int p = sub; p < P; p += 4) s += f64_of(rbuf[p * nw + 2 * vv], rbuf[p * nw + 2 * vv + 1]);
                    s += dpp_f64<0xB1>(s);
                    s += dpp_f64<0x4E>(s);
                    if (sub == 0) put(v0 + c0 + vv, s, k);
                }
                if (c0 + chunk < nv) __syncthreads();
            }
        } else {
            for (int j = wave(); w + j * P < nv; j += NW) {
                const int v = v0 + w + j * P;
                const uint64_t* word[2 * (PMAX_G / 64)];
                uint32_t got[2 * (PMAX_G / 64)];
#pragma unroll
                for (int t = 0; t < PMAX_G / 64; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        word[2 * t + h] = lane() + 64 * t < P ? slot(v, lane() + 64 * t) + h : nullptr;
                poll<2 * (PMAX_G / 64)>(word, got, seq);
                double s = 0.0;
#pragma unroll
                for (int t = 0; t < PMAX_G / 64; ++t) s += lane() + 64 * t < P ? f64_of(got[2 * t], got[2 * t + 1]) : 0.0;
                s = wave_sum(s);
                if (lane() == 0) send(total_slot(v), s, seq);
            }
            if (tid < nv) {
                const uint64_t* const word[2] = {total_slot(v0 + tid), total_slot(v0 + tid) + 1};
                uint32_t got[2];
                poll<2>(word, got, seq);
                put(v0 + tid, f64_of(got[0], got[1]), k);
            }
            __syncthreads();
            dead = sh.abort != 0;
        }
    }
    // hs := (I + L)^{-1} hs (k unknowns), by blocks of 64: the contributions of earlier blocks by all
    // threads, the block itself by one wave (lane j keeps unknown j, each solved one is broadcast).
    __device__ __forceinline__ void subst(int k) {
        for (int b0 = 0; b0 < k; b0 += 64) {
            const int nb = min(64, k - b0);
            if (b0 > 0) {
                constexpr int TR = NT / 64;  // threads per unknown: 4, 8 or 16 (a row of lanes at most)
                static_assert(TR == 4 || TR == 8 || TR == 16, "the sum over an unknown's threads");
                const int j = b0 + tid / TR, sub = tid % TR;
                double s = 0.0;
                if (j < k) {
                    const double* Lj = L + (int64_t)j * (j - 1) / 2;
                    for (int i = sub; i < b0; i += TR) s = fma(Lj[i], hs[i], s);
                }
                s += dpp_f64<0xB1>(s);
                s += dpp_f64<0x4E>(s);
                if constexpr (TR > 4) s += dpp_f64<0x141>(s);  // row_half_mirror
                if constexpr (TR > 8) s += dpp_f64<0x140>(s);  // row_mirror
                if (sub == 0 && j < k) hs[j] -= s;
                __syncthreads();
            }
            if (wave() == 0) {
                const int j = b0 + lane();
                const double* Lj = L + (int64_t)j * (j - 1) / 2 + b0;
                double h = lane() < nb ? hs[j] : 0.0;
                for (int i0 = 0; i0 < nb - 1; i0 += 8) {
                    double l[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) l[t] = (lane() < nb && i0 + t < lane()) ? Lj[i0 + t] : 0.0;
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const double hi = readlane_f64(h, (i0 + t) & 63);
                        if (i0 + t < lane()) h = fma(-l[t], hi, h);
                    }
                }
                if (lane() < nb) hs[j] = h;
            }
            __syncthreads();
        }
    }

    __device__ __forceinline__ void run() {
        if (tid == 0) sh.abort = 0;  // ordered before any poll by the first all-reduce's barrier
        double q[RPT], u[RPT];
        load_rows();
        double part = 0.0;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const int r = row(i);
            q[i] = 0.0;
            if (r < N) {
                q[i] = a.pl ? a.b[r] / a.pl[r] : a.b[r];
                part = fma(q[i], q[i], part);
            }
            if (i & 1) __builtin_amdgcn_sched_barrier(0);
        }
        vstore(0, q);
        const double beta0 = sqrt(allreduce(part));
        const double eps_ = a.abstol + a.reltol * beta0;
        double rNorm = beta0;
        int64_t iter = 0;
        int status = LSX_RET_DEFAULT;
        bool first = true;  // no pass has begun
        bool written = false;  // x holds an iterate
        if (dead) {
            // a wait gave up: the error word tells the host, nothing else is computed
        } else if (beta0 == 0.0) {
            status = LSX_RET_SUCCESS;
        } else {
            const double btol = 1.8189894035458565e-12;  // eps^(3/4) = 2^-39
            bool breakdown = false, inconsistent = false;
            bool solved = rNorm <= eps_;
            int64_t inner_maxiters = a.maxiters;
            bool tired = iter >= a.maxiters;
            double nrm = beta0;
            while (!(solved || tired || breakdown || dead)) {
                if (!first) {
                    // r0 = Pl \ (b - A x): x complete in every workgroup before the product reads it
                    if (a.P > 1) (void)allreduce(0.0);
                    else __syncthreads();
                    if (dead) break;
                    spmv<true>(a.x, 1.0, q);
                    part = 0.0;
#pragma unroll
                    for (int i = 0; i < RPT; ++i) part = fma(q[i], q[i], part);
                    __syncthreads();  // own rows of x are no longer read from us
                    vstore(0, q);
                    nrm = sqrt(allreduce(part));
                    if (dead) break;
                }
                first = false;
                // zeta_1 = ||r0||, v_1 = r0 / ||r0||
                double zeta = nrm;
                int64_t nr = 0;
                int k = 0;
                bool inner_tired = false;
                while (!(solved || inner_tired || breakdown || dead)) {
                    ++k;
                    refresh();
                    const double s = 1.0 / nrm;
                    if (tid == 0) sc[k - 1] = s;
                    // q = Pl \ (A (Pr \ v_k))
#pragma unroll
                    for (int i = 0; i < RPT; ++i) u[i] = q[i];
                    spmv<false>(a.pr ? a.xp : a.V + (int64_t)(k - 1) * ldv, s, q);
                    products(k, q, u);
                    if (dead) break;
                    if (k > 1) subst(k);
                    refresh();
                    // q -= sum_i h_i v_i
                    {
                        const int nc = min(k - 1, a.ncache);
                        axpys<true>(0, nc, -1.0, hs, q);
                        axpys<false>(nc, k - 1, -1.0, hs, q);
                        const double f = hs[k - 1] * s;
                        part = 0.0;
#pragma unroll
                        for (int i = 0; i < RPT; ++i) {
                            q[i] = row(i) < N ? fma(-f, u[i], q[i]) : 0.0;
                            part = fma(q[i], q[i], part);
                        }
                    }
                    vstore(k, q);
                    // the earlier rotations on the new column, while the norm travels
                    if (tid == NT - 64) {
                        double cur = hs[0];
                        for (int i = 1; i <= k - 1; ++i) {
                            const double nx = hs[i], ci = cs[i - 1], si = sn[i - 1];
                            Rm[nr + i - 1] = ci * cur + si * nx;
                            cur = si * cur - ci * nx;
                        }
                        sh.cur = cur;
                    }
                    const double Hbis = sqrt(allreduce(part));
                    if (dead) break;
                    double c_, s_, rho;
                    sym_givens(sh.cur, Hbis, c_, s_, rho);
                    if (tid == NT - 64) {
                        cs[k - 1] = c_;
                        sn[k - 1] = s_;
                        Rm[nr + k - 1] = rho;
                        z[k - 1] = c_ * zeta;
                    }
                    zeta = s_ * zeta;  // consumed only if the iteration continues
                    rNorm = fabs(zeta);
                    nr += k;
                    nrm = Hbis;
                    const bool mach = (rNorm + 1.0 <= 1.0);
                    const bool lim = rNorm <= eps_;
                    breakdown = Hbis <= btol;
                    solved = lim || mach;
                    inner_tired = a.restart ? (k >= (int64_t)min((int64_t)a.memory, inner_maxiters))
                                            : (k >= inner_maxiters);
                }
                if (dead) break;
                __syncthreads();
                // back-substitution R y = z (y overwrites z)
                if (tid == 0) {
                    int inc = 0;
                    for (int i = k; i >= 1; --i) {
                        int64_t pos = nr + i - k;
                        double y = z[i - 1];
                        for (int j = k; j >= i + 1; --j) {
                            y = y - Rm[pos - 1] * z[j - 1];
                            pos = pos - j + 1;
                        }
                        if (fabs(Rm[pos - 1]) <= btol) {
                            y = 0.0;
                            inc = 1;
                        } else {
                            y = y / Rm[pos - 1];
                        }
                        z[i - 1] = y;
                    }
                    sh.inc = inc;
                }
                __syncthreads();
                inconsistent = inconsistent || sh.inc;
                // x_r = Pr \ sum_i y_i v_i; x += x_r
#pragma unroll
                for (int i = 0; i < RPT; ++i) u[i] = 0.0;
                {
                    const int nc = min(k, a.ncache);
                    axpys<true>(0, nc, 1.0, z, u);
                    axpys<false>(nc, k, 1.0, z, u);
                }
                const bool more = a.restart != 0;  // another pass may read x
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const int r = row(i);
                    double xn = 0.0;
                    if (r < N) {
                        double acc = u[i];
                        if (a.pr) acc = acc / a.pr[r];
                        xn = written ? a.x[r] + acc : acc;
                        if (more && a.P > 1) st_relaxed_u64((uint64_t*)(a.x + r), (uint64_t)__double_as_longlong(xn));
                        else a.x[r] = xn;
                    }
                    if (us) us[loc(i)] = xn;
                    if (i & 1) __builtin_amdgcn_sched_barrier(0);
                }
                written = true;
                inner_maxiters -= k;
                iter += k;
                tired = iter >= a.maxiters;
            }
            if (tired) status = LSX_RET_MAXITERS;
            if (solved) status = LSX_RET_SUCCESS;
            if (inconsistent) status = LSX_RET_INFEASIBLE;
        }
        if (!written) {
#pragma unroll
            for (int i = 0; i < RPT; ++i)
                if (row(i) < N) a.x[row(i)] = 0.0;
        }
        if (w == 0 && tid == 0) {
            a.out->retcode = status;
            a.out->iters = iter;
            a.out->resid = rNorm;
        }
    }
};

}  // namespace lsx
