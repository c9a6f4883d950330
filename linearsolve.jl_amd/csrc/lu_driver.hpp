// lu_driver.hpp — the blocked right-looking getrf and the getrs of the resident factors,
// templated on the working type; the trailing-update GEMM is supplied by the caller (FP64 MFMA
// for the plain path, FP32 or BF16 MFMA for the mixed path).
//
// Structure of LAPACK dgetrf and of src/blocked_lufact.jl:658-679, with two block levels:
// outer blocks of NBO to 4 NBO columns (K of the trailing update; the last one wider) split into inner
// panels of PW columns.
#pragma once
#include <algorithm>

#include "coop.hpp"
#include "gemm.hpp"
#include "lu_kernels.hpp"

namespace lsx {

template <typename T>
static void launch_panel_t(lsx_lu* lu, T* F, int64_t ld, int64_t j0, int W, int64_t* list, int* count) {
    const int64_t m_rows = lu->n - j0;
    PanelArgs<T> a;
    a.A = F;
    a.ld = ld;
    a.m = lu->n;
    a.j0 = j0;
    a.W = W;
    a.ipiv = lu->ipiv;
    a.dinfo = lu->dinfo;
    a.slots = lu->slots;
    a.seq = lu->seq;
    a.timeout = wait_ticks(lu->ctx, 5.0);
    a.list = list;
    a.count = count;
    lu->seq += (uint32_t)W + 1u;
    const int pi = lu->prof.begin(lu->cur, PK_PANEL, (double)m_rows * W * W,
                                  2.0 * sizeof(T) * (double)m_rows * W);
    // one row per thread while 512 threads cover the panel, then two: the fewest entries to update per
    // column (256 rows 32 us, 512 rows 38 us per panel), and no exchange between workgroups up to 1024
    // rows (47 us; two workgroups of 512 rows took 105)
    a.P = (int)cdiv(m_rows, PROWS);
    if (m_rows <= 256) hipLaunchKernelGGL((k_panel<T, 256, 1>), dim3(1), dim3(256), 0, lu->cur, a);
    else if (m_rows <= 512) hipLaunchKernelGGL((k_panel<T, 512, 1>), dim3(1), dim3(512), 0, lu->cur, a);
    else if (sizeof(T) == 8 || m_rows <= 1024 || m_rows > 2048)
        hipLaunchKernelGGL((k_panel<T, 512, 2>), dim3(a.P), dim3(512), 0, lu->cur, a);
    else if constexpr (sizeof(T) == 4) {
        // FP32 rows leave the registers for 2048 rows in one workgroup: still no exchange (with refinement,
        // n = 2000 5.08 -> 4.10 ms, 9000 34.4 -> 33.2); two or more such workgroups are slower than twice as many of 1024
        a.P = 1;
        hipLaunchKernelGGL((k_panel<T, 1024, 2>), dim3(1), dim3(1024), 0, lu->cur, a);
    }
    lu->prof.end(lu->cur, pi);
}

template <typename T>
static void launch_laswp_t(lsx_lu* lu, T* F, int64_t ld, int kb, const int64_t* list, const int* count, int64_t c0,
                           int64_t c1) {
    if (c1 <= c0) return;
    const int pi = lu->prof.begin(lu->cur, PK_LASWP, 0.0, sizeof(T) * 4.0 * kb * (c1 - c0));
    hipLaunchKernelGGL(k_laswp<T>, dim3((unsigned)cdiv(c1 - c0, LCW)), dim3(256), 0, lu->cur, F, ld, list, count, c0, c1);
    lu->prof.end(lu->cur, pi);
}

// Factors F (n x n, ld) in place; pivots into lu->ipiv, row map into lu->perm, diagonal-block
// inverses into DL / DU.  gemm_upd does the trailing updates (mode 0: C -= A B),
// gemm_trsm the products of the blocked TRSM (mode 1: C = A B in place, mode 0), gemm_in a panel's update
// inside its block (C -= A B, K = PW); all launch on lu->cur.
//
// Lookahead: the trailing update of outer block b first updates the columns of block b + 1 on
// lu->stream, then block b + 1 is factored on lu->stream2 while lu->stream updates the remaining
// columns.  The row interchanges of a block are applied right of it at once and, when a column
// segment fits in LDS, left of it (the L columns) in one pass at the end.
template <typename T, typename GU, typename GT, typename GI>
int getrf_blocked(lsx_lu* lu, T* F, int64_t ld, T* DL, T* DU, GU gemm_upd, GT gemm_trsm, GI gemm_in) {
    lsx_ctx* ctx = lu->ctx;
    const int64_t n = lu->n;
    const hipStream_t s0 = lu->stream_upd ? lu->stream_upd : lu->stream, s1 = lu->stream2;
    CoopHold hold;  // (the serving lanes, without lookahead, hold theirs themselves)
    if (lu->lookahead && cdiv(n, PROWS) > COOP_MARGIN) hold.take(ctx->device, ctx->num_cus, (int)cdiv(n, PROWS));
    const bool defer = lu->pinv != nullptr && (n - NBO) * (int64_t)sizeof(T) <= LGMAX_BYTES;
    if (s0 != lu->stream) {  // the input (copied on lu->stream) before anything on s0
        LSX_HIP(ctx, hipEventRecord(lu->ev_start, lu->stream));
        LSX_HIP(ctx, hipStreamWaitEvent(s0, lu->ev_start, 0));
    }
    lu->cur = s0;
    if (lu->seq > 0xF0000000u) {
        LSX_HIP(ctx, hipMemsetAsync(lu->slots, 0, sizeof(uint64_t) * 2 * (PMAX + 1) * RECS, s0));
        lu->seq = 1;
    }
    LSX_HIP(ctx, hipMemsetAsync(lu->dinfo, 0, 2 * sizeof(int64_t), s0));
    hipLaunchKernelGGL(k_iota, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, s0, lu->perm, n);
    int64_t* il = lu->plist;
    int* ic = lu->pcount;

    // The widths of the outer blocks, from the rows m that are left:
    //   m <= MTAIL: all the columns left are one block, every panel updating all of them (K = PW), on
    //     every CU.  The trailing matrix is then small enough for its update to take 5 to 20 us a panel,
    //     and a block of NBO would spend 110 us between its last panel and the next block's first (lists,
    //     interchanges and TRSM of the next columns, inverses).  Factor + one solve without and with it:
    //     n = 500 1.12 -> 0.82 ms, 1024 2.39 -> 1.78, 3001 10.3 -> 9.2, 16384 99.8 -> 98.5; a limit of 1024
    //     gives 9.7 at 3001, one of 4096 22.3 against 21.8 at 6000;
    //   m > MWIDE: 2 NBO columns, so that the trailing matrix is read and written half as often, where
    //     its update and not the panels' chain is the longer of the two: n = 16384 110.0 -> 100.6 ms, 12000
    //     58.4 -> 55.5, 9000 no change; in FP64 4 NBO above MWIDE4: 13000 64.8 -> 64.6, 14000 73.6 -> 72.7,
    //     15000 83.6 -> 82.1, 16384 100.6 -> 98.3 (10300 to 11000 lose 1.3 %; limits of 11000, 12000 and 13500
    //     take 0.3 to 2 % back from 13000 to 16384; FP32's shorter updates lose to the longer inner ones:
    //     mixed 14000 58.1 -> 59.2);
    //   else NBO.
    auto width = [&](int64_t jo) -> int {
        const int64_t m = n - jo;
        if (m <= MTAIL) return (int)m;
        return m <= MWIDE ? NBO : sizeof(T) == 8 && m > MWIDE4 ? 4 * NBO : 2 * NBO;
    };
    auto plist = [&](int par, int h) { return lu->plist + (1 + 4 * par + h) * 4 * NBO; };
    auto pcount = [&](int par, int h) { return lu->pcount + 1 + 4 * par + h; };
    auto build_list = [&](int64_t k0, int kb, int par, int h) {
        hipLaunchKernelGGL(k_perm_build, dim3(1), dim3(256), 0, lu->cur, lu->ipiv, k0, kb, plist(par, h), pcount(par, h));
    };
    // factorization of outer block [jo, jo + jbo) (its columns already updated): inner panels,
    // their interchanges (also of the row map) and updates inside the block, the block's interchange
    // lists (parity par; of a last block only for undeferred interchanges), diagonal-block inverses
    auto panel_block = [&](int64_t jo, int jbo, int par) -> int {
        for (int64_t ji = jo; ji < jo + jbo; ji += PW) {
            const int W = (int)std::min<int64_t>(PW, jo + jbo - ji);
            launch_panel_t<T>(lu, F, ld, ji, W, il, ic);
            const int64_t nleft = ji - jo, nright = jo + jbo - ji - W;
            const int pi = lu->prof.begin(lu->cur, PK_LASWP, (double)W * W * nright,
                                          sizeof(T) * 4.0 * W * (nleft + nright));
            hipLaunchKernelGGL(k_inner_swap<T>, dim3((unsigned)std::max<int64_t>(1, cdiv(nleft + nright, ICW))), dim3(256),
                               0, lu->cur, F, ld, n, ji, W, il, ic, jo, (int)nleft, ji + W, jo + jbo, lu->perm);
            lu->prof.end(lu->cur, pi);
            if (nright > 0)
                gemm_in(F + ji * ld + ji + W, F + (ji + W) * ld + ji, F + (ji + W) * ld + ji + W, ld, n - ji - W, nright);
        }
        // the interchange lists first: the update stream applies them to the columns right of the
        // block while the diagonal-block inverses are formed
        if (jo + jbo < n)
            for (int k = 0; k < jbo; k += NBO) build_list(jo + k, std::min(NBO, jbo - k), par, k / NBO);
        LSX_HIP(ctx, hipEventRecord(lu->ev_perm, lu->cur));
        const int64_t b0 = jo / DB, nbk = cdiv(jbo, DB);
        const int pi = lu->prof.begin(lu->cur, PK_OTHER, 0.0, 0.0);
        hipLaunchKernelGGL(k_diag_inv<T>, dim3((unsigned)nbk, 2), dim3(256), 0, lu->cur, F, ld, n, b0, DL, DU);
        lu->prof.end(lu->cur, pi);
        return LSX_OK;
    };
    // the inverse of the row map after block [jo, jo + jbo), for the deferred L-column gather; launched
    // after the block's ev_panel so that the update stream does not wait for it
    auto inv_perm = [&](int64_t jo, int jbo) {
        if (defer && jo + jbo < n)
            hipLaunchKernelGGL(k_inv_perm, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, lu->cur, lu->perm,
                               lu->pinv + (jo / NBO) * n, jbo / NBO, n);
    };
    auto interchange = [&](int64_t jo, int jbo, int par, int64_t c0, int64_t c1) {
        for (int k = 0; k < jbo; k += NBO)
            launch_laswp_t<T>(lu, F, ld, std::min(NBO, jbo - k), plist(par, k / NBO), pcount(par, k / NBO), c0, c1);
    };
    // interchanges, U12 = L11^{-1} A12 and A22 -= L21 U12 of block [jo, jo + jbo) on columns
    // [c0, c1); wait_inv: the block's diagonal-block inverses may still be in the making on the
    // panel stream (ev_panel), so the products wait for them after the interchanges
    auto update = [&](int64_t jo, int jbo, int par, int64_t c0, int64_t c1, bool wait_inv) -> int {
        if (c1 <= c0) return LSX_OK;
        const int64_t r1 = jo + jbo, nc = c1 - c0;
        interchange(jo, jbo, par, c0, c1);
        if (wait_inv && lu->cur != s1) LSX_HIP(ctx, hipStreamWaitEvent(lu->cur, lu->ev_panel, 0));
        // by 64-blocks of L11: X_i = L_ii^{-1} A12_i, then the rows below it in the block -= L_ki X_i
        for (int64_t k = 0; k < jbo; k += DB) {
            T* Ai = F + c0 * ld + jo + k;
            const int64_t h = std::min<int64_t>(DB, jbo - k), below = jbo - k - h;
            gemm_trsm(DL + (jo + k) / DB * DB * DB, DB, Ai, ld, Ai, ld, h, nc, h, 1);
            if (below > 0) gemm_trsm(F + (jo + k) * ld + jo + k + DB, ld, Ai, ld, Ai + DB, ld, below, nc, DB, 0);
        }
        gemm_upd(F + jo * ld + r1, ld, F + c0 * ld + jo, ld, F + c0 * ld + r1, ld, n - r1, nc, jbo, 0);
        return LSX_OK;
    };

    int jbo = width(0);
    int rc_ = panel_block(0, jbo, 0);
    if (rc_) return rc_;
    LSX_HIP(ctx, hipEventRecord(lu->ev_panel, s0));
    inv_perm(0, jbo);
    int par = 0, jbn = 0;
    int64_t deferred = 0;  // columns whose interchanges of later blocks are left to the end
    for (int64_t jo = 0; jo < n; jo += jbo, jbo = jbn, par ^= 1) {
        const int64_t c1 = jo + jbo;
        lu->cur = s0;
        if (!defer && jo > 0) {
            if (c1 < n) interchange(jo, jbo, par, 0, jo);
            else
                for (int64_t k = jo; k < n; k += NBO) {  // the last block made no lists
                    const int kb = (int)std::min<int64_t>(NBO, n - k);
                    build_list(k, kb, par, 0);
                    launch_laswp_t<T>(lu, F, ld, kb, plist(par, 0), pcount(par, 0), 0, jo);
                }
        }
        if (c1 >= n) break;
        deferred = c1;
        jbn = width(c1);
        const bool last = c1 + jbn >= n;  // nothing to overlap the last block with: it takes every CU
        if ((rc_ = update(jo, jbo, par, c1, c1 + jbn, true))) return rc_;
        if (last && s1 != s0) {  // its interchanges move the row map, which the last inv_perm on s1 reads
            LSX_HIP(ctx, hipEventRecord(lu->ev_next, s1));
            LSX_HIP(ctx, hipStreamWaitEvent(s0, lu->ev_next, 0));
        } else if (!last) {
            LSX_HIP(ctx, hipEventRecord(lu->ev_next, s0));
            LSX_HIP(ctx, hipStreamWaitEvent(s1, lu->ev_next, 0));
            lu->cur = s1;
        }
        if ((rc_ = panel_block(c1, jbn, par ^ 1))) return rc_;
        LSX_HIP(ctx, hipEventRecord(lu->ev_panel, lu->cur));
        inv_perm(c1, jbn);
        lu->cur = s0;
        if ((rc_ = update(jo, jbo, par, c1 + jbn, n, false))) return rc_;
        // the next block's interchange list (ev_perm) is all the next iteration's first step
        // needs; its products wait for the inverses (ev_panel) themselves
        LSX_HIP(ctx, hipStreamWaitEvent(s0, lu->ev_perm, 0));
    }
    lu->cur = s0;
    LSX_HIP(ctx, hipStreamWaitEvent(s0, lu->ev_panel, 0));  // the last block's inverses and row map
    if (defer && s1 != s0) {  // and every block's inverse row map (launched on s1 after its ev_panel)
        LSX_HIP(ctx, hipEventRecord(lu->ev_next, s1));
        LSX_HIP(ctx, hipStreamWaitEvent(s0, lu->ev_next, 0));
    }
    if (defer && deferred > 0) {
        const size_t lds = sizeof(T) * (size_t)(n - NBO);
        const int pi = lu->prof.begin(s0, PK_LASWP, 0.0, 2.0 * sizeof(T) * (double)n * n / 2);
        hipLaunchKernelGGL(k_left_gather<T>, dim3((unsigned)deferred), dim3(256), lds, s0, F, ld, n,
                           (const int*)lu->perm, (const int*)lu->pinv);
        lu->prof.end(s0, pi);
    }
    LSX_HIP(ctx, hipGetLastError());
    LSX_HIP(ctx, hipMemcpyAsync(lu->hinfo, lu->dinfo, 2 * sizeof(int64_t), hipMemcpyDeviceToHost, s0));
    LSX_HIP(ctx, hipStreamSynchronize(s0));
    lu->cur = lu->stream;
    lu->prof.collect();
    if (lu->hinfo[1] != 0)
        return fail(ctx, LSX_ETIMEOUT, "getrf: a panel exchange wait exceeded its bound (flags %lld)",
                    (long long)lu->hinfo[1]);
    return (int)std::min<int64_t>(lu->hinfo[0], INT32_MAX);
}

// X = A \ B (TR: X = A^{-T} B) with the resident factors (device buffers; FP64 right-hand sides,
// arithmetic in FP64 whatever the factor type).  The first solve writes lu->wy; X may alias B.  A
// wait that gives up sets lu->dinfo[1], which the public entry point clears once (lu_clear_err) and
// reads after its last launch, so a timeout in any of its solves is reported.
template <typename T, bool TR = false>
int getrs_blocked(lsx_lu* lu, const T* F, int64_t ld, const T* DL, const T* DU, int64_t nrhs, const double* dB,
                  int64_t ldb, double* dX, int64_t ldx) {
    lsx_ctx* ctx = lu->ctx;
    const int64_t n = lu->n;
    const int nblk = (int)cdiv(n, DB);
    if (lu->tseq > 0xF0000000u) {
        LSX_HIP(ctx, hipMemsetAsync(lu->tmsg, 0, sizeof(uint64_t) * nblk * TMW, lu->stream));
        lu->tseq = 1;
    }
    const int64_t timeout = wait_ticks(ctx, 5.0);
    const T *d1 = TR ? DU : DL, *d2 = TR ? DL : DU;  // the triangle solved first (blocks forward), then the other
    for (int64_t c0 = 0; c0 < nrhs; c0 += TRHS) {
        const int nr = (int)std::min<int64_t>(TRHS, nrhs - c0);
        const uint32_t s1 = lu->tseq++, s2 = lu->tseq++;
        const int pi = lu->prof.begin(lu->stream, PK_TRSV, 2.0 * n * n * nr, sizeof(T) * (double)n * n);
        const double *b = dB + c0 * ldb, *y = lu->wy;
        double* x = dX + c0 * ldx;
        auto grid = [&](auto kern, auto... args) {
            hipLaunchKernelGGL(kern, dim3(nblk), dim3(256), 0, lu->stream, F, ld, n, (const int*)lu->perm, args...);
        };
        if (nr == 1) {
            grid(k_trsv<T, true, TR>, d1, b, lu->wy, lu->tmsg, s1, timeout, lu->dinfo + 1);
            grid(k_trsv<T, false, TR>, d2, y, x, lu->tmsg, s2, timeout, lu->dinfo + 1);
        } else {
            grid(k_trsv_mrhs<T, true, TR>, d1, b, ldb, lu->wy, n, nr, lu->tmsg, s1, timeout, lu->dinfo + 1);
            grid(k_trsv_mrhs<T, false, TR>, d2, y, n, x, ldx, nr, lu->tmsg, s2, timeout, lu->dinfo + 1);
        }
        lu->prof.end(lu->stream, pi);
    }
    LSX_HIP(ctx, hipGetLastError());
    return LSX_OK;
}

}  // namespace lsx
