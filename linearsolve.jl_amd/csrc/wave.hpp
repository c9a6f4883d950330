// wave.hpp — wave-wide (64-lane) reductions on DPP and permlane swaps, and the pivot key of
// partial pivoting, shared by the panel kernels of the blocked LU and the batched LU.
#pragma once
#include <climits>
#include <cstdint>
#include <type_traits>

#include <hip/hip_runtime.h>

namespace lsx {

// f(integral_constant<int, I>) for I = 0 .. N-1, each call with its index a compile-time constant
// (a loop whose steps index register arrays, too long for the unroller).
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// ---- wave-wide reductions (64 lanes): DPP within rows of 16 lanes, then two cross-row steps
template <int CTRL> __device__ __forceinline__ uint32_t dpp32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}
// Value of the lane 16 (32) apart across rows of 16 (halves of 32), by v_permlane16_swap /
// v_permlane32_swap of x with itself: the swap gives each lane its own value in one result and the
// partner's in the other.
__device__ __forceinline__ uint32_t xrow16(uint32_t x) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return ((threadIdx.x >> 4) & 1) ? r[0] : r[1];
}
__device__ __forceinline__ uint32_t xrow32(uint32_t x) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return ((threadIdx.x >> 5) & 1) ? r[0] : r[1];
}
__device__ __forceinline__ int wave_min_i32(int x) {
    int y;
    y = (int)dpp32<0xB1>((uint32_t)x);  x = y < x ? y : x;
    y = (int)dpp32<0x4E>((uint32_t)x);  x = y < x ? y : x;
    y = (int)dpp32<0x141>((uint32_t)x); x = y < x ? y : x;
    y = (int)dpp32<0x140>((uint32_t)x); x = y < x ? y : x;
    y = (int)xrow16((uint32_t)x);       x = y < x ? y : x;
    y = (int)xrow32((uint32_t)x);       x = y < x ? y : x;
    return x;
}
template <int CTRL> __device__ __forceinline__ uint32_t dpp_max_u32(uint32_t x) {
    const uint32_t y = dpp32<CTRL>(x);
    return y > x ? y : x;
}
// Largest 32-bit value of the wave, uniform.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    x = dpp_max_u32<0xB1>(x);
    x = dpp_max_u32<0x4E>(x);
    x = dpp_max_u32<0x141>(x);
    x = dpp_max_u32<0x140>(x);
    uint32_t y = xrow16(x);
    x = y > x ? y : x;
    y = xrow32(x);
    x = y > x ? y : x;
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
}
// Lane holding the best (u, lr) pair of the wave: largest u, then smallest logical row lr; u = 0 marks "no
// candidate"; the result is uniform.  In 32-bit steps: the upper halves decide almost always, the lower
// halves and then the rows are compared only among lanes that tie.
__device__ __forceinline__ int wave_argmax32(uint64_t u, int lr) {
    const uint32_t hi = (uint32_t)(u >> 32);
    uint64_t tie = __ballot(hi == wave_max_u32(hi));
    if (__popcll(tie) > 1) {
        const uint32_t lo = (tie >> (threadIdx.x & 63)) & 1 ? (uint32_t)u : 0u;
        const uint32_t ml = wave_max_u32(lo);
        tie &= __ballot(lo == ml);
        if (__popcll(tie) > 1) {
            const bool in = (tie >> (threadIdx.x & 63)) & 1;
            const int mn = wave_min_i32(in ? lr : INT_MAX);
            tie &= __ballot(in && lr == mn);
        }
    }
    return __ffsll((unsigned long long)tie) - 1;
}
// The same over N candidates (N = 2, 4, 8 or 16), candidate l & (N - 1) in lane l.
template <int N>
__device__ __forceinline__ int wave_argmax_rep(uint64_t u, int lr) {
    static_assert(N == 2 || N == 4 || N == 8 || N == 16, "up to a row of lanes");
    constexpr uint64_t first = (1ull << N) - 1;
    auto mx = [](uint32_t x) {
        x = dpp_max_u32<0xB1>(x);
        if constexpr (N > 2) x = dpp_max_u32<0x4E>(x);
        if constexpr (N > 4) x = dpp_max_u32<0x141>(x);
        if constexpr (N > 8) x = dpp_max_u32<0x140>(x);
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
    };
    const uint32_t hi = (uint32_t)(u >> 32);
    uint64_t tie = __ballot(hi == mx(hi));
    if (__popcll(tie & first) > 1) {
        const uint32_t lo = (tie >> (threadIdx.x & 63)) & 1 ? (uint32_t)u : 0u;
        tie &= __ballot(lo == mx(lo));
        if (__popcll(tie & first) > 1) {
            const bool in = (tie >> (threadIdx.x & 63)) & 1;
            tie &= __ballot(in && ~(uint32_t)lr == mx(in ? ~(uint32_t)lr : 0u));  // the smallest row
        }
    }
    return __ffsll((unsigned long long)(tie & first)) - 1;
}
// Value of lane S of each row of 16 lanes, in all lanes of the row (all lanes active).
template <int S> __device__ __forceinline__ double row_bcast(double x) {
    return __longlong_as_double(__builtin_amdgcn_mov_dpp((long long)__double_as_longlong(x), 0x150 + S, 0xF, 0xF, true));
}
template <int S> __device__ __forceinline__ float row_bcast(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(x), 0x150 + S, 0xF, 0xF, true));
}
// Pivot key: |a| as its (monotone) bit pattern + 1, NaN counted as 0; 0 = not a candidate.
template <typename T> __device__ __forceinline__ uint64_t pivot_key(T x) {
    double t = fabs((double)x);
    if (!(t == t)) t = 0.0;
    return (uint64_t)__double_as_longlong(t) + 1u;
}

}  // namespace lsx
