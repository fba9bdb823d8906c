// Requantisation of 64-bit accumulators (acc64 of op_impls/utils/precision.py:122-123).
#pragma once

#include <type_traits>

#include "common.hpp"

namespace a4g {

// Rounding and saturation of the 64-bit sums of int16 x int16 products as one add before the shift: v + c0, plus a tie term of -1, 0 or 1
// that the mode takes from the sign of v or from bit s of v, then the shift and the saturation. c0 and en depend
// on the column's shift and on the mode only; en is 0 where the shift is 0 (nothing to round) and -1 elsewhere.
// |v| stays below 2^48 (K <= 32768) and c0 below 2^62, so the sum cannot overflow.
struct Round64 {
    long long c0;
    int s, en;
};

__device__ __forceinline__ Round64 make_round64(int shift, int mode) {
    Round64 r;
    r.s = min(max(shift, 0), 62);
    r.en = r.s > 0 ? -1 : 0;
    const long long h = (1ll << r.s) >> 1;
    switch (mode) {
    case A4G_RND_FLOOR: r.c0 = 0; break;
    case A4G_RND_CEIL: r.c0 = (1ll << r.s) - 1; break;
    case A4G_RND_POSITIVE_INF:
    case A4G_RND_SYMMETRIC_INF:
    case A4G_RND_CONV_ODD: r.c0 = h; break;
    default: r.c0 = h + r.en; break;  // ties go down unless the tie term says otherwise
    }
    return r;
}

template <int MODE>
__device__ __forceinline__ int requant64_m(long long v, long long c0, int s, int en, int lo, int hi) {
    long long t = v + c0;
    if constexpr (MODE == A4G_RND_SYMMETRIC_INF) t += static_cast<int>(v >> 63) & en;   // below zero: h - 1
    if constexpr (MODE == A4G_RND_SYMMETRIC_ZERO) t -= static_cast<int>(v >> 63) & en;  // below zero: h
    if constexpr (MODE == A4G_RND_CONV_EVEN) t += static_cast<int>(v >> s) & 1 & en;
    if constexpr (MODE == A4G_RND_CONV_ODD) t -= static_cast<int>(v >> s) & 1 & en;
    const long long q = t >> s;
    const int ql = static_cast<int>(q), qh = static_cast<int>(q >> 32);
    const int y = qh == (ql >> 31) ? ql : ((qh >> 31) ^ 0x7fffffff);  // beyond 32 bits: the bound on q's side
    return clamp_med3(y, lo, hi);
}

// Calls f with the rounding mode as a compile-time constant.
template <typename F>
__device__ __forceinline__ void with_round_mode(int mode, F&& f) {
    switch (mode) {
    case A4G_RND_FLOOR: f(std::integral_constant<int, A4G_RND_FLOOR>{}); break;
    case A4G_RND_CEIL: f(std::integral_constant<int, A4G_RND_CEIL>{}); break;
    case A4G_RND_POSITIVE_INF: f(std::integral_constant<int, A4G_RND_POSITIVE_INF>{}); break;
    case A4G_RND_NEGATIVE_INF: f(std::integral_constant<int, A4G_RND_NEGATIVE_INF>{}); break;
    case A4G_RND_SYMMETRIC_INF: f(std::integral_constant<int, A4G_RND_SYMMETRIC_INF>{}); break;
    case A4G_RND_SYMMETRIC_ZERO: f(std::integral_constant<int, A4G_RND_SYMMETRIC_ZERO>{}); break;
    case A4G_RND_CONV_EVEN: f(std::integral_constant<int, A4G_RND_CONV_EVEN>{}); break;
    default: f(std::integral_constant<int, A4G_RND_CONV_ODD>{}); break;
    }
}

}  // namespace a4g
