// nfft_tcol_impl.h -- size dispatch of the strided DCT / DST kernels.
#pragma once
#include "nfft_internal.h"

namespace nfft {

template <typename T, int N> constexpr bool tcol_fits()
{
    constexpr int lpb = col_lpb<T, N>();
    return N >= 2 && N <= 4096 && (size_t)N * lpb * sizeof(Cx<T>) <= kLdsLimit && Sched<N>::NT * lpb <= 1024;
}

// query: only whether a kernel takes these arguments
template <typename T> hipError_t tcol_impl(int N, int op, const TrigColArgs &a, hipStream_t s, bool query)
{
    switch (N) {
#define NFFT_CASE(LL)                                                                                           \
    case LL:                                                                                                    \
        if constexpr (tcol_fits<T, LL>()) {                                                                     \
            constexpr int lpb = col_lpb<T, LL>();                                                               \
            /* a tile's columns are addressed from its first array by 32-bit offsets */                         \
            const long long span = ((lpb - 1) / a.ncols + 2) * a.dist * (long long)sizeof(Cx<T>);               \
            const long long grid = (a.total + lpb - 1) / lpb;                                                   \
            if (span >= (1LL << 32) || grid > 0x7fffffffLL) return hipErrorInvalidValue;                        \
            if (query) return hipSuccess;                                                                       \
            const dim3 g((unsigned)grid), b2(Sched<LL>::NT *lpb), b4(Sched<LL / 2>::NT *lpb);                   \
            switch (op) {                                                                                       \
            case T_DCT2: hipLaunchKernelGGL((k_t23_col<T, LL, lpb, T_DCT2>), g, b2, 0, s, a); break;            \
            case T_DST2: hipLaunchKernelGGL((k_t23_col<T, LL, lpb, T_DST2>), g, b2, 0, s, a); break;            \
            case T_DCT3: hipLaunchKernelGGL((k_t23_col<T, LL, lpb, T_DCT3>), g, b2, 0, s, a); break;            \
            case T_DST3: hipLaunchKernelGGL((k_t23_col<T, LL, lpb, T_DST3>), g, b2, 0, s, a); break;            \
            case T_DCT4: hipLaunchKernelGGL((k_t4_col<T, LL, lpb, T_DCT4>), g, b4, 0, s, a); break;             \
            default: hipLaunchKernelGGL((k_t4_col<T, LL, lpb, T_DST4>), g, b4, 0, s, a); break;                 \
            }                                                                                                   \
            return hipGetLastError();                                                                           \
        }                                                                                                       \
        break;
        NFFT_CASE(2) NFFT_CASE(4) NFFT_CASE(8) NFFT_CASE(16) NFFT_CASE(32) NFFT_CASE(64) NFFT_CASE(128)
        NFFT_CASE(256) NFFT_CASE(512) NFFT_CASE(1024) NFFT_CASE(2048) NFFT_CASE(4096)
#undef NFFT_CASE
    }
    return hipErrorInvalidValue;
}

}  // namespace nfft
