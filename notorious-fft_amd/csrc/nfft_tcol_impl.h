// nfft_tcol_impl.h -- size dispatch of the strided DCT / DST kernels.
#pragma once
#include "nfft_internal.h"

namespace nfft {

template <typename T, int N, int lpb> constexpr bool tcol_fits()
{
    return N >= 2 && N <= 4096 && (size_t)N * lpb * sizeof(Cx<T>) <= kLdsLimit && Sched<N>::NT * lpb <= 1024;
}

template <typename T, int N, int LPB>
hipError_t tcol_go(int op, const TrigColArgs &a, long long grid, hipStream_t s)
{
    const dim3 g((unsigned)grid), b2(Sched<N>::NT *LPB), b4(Sched<N / 2>::NT *LPB);
    switch (op) {
    case T_DCT2: hipLaunchKernelGGL((k_t23_col<T, N, LPB, T_DCT2>), g, b2, 0, s, a); break;
    case T_DST2: hipLaunchKernelGGL((k_t23_col<T, N, LPB, T_DST2>), g, b2, 0, s, a); break;
    case T_DCT3: hipLaunchKernelGGL((k_t23_col<T, N, LPB, T_DCT3>), g, b2, 0, s, a); break;
    case T_DST3: hipLaunchKernelGGL((k_t23_col<T, N, LPB, T_DST3>), g, b2, 0, s, a); break;
    case T_DCT4: hipLaunchKernelGGL((k_t4_col<T, N, LPB, T_DCT4>), g, b4, 0, s, a); break;
    default: hipLaunchKernelGGL((k_t4_col<T, N, LPB, T_DST4>), g, b4, 0, s, a); break;
    }
    return hipGetLastError();
}

// query: only whether a kernel takes these arguments
template <typename T> hipError_t tcol_impl(int N, int op, const TrigColArgs &a0, hipStream_t s, bool query)
{
    TrigColArgs a = a0;
    a.order = col_order(sizeof(T) == 4 ? F32 : F64, a.total * N);
    switch (N) {
#define NFFT_CASE(LL)                                                                                           \
    case LL:                                                                                                    \
        if constexpr (tcol_fits<T, LL, col_lpb<T, LL>()>()) {                                                   \
            constexpr int lpb = col_lpb<T, LL>();                                                               \
            /* a tile's columns are addressed from its first array by 32-bit offsets */                         \
            const long long span = ((lpb - 1) / a.ncols + 2) * a.dist * (long long)sizeof(Cx<T>);               \
            const long long grid = (a.total + lpb - 1) / lpb;                                                   \
            if (span >= (1LL << 32) || grid > 0x7fffffffLL) return hipErrorInvalidValue;                        \
            if (query) return hipSuccess;                                                                       \
            /* few tiles: narrower ones (us, FP32 1024^2 DCT-2 and back, 32 tiles 51 -> 43, x 3 57 -> 53,     */ \
            /* 1024 x 32 x 8 41 -> 33; FP64 1024^2 55 -> 53, x 3, 192 tiles, 72.8 -> 73.4)                    */ \
            if constexpr (LL >= 512 && lpb > 4)                                                                 \
                if (grid <= 128) return tcol_go<T, LL, 4>(op, a, (a.total + 3) / 4, s);                         \
            return tcol_go<T, LL, lpb>(op, a, grid, s);                                                         \
        }                                                                                                       \
        break;
        NFFT_CASE(2) NFFT_CASE(4) NFFT_CASE(8) NFFT_CASE(16) NFFT_CASE(32) NFFT_CASE(64) NFFT_CASE(128)
        NFFT_CASE(256) NFFT_CASE(512) NFFT_CASE(1024) NFFT_CASE(2048) NFFT_CASE(4096)
#undef NFFT_CASE
    }
    return hipErrorInvalidValue;
}

}  // namespace nfft
