// nfft_k_c2r.hip -- launcher of the packing column pass (both precisions).
#include "nfft_launch_impl.h"

namespace nfft {

namespace {
template <typename T> hipError_t col_pack_impl(int L, bool twid, const ColPackArgs &a, hipStream_t s, bool query)
{
    switch (L) {
#define NFFT_CASE(LL)                                                                                           \
    case LL:                                                                                                    \
        if constexpr (col_fits<T, LL>()) {                                                                      \
            constexpr int lpb = col_lpb<T, LL>();                                                               \
            /* whole tiles, 32-bit offsets within a transform */                                                \
            if (a.c.ncols % lpb || (long long)LL * a.c.S * (long long)sizeof(Cx<T>) >= (1LL << 32))             \
                return hipErrorInvalidValue;                                                                    \
            if (query) return hipSuccess;                                                                       \
            unsigned gy, gz;                                                                                    \
            grid_trans(a.c.ntrans, gy, gz);                                                                     \
            const dim3 g((unsigned)(a.c.ncols / lpb), gy, gz), b(Sched<LL>::NT *lpb);                           \
            if (twid) hipLaunchKernelGGL((k_col_pack<T, LL, lpb, true>), g, b, 0, s, a);                        \
            else hipLaunchKernelGGL((k_col_pack<T, LL, lpb, false>), g, b, 0, s, a);                            \
            return hipGetLastError();                                                                           \
        }                                                                                                       \
        break;
        NFFT_CASE(16) NFFT_CASE(32) NFFT_CASE(64) NFFT_CASE(128) NFFT_CASE(256) NFFT_CASE(512) NFFT_CASE(1024)
        NFFT_CASE(2048) NFFT_CASE(4096)
#undef NFFT_CASE
    }
    return hipErrorInvalidValue;
}
}  // namespace

bool col_pack_supported(int prec, int L, int S)
{
    ColPackArgs a{};
    a.c.ncols = S;
    a.c.S = S;
    return (prec == F32 ? col_pack_impl<float>(L, false, a, nullptr, true)
                        : col_pack_impl<double>(L, false, a, nullptr, true)) == hipSuccess;
}

hipError_t launch_col_pack(int prec, int L, bool twid, const ColPackArgs &a, hipStream_t s)
{
    const int slot = prof_on() ? prof_begin(s) : -1;
    const hipError_t e = prec == F32 ? col_pack_impl<float>(L, twid, a, s, false) : col_pack_impl<double>(L, twid, a, s, false);
    if (slot >= 0)
        prof_end(slot, s, "k_col_pack", prec, L, 2.0 * (double)a.c.ntrans * L * a.c.S * (double)cx_bytes(prec));
    return e;
}

}  // namespace nfft
