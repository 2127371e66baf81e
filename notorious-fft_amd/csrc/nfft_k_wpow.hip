// nfft_k_wpow.hip -- instantiations and launchers of the weighted spectral
// power kernels (nfft_kernels_wpow.h) for both precisions.
#include "nfft_launch_impl.h"
#include "nfft_kernels_wpow.h"

namespace nfft {

namespace {

template <typename T, int L> constexpr bool wpow_fits()
{
    constexpr int lpb = col_lpb<T, L>();
    return col_fits_v<T, L, lpb>() && wpow_threads<L, lpb>() % 64 == 0;
}

template <typename T, int L, int LPB> void wpow_h_go(unsigned gx, const WpowArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL((k_col_wpow_h<T, L, LPB>), dim3(gx, (unsigned)a.ntrans), dim3(Sched<L>::NT / 2 * LPB), 0, s, a);
}

// The order of other column passes; but tiles that share no 128-byte line keep
// the workgroups' own order, the row passes' too, in arrays below the 256 MiB of
// the memory-side cache: what fits one workgroup of either is then on one XCD
// throughout, and no XCD starts far from the part written last (us, workgroups'
// order / eighths: FP32 64^2 x 256 23.1 / 30.5, 256 x 64 x 128 36.4 / 44.3, 512 x 32 x
// 128 40.0 / 46.6, 1024^2 x 2 42.3 / 46.3; FP64 64^2 x 128 24.3 / 31.8, 512 x 32 x 64 37.0 /
// 38.8, 256^2 x 200 203 / 221; 400 MiB of it 500 / 470).  Not FP64 columns of up to 64
// points in several tiles, whose rows are runs of 1 KiB and more (32 x 512 x 64
// 36.4 / 32.1, 64 x 256 x 64 33.7 / 30.3).
template <typename T> int wpow_order(int L, int w, const WpowArgs &a)
{
    constexpr long long cb = (long long)sizeof(Cx<T>);
    const bool lines = w * cb % 128 == 0 && a.ncols * cb % 128 == 0;
    const bool wide = cb == 16 && L <= 64 && a.ncols > w;
    if (lines && !wide && a.ntrans * a.dist * cb < 8 * kL2Bytes) return ORDER_PLAIN;
    return col_order(sizeof(T) == 4 ? F32 : F64, a.ntrans * a.dist);
}

// launch == false: only the form that the whole batch takes and its workgroups
// per transform
template <typename T> hipError_t col_wpow_impl(int L, WpowArgs &a, hipStream_t s, long long *per, bool launch)
{
    switch (L) {
#define NFFT_CASE(LL)                                                                                         \
    case LL:                                                                                                  \
        if constexpr (wpow_fits<T, LL>()) {                                                                   \
            constexpr int lpb = col_lpb<T, LL>();                                                             \
            if (!launch) {                                                                                    \
                ColArgs c{};                                                                                  \
                c.ncols = a.ncols;                                                                            \
                c.S = a.ncols;                                                                                \
                c.ntrans = a.ntrans;                                                                          \
                a.form = LL >= 512 ? col_form<T, LL>(COL_PLAIN, c) : 0;                                       \
            }                                                                                                 \
            const int w = a.form == 2 ? 2 * lpb : lpb;                                                        \
            a.order = wpow_order<T>(LL, w, a);                                                                \
            const unsigned gx = (unsigned)((a.ncols + w - 1) / w);                                            \
            *per = gx;                                                                                        \
            if (!launch) return hipSuccess;                                                                   \
            if constexpr (LL >= 512) {                                                                        \
                if (a.form == 1) wpow_h_go<T, LL, lpb>(gx, a, s);                                             \
                if (a.form == 2) wpow_h_go<T, LL, 2 * lpb>(gx, a, s);                                         \
            }                                                                                                 \
            if (a.form == 0)                                                                                  \
                hipLaunchKernelGGL((k_col_wpow<T, LL, lpb>), dim3(gx, (unsigned)a.ntrans),                    \
                                   dim3((wpow_threads<LL, lpb>())), 0, s, a);                                 \
            return hipGetLastError();                                                                         \
        }                                                                                                     \
        break;
        NFFT_POW2_LIST(NFFT_CASE)
#undef NFFT_CASE
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool col_wpow_supported(int prec, int L)
{
    int form = 0;
    return col_wpow_tiles(prec, L, 1, 1, &form) > 0;
}

long long col_wpow_tiles(int prec, int L, int ncols, long long batch, int *form)
{
    long long per = 0;
    WpowArgs a{};
    a.ncols = ncols;
    a.ntrans = batch;
    if ((prec == F32 ? col_wpow_impl<float>(L, a, nullptr, &per, false)
                     : col_wpow_impl<double>(L, a, nullptr, &per, false)) != hipSuccess)
        return 0;
    *form = a.form;
    return per;
}

hipError_t launch_col_wpow(int prec, int L, const WpowArgs &a0, hipStream_t s)
{
    WpowArgs a = a0;
    if (a.ntrans < 1 || a.ntrans > 65535 || !a.buf) return hipErrorInvalidValue;
    long long per = 0;
    const int slot = prof_on() ? prof_begin(s) : -1;
    const hipError_t e = prec == F32 ? col_wpow_impl<float>(L, a, s, &per, true) : col_wpow_impl<double>(L, a, s, &per, true);
    if (slot >= 0)
        prof_end(slot, s, "k_col_wpow", prec, L,
                 (double)a.ntrans * a.dist * (prec == F32 ? 16.0 : 32.0) + (double)a.dist * (prec == F32 ? 4 : 8));
    return e;
}

long long wpow_mask_chunks(long long P) { return std::max(1LL, std::min(1024LL, (P + 2047) / 2048)); }

hipError_t launch_wpow_mask(int prec, void *buf, const void *w, double *partial, long long P, long long ntrans,
                            hipStream_t s)
{
    if (ntrans < 1 || ntrans > 65535) return hipErrorInvalidValue;
    const dim3 g((unsigned)wpow_mask_chunks(P), (unsigned)ntrans);
    if (prec == F32) hipLaunchKernelGGL(k_wpow_mask<float>, g, dim3(256), 0, s, buf, w, partial, P);
    else hipLaunchKernelGGL(k_wpow_mask<double>, g, dim3(256), 0, s, buf, w, partial, P);
    return hipGetLastError();
}

hipError_t launch_wpow_reduce(const double *partial, double *loss, long long per, long long ntrans, hipStream_t s)
{
    if (ntrans < 1) return hipSuccess;
    hipLaunchKernelGGL(k_wpow_reduce, dim3((unsigned)ntrans), dim3(64), 0, s, partial, loss, per);
    return hipGetLastError();
}

}  // namespace nfft
