// nfft_kernels_c2r.h -- first pass of a long invrealdft: pack, column FFT.
//
// invrealdft of N = 2 Lc reals (src/07_legacy.h:239-293) is the inverse FFT
// of the Lc packed points Z[k] = pack(X[k], X[Lc-k]); as a four-step Lc = L x
// S its first pass transforms columns of L points.  k_col_pack forms Z as it
// loads: point k = p S + c of column c pairs with point Lc - k, in column S - c
// of the spectrum, so a tile reads its own columns and the mirrored ones.
// Tiles are taken in mirrored pairs (neighbouring workgroups of one XCD), so
// the second read of a line is served by the L2 the first one filled.
//
// Bound: one read of the spectrum and one write of the intermediate in
// 128-byte segments.  The elementwise pack pass it replaces read and wrote
// the whole spectrum once more (N = 2^20 x 200 FP32: inverse 1095 -> 670 us,
// 2^17 x 1024 727 -> 435 us; FP64 2^18 x 256 650 -> 440 us).
#pragma once
#include "nfft_kernels_rt.h"
#include "nfft_kernels_smooth.h"  // RootTab

namespace nfft {

struct ColPackArgs {
    ColArgs c;        // in: spectrum (in_dist apart), out, tables, S = ncols
    const void *w;    // FP64 e^{-2 pi i k / N}, k < Lc / 16
    int half;         // adjoint of realdft: bins 0 < k < Lc times 1/2
};

// TWID: inter-pass twiddle here (else the row pass applies it)
template <typename T, int L, int LPB, bool TWID>
__global__ void __launch_bounds__((col_threads<L, LPB>()),
                                  (wpe_hint<T>(col_threads<L, LPB>(), (long)L *LPB * sizeof(Cx<T>))))
k_col_pack(ColPackArgs g)
{
    using S = Sched<L>;
    using C = Cx<T>;
    static_assert(S::R == 16, "16 points per thread");
    __shared__ C lds[L * LPB];
    const ColArgs &a = g.c;
    const int b = threadIdx.x % LPB, j = threadIdx.x / LPB;
    const long long lin = blockIdx.x + (long long)gridDim.x * (blockIdx.y + (long long)gridDim.y * blockIdx.z);
    const long long lg = xcd_logical(lin, (long long)gridDim.x * gridDim.y * gridDim.z);
    const int l = (int)(lg % gridDim.x);
    const int c0 = ((l & 1) ? (int)gridDim.x - 1 - (l >> 1) : l >> 1) * LPB, c = c0 + b;
    const long long t = lg / gridDim.x;
    if (t >= a.ntrans) return;  // uniform per workgroup
    const uint32_t qst = (uint32_t)(S::NT * a.S) * (uint32_t)sizeof(C);
    const C *src = (const C *)a.in + t * a.in_dist;
    const double2 *w = (const double2 *)g.w;
    // partner of point (j + NT q) S + c: counted from S - c0 - (LPB - 1)
    const auto r1 = buf_rsrc(src + c0), r2 = buf_rsrc(src + a.S - c0 - (LPB - 1));
    const uint32_t o1 = (uint32_t)(j * a.S + b) * (uint32_t)sizeof(C);
    const uint32_t o2 = (uint32_t)((S::NT - 1 - j) * a.S + (LPB - 1 - b)) * (uint32_t)sizeof(C);
    C reg[16], par[16];
#pragma unroll
    for (int q = 0; q < 16; q++) reg[q] = buf_ld<C>(r1, o1, q * qst);
#pragma unroll
    for (int q = 0; q < 16; q++) par[q] = buf_ld<C>(r2, o2, (15 - q) * qst);
    // w_k = w_{j S + c} e^{-2 pi i q / 32}, formed in FP64 (rounded once in
    // FP32 kernels: as exact as a table of all k)
    const double2 wk = w[(long long)j * a.S + c];
    const T hw = g.half ? (T)0.5 : (T)1;
    sfor<0, 16>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        C xk = cscale(reg[q], hw), xm = cscale(par[q], hw);
        if (q == 0 && j == 0 && c == 0) {  // bins 0 and Lc: whole, imaginary parts ignored
            xk = cmk<C>(reg[q].x, (T)0);
            xm = cmk<C>(par[q].x, (T)0);
        }
        reg[q] = pack_pair(xk, xm, to_cx<T>(twp<-1, 32, q>(wk)));
    });
    line_fft<T, L, 1>(reg, lds, LayCol<LPB>{b}, j, (const double2 *)a.tw);
    if constexpr (TWID) apply_tw2_series<1>(reg, a.tw2, (uint32_t)c * (uint32_t)j, (uint32_t)c * (uint32_t)S::NT);
    const auto rd = buf_rsrc((C *)a.out + t * a.out_dist + c0);
#pragma unroll
    for (int q = 0; q < 16; q++) buf_st(rd, o1, q * qst, reg[q]);
}

}  // namespace nfft
