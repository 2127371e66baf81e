// nfft_kernels_wpow.h -- weighted spectral power and its gradient:
//     L(x) = sum_k |W_k Y_k|^2,  Y = DFT(x),   grad = 2 DFT^H (W^2 . Y)
// (g = dL/dRe x + i dL/dIm x), per transform of a batch.
//
// k_col_wpow fuses the last pass of the forward transform, the weighting and
// the first pass of the adjoint: a tile of columns of axis 0 (length L,
// stride S) is transformed forward, each bin k multiplied by 2 W_k^2 while
// W_k^2 |Y_k|^2 is summed (in FP64), and transformed back (unnormalised
// inverse) before it is stored: one HBM round trip instead of three.  The
// other axes run as ordinary passes before and after it.
// k_wpow_mask is the same weighting as an elementwise pass, for plans whose
// axis 0 is not a single-pass column length.
// Loss partial sums go to one slot per workgroup; k_wpow_reduce adds each
// transform's slots in a fixed order (deterministic, FP64).
#pragma once
#include "nfft_internal.h"

namespace nfft {

template <int L, int LPB> __host__ __device__ constexpr int wpow_threads() { return Sched<L>::NT * LPB; }

// Sum of v over the block, returned to thread 0 (FP64; red holds one entry per wave).
template <int NTH> __device__ __forceinline__ double block_sum(double v, double *red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < NTH / 64; i++) t += red[i];
    return t;
}

template <typename T, int L, int LPB>
__global__ void __launch_bounds__((wpow_threads<L, LPB>())) k_col_wpow(WpowArgs a)
{
    using S = Sched<L>;
    using C = Cx<T>;
    constexpr int NTH = wpow_threads<L, LPB>();
    static_assert(NTH % 64 == 0, "whole waves");
    constexpr int NLDS = S::S > 1 ? L * LPB : 1;
    constexpr int TWN = S::TWN > 0 ? S::TWN : 1;
    __shared__ C lds[NLDS];
    __shared__ C ltw[TWN];
    __shared__ double red[NTH / 64];
    if constexpr (S::S > 1) stage_tw_to_lds<T, L>(ltw, (const double2 *)a.tw);
    const int b = threadIdx.x % LPB, j = threadIdx.x / LPB;
    // neighbouring tiles on one XCD where they share lines: 2048-point columns fit 8
    // FP32 columns, half a 128-byte line, whose other half the next tile reads and writes
    const long long tile = xcd_order(blockIdx.x + (long long)gridDim.x * blockIdx.y,
                                     (long long)gridDim.x * gridDim.y, a.order);  // (transform, column tile)
    const long long t = tile / gridDim.x;
    const int c0 = (int)(tile % gridDim.x) * LPB, c = c0 + b;
    const bool valid = c < a.ncols;
    // uniform: every column of the tile exists and tile offsets fit 32 bits
    const bool full = c0 + LPB <= a.ncols && off_fits<C>((long long)L * a.ncols);
    C *col = (C *)a.buf + t * a.dist + c;
    const T *w = (const T *)a.w + c;
    const auto rs = buf_rsrc((C *)a.buf + t * a.dist + c0);
    const uint32_t off = (uint32_t)(j * a.ncols + b) * (uint32_t)sizeof(C);
    const uint32_t qst = (uint32_t)(S::NT * a.ncols) * (uint32_t)sizeof(C);
    C reg[S::R];
    if (full) {
#pragma unroll
        for (int q = 0; q < S::R; q++) reg[q] = buf_ld<C>(rs, off, q * qst);
    } else {
#pragma unroll
        for (int q = 0; q < S::R; q++) reg[q] = valid ? col[(long long)(j + S::NT * q) * a.ncols] : czero<T>();
    }
    __syncthreads();  // stage table in LDS
    LayCol<LPB> lay{b};
    line_fft_tw<T, L, -1>(reg, lds, lay, j, StageTwLds<T>{ltw});
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < S::R; q++) {
        const T wk = valid ? w[(long long)(j + S::NT * q) * a.ncols] : (T)0;
        const T w2 = wk * wk;
        const C y = reg[q];
        part += (double)w2 * ((double)y.x * y.x + (double)y.y * y.y);
        reg[q] = cscale(y, (T)2 * w2);
    }
    line_fft_tw<T, L, 1>(reg, lds, lay, j, StageTwLds<T>{ltw});
    if (full) {
#pragma unroll
        for (int q = 0; q < S::R; q++) buf_st<C>(rs, off, q * qst, reg[q]);
    } else if (valid) {
#pragma unroll
        for (int q = 0; q < S::R; q++) col[(long long)(j + S::NT * q) * a.ncols] = reg[q];
    }
    const double tot = block_sum<NTH>(part, red);
    if (threadIdx.x == 0) a.partial[tile] = tot;
}

// The same with the exchanges through half a tile of LDS, two sets of 16 points
// per thread, where col_form (nfft_launch_impl.h) takes k_col_h: two workgroups
// a CU, or twice the columns.
template <typename T, int L, int LPB>
__global__ void __launch_bounds__((Sched<L>::NT / 2 * LPB), (col_h_wpe<T, L, LPB>())) k_col_wpow_h(WpowArgs a)
{
    using S = Sched<L>;
    using C = Cx<T>;
    constexpr int NH = S::NT / 2, NTH = NH * LPB;
    static_assert(NTH % 64 == 0, "whole waves");
    __shared__ C lds[L / 2 * LPB];
    __shared__ C ltw[S::TWN];
    __shared__ double red[NTH / 64];
    const int b = threadIdx.x % LPB;
    int j = threadIdx.x / LPB;
    const long long tile = xcd_order(blockIdx.x + (long long)gridDim.x * blockIdx.y,
                                     (long long)gridDim.x * gridDim.y, a.order);
    const long long t = tile / gridDim.x;
    const int c0 = (int)(tile % gridDim.x) * LPB, c = c0 + b;
    const bool valid = c < a.ncols;
    const bool full = c0 + LPB <= a.ncols && off_fits<C>((long long)L * a.ncols);
    C *col = (C *)a.buf + t * a.dist + c;
    const T *w = (const T *)a.w + (valid ? c : 0);  // columns past the last one weigh zero
    const auto rs = buf_rsrc((C *)a.buf + t * a.dist + c0);
    const auto off = [&] { return (uint32_t)(j * a.ncols + b) * (uint32_t)sizeof(C); };
    const uint32_t qst = (uint32_t)(S::NT * a.ncols) * (uint32_t)sizeof(C);
    const uint32_t lst = (uint32_t)(NH * a.ncols) * (uint32_t)sizeof(C);
    const auto row = [&](int l, int q) { return (long long)(j + l * NH + S::NT * q) * a.ncols; };
    C reg[2][16];
    if (full) {
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int q = 0; q < 16; q++) reg[l][q] = buf_ld<C>(rs, off(), l * lst + q * qst);
    } else {
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int q = 0; q < 16; q++) reg[l][q] = valid ? col[row(l, q)] : czero<T>();
    }
    stage_tw_to_lds<T, L>(ltw, (const double2 *)a.tw);  // visible after the first exchange's barriers
    line_fft_halves<T, L, -1>(reg, lds, LayCol<LPB>{b}, j, StageTwLds<T>{ltw});
    double part = 0.0;
    // The points fill half the registers: eight weights at a time, the sum
    // formed here (not put off until after the second transform, its points
    // kept for it), and no address kept through a transform.
#pragma unroll
    for (int l = 0; l < 2; l++)
#pragma unroll
        for (int h = 0; h < 16; h += 8) {
            asm volatile("" : "+v"(j));
            __builtin_amdgcn_sched_barrier(0);
            T w2[8];
#pragma unroll
            for (int q = 0; q < 8; q++) w2[q] = w[row(l, h + q)];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                w2[q] = valid ? w2[q] * w2[q] : (T)0;
                const C y = reg[l][h + q];
                part += (double)w2[q] * ((double)y.x * y.x + (double)y.y * y.y);
                reg[l][h + q] = cscale(y, (T)2 * w2[q]);
            }
            asm volatile("" : "+v"(part));
        }
    asm volatile("" : "+v"(j));
    __builtin_amdgcn_sched_barrier(0);
    line_fft_halves<T, L, 1>(reg, lds, LayCol<LPB>{b}, j, StageTwLds<T>{ltw});
    asm volatile("" : "+v"(j));
    if (full) {
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int q = 0; q < 16; q++) buf_st<C>(rs, off(), l * lst + q * qst, reg[l][q]);
    } else if (valid) {
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int q = 0; q < 16; q++) col[row(l, q)] = reg[l][q];
    }
    const double tot = block_sum<NTH>(part, red);
    if (threadIdx.x == 0) a.partial[tile] = tot;
}

// Elementwise weighting of a spectrum (batch x P complex), with loss partials
// per workgroup: blockIdx.y = transform, blockIdx.x = chunk of P.
template <typename T>
__global__ void __launch_bounds__(256) k_wpow_mask(void *buf, const void *w, double *partial, long long P)
{
    using C = Cx<T>;
    __shared__ double red[4];
    C *y = (C *)buf + (long long)blockIdx.y * P;
    const T *wt = (const T *)w;
    double part = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < P; i += (long long)gridDim.x * 256) {
        const T w2 = wt[i] * wt[i];
        const C v = y[i];
        part += (double)w2 * ((double)v.x * v.x + (double)v.y * v.y);
        y[i] = cscale(v, (T)2 * w2);
    }
    const double tot = block_sum<256>(part, red);
    if (threadIdx.x == 0) partial[(long long)blockIdx.y * gridDim.x + blockIdx.x] = tot;
}

// loss[t] = sum of the `per` partials of transform t, in index order.
__global__ void __launch_bounds__(64) k_wpow_reduce(const double *partial, double *loss, long long per)
{
    __shared__ double red[1];
    const double *p = partial + (long long)blockIdx.x * per;
    double v = 0.0;
    for (long long i = threadIdx.x; i < per; i += 64) v += p[i];
    const double tot = block_sum<64>(v, red);
    if (threadIdx.x == 0) loss[blockIdx.x] = tot;
}

}  // namespace nfft
