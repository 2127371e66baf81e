// nfft_kernels_tcol.h -- DCT / DST along a strided axis, in place.
//
// The axis of an N-D array whose trailing dimensions hold B >= 2 reals is
// transformed down the columns it stands in, without transposing the array:
// two neighbouring real columns are one complex column (the transforms are
// real-linear, so they act on both parts at once), and LPB neighbouring
// complex columns make a tile whose accesses are whole segments, as in k_col.
//
//   types 2 and 3 (src/07_legacy.h:757-1066): with the reorder v[n] = x[2n],
//   v[N-1-n] = x[2n+1], V = FFT_N(v) and w_k = e^{-i pi k/(2N)},
//     REDFT10  y[k] = w_k V[k] + conj(w_k) V[N-k]          (y[0] = 2 V[0])
//     REDFT01  U[k] = conj(w_k) (x[k] - i x[N-k]), x[N] = 0; v = IFFT_N(U)
//   hold for complex x as they stand; the RODFTs negate odd points and
//   reverse the spectrum.
//   type 4 (src/07_legacy.h:1091-1387): the N/2-point form of k_t4_line, once
//   for the real and once for the imaginary parts of a column.
//
// Bound: one read and one write of the array, in 128-byte segments: 1024 x
// 1024 x 16 in FP32 takes 35 us (3.8 TB/s).  The transposes it replaces read
// and wrote the array twice more, 27 us each way around a 45 us row pass
// (DCT-2 then DCT-3 of that array over both axes: 268 -> 153 us).
#pragma once
#include "nfft_kernels_rt.h"

namespace nfft {

struct TrigColArgs {
    const void *in;
    void *out;
    long long ncols;       // complex columns of one array (B / 2)
    long long total;       // of all arrays
    long long dist;        // complex elements per array (N * ncols)
    const void *tw;        // stage table (types 2, 3: N; type 4: N / 2)
    const void *t1;        // types 2, 3: e^{-i pi k/(2N)}, k < N; type 4: e^{-i pi n/N}
    const void *t2;        // type 4: e^{-i pi (2n+1)/(4N)}
    double scale;
    double w0;             // weight of the DC term
    int order;             // TileOrder (col_order)
};

// Column `c0 + b` of all arrays as a buffer view at the tile's first array
// and a byte offset; columns past the last one read column c0 and are not
// stored.
template <typename C> struct TrigCol {
    __amdgpu_buffer_rsrc_t in, out;
    uint32_t off, step;  // of point 0, between points
    bool live;
    __device__ __forceinline__ TrigCol(const TrigColArgs &a, long long c0, int b)
    {
        const long long t0 = c0 / a.ncols;  // uniform
        live = c0 + b < a.total;
        const long long c = live ? c0 + b : c0, t = c / a.ncols;
        in = buf_rsrc((const C *)a.in + t0 * a.dist);
        out = buf_rsrc((C *)a.out + t0 * a.dist);
        off = (uint32_t)((t - t0) * a.dist + (c - t * a.ncols)) * (uint32_t)sizeof(C);
        step = (uint32_t)a.ncols * (uint32_t)sizeof(C);
    }
    __device__ __forceinline__ C load(int p) const { return buf_ld<C>(in, off + (uint32_t)p * step, 0); }
    __device__ __forceinline__ void store(int p, C v) const { buf_st<C>(out, off + (uint32_t)p * step, 0, v); }
};

template <typename T, int N, int LPB, int OP>
__global__ void __launch_bounds__(Sched<N>::NT *LPB, (wpe_hint<T>(Sched<N>::NT *LPB, (long)N *LPB * sizeof(Cx<T>))))
k_t23_col(TrigColArgs a)
{
    using S = Sched<N>;
    using C = Cx<T>;
    __shared__ C lds[N * LPB];
    const int b = threadIdx.x % LPB, j = threadIdx.x / LPB;
    const TrigCol<C> col(a, xcd_order(blockIdx.x, gridDim.x, a.order) * LPB, b);
    const C *w = (const C *)a.t1;
    const T sc = (T)a.scale;
    const LayCol<LPB> lay{b};
    // reordered point n is point perm(n); odd points are negated by the DSTs
    auto perm = [](int n) { return n < (N + 1) / 2 ? 2 * n : 2 * (N - 1 - n) + 1; };
    auto sign = [](int n, C v) { return (OP == T_DST2 || OP == T_DST3) && n >= N / 2 ? cneg(v) : v; };
    C reg[S::R];
    if constexpr (OP == T_DCT2 || OP == T_DST2) {
#pragma unroll
        for (int q = 0; q < S::R; q++) {
            const int n = j + S::NT * q;
            reg[q] = sign(n, col.load(perm(n)));
        }
        line_fft<T, N, -1>(reg, lds, lay, j, (const double2 *)a.tw);
#pragma unroll
        for (int q = 0; q < S::R; q++) lds[lay(j + S::NT * q)] = reg[q];
        __syncthreads();
        if (!col.live) return;
#pragma unroll
        for (int q = 0; q < S::R; q++) {
            const int k = j + S::NT * q;
            const C u = cmul(reg[q], w[k]), v = cmulc(lds[lay((N - k) & (N - 1))], w[k]);
            C y = cscale(cadd(u, v), sc);
            if (k == 0) y = cscale(y, (T)a.w0);
            col.store(OP == T_DCT2 ? k : N - 1 - k, y);
        }
    } else {
#pragma unroll
        for (int q = 0; q < S::R; q++) {
            const int k = j + S::NT * q;
            reg[q] = col.load(OP == T_DCT3 ? k : N - 1 - k);
            lds[lay(k)] = reg[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < S::R; q++) {
            const int k = j + S::NT * q;
            const C m = lds[lay((N - k) & (N - 1))];
            reg[q] = k == 0 ? cscale(reg[q], (T)a.w0) : cmulc(cmk<C>(reg[q].x + m.y, reg[q].y - m.x), w[k]);
        }
        __syncthreads();
        line_fft<T, N, 1>(reg, lds, lay, j, (const double2 *)a.tw);
        if (!col.live) return;
#pragma unroll
        for (int q = 0; q < S::R; q++) {
            const int n = j + S::NT * q;
            col.store(perm(n), sign(n, cscale(reg[q], sc)));
        }
    }
}

template <typename T, int N, int LPB, int OP>
__global__ void __launch_bounds__(Sched<N / 2>::NT *LPB,
                                  (wpe_hint<T>(Sched<N / 2>::NT *LPB, (long)N *LPB * sizeof(Cx<T>))))
k_t4_col(TrigColArgs a)
{
    constexpr int L = N / 2;
    using S = Sched<L>;
    using C = Cx<T>;
    __shared__ C lds[N * LPB];
    const int b = threadIdx.x % LPB, j = threadIdx.x / LPB;
    const TrigCol<C> col(a, xcd_order(blockIdx.x, gridDim.x, a.order) * LPB, b);
    const C *pre = (const C *)a.t1, *post = (const C *)a.t2;
    const T sc = (T)2 * (T)a.scale;
    const LayCol<2 * LPB> lay[2] = {{b}, {b + LPB}};  // real parts, imaginary parts
    const int jj[2] = {j, j};
    C reg[2][S::R];
#pragma unroll
    for (int q = 0; q < S::R; q++) {
        const int n = j + S::NT * q;
        const C xe = col.load(2 * n), xo = col.load(N - 1 - 2 * n), p = pre[n];
        if constexpr (OP == T_DCT4) {
            reg[0][q] = cmul(p, cmk<C>(xe.x, xo.x));
            reg[1][q] = cmul(p, cmk<C>(xe.y, xo.y));
        } else {
            reg[0][q] = cneg(cmul(p, cmk<C>(xe.x, -xo.x)));
            reg[1][q] = cneg(cmul(p, cmk<C>(xe.y, -xo.y)));
        }
    }
    line_fft_tw_n<T, L, -1, 2>(reg, lds, lay, jj, StageTwGlobal{(const double2 *)a.tw});
#pragma unroll
    for (int l = 0; l < 2; l++)
#pragma unroll
        for (int q = 0; q < S::R; q++) lds[lay[l](j + S::NT * q)] = reg[l][q];
    __syncthreads();
    if (!col.live) return;
#pragma unroll
    for (int q = 0; q < S::R; q++) {
        const int k = j + S::NT * q;
        const C w0 = post[2 * k], w1 = post[2 * k + 1];
        T y0[2], y1[2];
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const C p0 = cmul(w0, reg[l][q]), p1 = cmul(w1, cconj(lds[lay[l](L - 1 - k)]));
            y0[l] = sc * (OP == T_DCT4 ? p0.x : p0.y);
            y1[l] = sc * (OP == T_DCT4 ? p1.x : p1.y);
        }
        col.store(2 * k, cmk<C>(y0[0], y0[1]));
        col.store(2 * k + 1, cmk<C>(y1[0], y1[1]));
    }
}

}  // namespace nfft
