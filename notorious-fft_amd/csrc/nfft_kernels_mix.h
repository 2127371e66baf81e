// nfft_kernels_mix.h -- one-pass mixed-radix lines: 7-smooth lengths, and
// Bluestein over a 7-smooth convolution length, in one workgroup.
//
// A line of L = 2^a 3^b 5^c 7^d points is transformed by a self-sorting
// Stockham sequence of large register butterflies (radices up to 32, mostly
// 16 to 32, so that three stages cover up to 20480 points), one runtime
// schedule per length.  Stage s of radix R and stride Ns maps butterfly j
// (jq = j / Ns, k = j mod Ns) from points j + t L/R to points
// jq Ns R + k + t Ns.  The stage loop differs from smooth_lines in what it
// moves:
//   - the first stage reads its points from global memory and the last one
//     writes them there, so S stages make S - 1 exchanges through LDS and
//     the line crosses HBM once each way;
//   - one LDS buffer, not two: a stage's butterflies are all held in
//     registers (mix_reps of them per thread) between its reads and its
//     writes, so a line of 20480 FP32 points fits the 160 KB of a CU;
//   - a stage's output blocks of U = Ns R points are padded to U + pad
//     points.  The next radix divides L / U, so its reads L/R' apart are
//     whole blocks apart: the padding costs one term per butterfly, none per
//     point, and takes the strided writes of the first stages off one bank;
//   - the twiddles w^t of a butterfly come from about 2 sqrt(R) table
//     entries and one product each.
// The inverse transform conjugates on the way in and out.
//
// Bounds and measurements stand at k_mix_line.
#pragma once
#include "nfft_kernels_smooth.h"

namespace nfft {

constexpr int kMixMaxStages = 6;
constexpr int kMixMaxSteps = 2 * kMixMaxStages - 1;  // Bluestein: forward and inverse share the middle step
constexpr size_t kMixLds = 160 * 1024;

// One step of the schedule (all uniform): radix R at stride ns, nb = L / R
// butterflies per line in blocks of ns, q = nb / ns of them; `pad` points are
// added to each output block; inb / ins: reciprocals for fdiv.
struct MixStep {
    int radix, pad, nb, ns, q;
    float inb, ins;
};
struct MixPlan {
    int L = 0;
    int stages = 0, steps = 0;  // steps: stages, or 2 stages - 1 for Bluestein
    int G = 1;                  // lines per workgroup
    int nth = 0;                // threads per workgroup
    int lp = 0;                 // LDS points per line, padding included
    MixStep st[kMixMaxSteps];
};

// Threads the kernels are compiled for, and butterflies of radix R a thread
// may hold: 32 points (FP32: 64 VGPRs of data under the 128 of a
// 1024-thread workgroup; FP64: 128 under the 256 of 512 threads).
template <typename T> __host__ __device__ constexpr int mix_threads() { return sizeof(T) == 4 ? 1024 : 512; }
__host__ __device__ constexpr int mix_reps(int R) { return 32 / R; }

// w^t, t < R, applied to v: entry e of the table is e^{-2 pi i e / L}, w the
// entry `e`.  Powers t = Q h + l from the entries of l and Q h.
template <typename T, int R>
__device__ __forceinline__ void mix_twiddle(Cx<T> (&v)[R], __amdgpu_buffer_rsrc_t tw, int e)
{
    using C = Cx<T>;
    constexpr int Q = R <= 5 ? R : R <= 9 ? 3 : R <= 16 ? 4 : R <= 25 ? 5 : 6;
    constexpr int NH = (R - 1) / Q;
    const uint32_t eb = (uint32_t)e * (uint32_t)sizeof(C);
    C lo[Q], hi[NH + 1];
#pragma unroll
    for (int l = 1; l < Q; l++) lo[l] = buf_ld<C>(tw, eb * (uint32_t)l, 0);
#pragma unroll
    for (int h = 1; h <= NH; h++) hi[h] = buf_ld<C>(tw, eb * (uint32_t)(Q * h), 0);
#pragma unroll
    for (int t = 1; t < R; t++) {
        const int h = t / Q, l = t % Q;
        v[t] = cmul(v[t], h == 0 ? lo[l] : l == 0 ? hi[h] : cmul(hi[h], lo[l]));
    }
}

// One step of all the lines of a workgroup.  Every thread must call it.
template <typename T, int R, bool BLUE, class IO>
__device__ __forceinline__ void mix_step(const MixPlan &pl, int s, Cx<T> *lds, __amdgpu_buffer_rsrc_t tw, const IO &io)
{
    using C = Cx<T>;
    constexpr int B = mix_reps(R);
    const MixStep st = pl.st[s];
    const int total = pl.G * st.nb, nth = blockDim.x;
    const bool first = s == 0, last = s + 1 == pl.steps, mid = BLUE && s + 1 == pl.stages;
    const int up = st.ns + (first ? 0 : pl.st[s - 1].pad);  // padded input blocks
    const int rs = st.q * up;                               // LDS distance of points L / R apart
    const int so = mid ? 1 : st.ns;                         // output distance of a butterfly's points
    const int uo = so * R + st.pad;                         // padded output blocks
    C v[B][R];
    int wa[B], gg[B];
    const bool on = (int)threadIdx.x < total;
    if (on) {
#pragma unroll
        for (int i = 0; i < B; i++) {
            if (i > 0 && i * nth >= total) break;  // uniform
            int idx = threadIdx.x + i * nth;
            if (i > 0 && idx >= total) idx = total - 1;  // not stored
            const int g = fdiv(idx, st.inb), j = idx - __mul24(g, st.nb);
            gg[i] = g;
            int jq = j, k = 0;
            if (first) {
                io.template load<R>(v[i], g, j, st.nb);
            } else {
                jq = fdiv(j, st.ins);
                k = j - __mul24(jq, st.ns);
                const C *p = lds + (__mul24(g, pl.lp) + __mul24(jq, up) + k);
#pragma unroll
                for (int t = 0; t < R; t++) v[i][t] = p[t * rs];
                mix_twiddle<T, R>(v[i], tw, __mul24(k, st.q));
            }
            dft_any<R, -1>(v[i]);
            if constexpr (BLUE) {
                if (mid) {
                    io.template middle<R>(v[i], j, st.ns);
                    dft_any<R, -1>(v[i]);
                    jq = j;
                    k = 0;
                }
            }
            wa[i] = last ? k : __mul24(g, pl.lp) + __mul24(jq, uo) + k;
        }
    }
    if (!first) __syncthreads();  // every read of this buffer is done
    if (on) {
#pragma unroll
        for (int i = 0; i < B; i++) {
            if (i > 0 && i * nth >= total) break;
            if (i > 0 && (int)threadIdx.x + i * nth >= total) break;
            if (last) {
                io.template store<R>(v[i], gg[i], wa[i], st.ns);
            } else {
                C *p = lds + wa[i];
#pragma unroll
                for (int t = 0; t < R; t++) p[t * so] = v[i][t];
            }
        }
    }
    if (!last) __syncthreads();
}

#define NFFT_MIX_RADICES(X)                                                                                     \
    X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16) X(18) X(20) X(21) X(24) X(25) X(27)   \
    X(28) X(30) X(32)

template <typename T, bool BLUE, class IO>
__device__ __forceinline__ void mix_lines(const MixPlan &pl, Cx<T> *lds, const void *tw, const IO &io)
{
    const auto rt = buf_rsrc(tw);
    for (int s = 0; s < pl.steps; s++) {
        switch (pl.st[s].radix) {
#define NFFT_MIX_CASE(R) case R: mix_step<T, R, BLUE>(pl, s, lds, rt, io); break;
            NFFT_MIX_RADICES(NFFT_MIX_CASE)
#undef NFFT_MIX_CASE
        }
    }
}

// Contiguous lines in global memory.  BLUE: n < L points per line, times the
// chirp on both sides, the filter spectrum between the two transforms; the
// inverse of the convolution is conj(FFT(conj(.))), folded into the products.
template <typename T, bool BLUE> struct MixIoLine {
    using C = Cx<T>;
    __amdgpu_buffer_rsrc_t in, out, chirp, H;
    uint32_t idist, odist;  // bytes between lines
    int glast;              // last line of this workgroup
    int n;                  // BLUE: points per line
    T sg, sc;               // sign of the imaginary parts (-1: inverse), output scale

    template <int R> __device__ __forceinline__ void load(C (&v)[R], int g, int j, int nb) const
    {
        const uint32_t off = (uint32_t)min(g, glast) * idist;
        if constexpr (BLUE) {
#pragma unroll
            for (int t = 0; t < R; t++) {
                const int p = j + t * nb;
                const uint32_t pb = p < n ? (uint32_t)p * (uint32_t)sizeof(C) : 0u;
                if (t * nb < n) {  // uniform
                    C x = buf_ld<C>(in, off + pb, 0);
                    x.y *= sg;
                    x = cmul(x, buf_ld<C>(chirp, pb, 0));
                    v[t] = p < n ? x : cmk<C>((T)0, (T)0);
                } else {
                    v[t] = cmk<C>((T)0, (T)0);
                }
            }
        } else {
            const uint32_t o = off + (uint32_t)j * (uint32_t)sizeof(C), step = (uint32_t)nb * (uint32_t)sizeof(C);
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = buf_ld<C>(in, o, (uint32_t)t * step);
#pragma unroll
            for (int t = 0; t < R; t++) v[t].y *= sg;
        }
    }
    // v (points j + t ns of the spectrum) -> conj(v H)
    template <int R> __device__ __forceinline__ void middle(C (&v)[R], int j, int ns) const
    {
#pragma unroll
        for (int t = 0; t < R; t++)
            v[t] = cconj(cmul(v[t], buf_ld<C>(H, (uint32_t)j * (uint32_t)sizeof(C),
                                              (uint32_t)(t * ns) * (uint32_t)sizeof(C))));
    }
    template <int R> __device__ __forceinline__ void store(const C (&v)[R], int g, int k, int ns) const
    {
        if (g > glast) return;
        const uint32_t o = (uint32_t)g * odist + (uint32_t)k * (uint32_t)sizeof(C);
        const uint32_t step = (uint32_t)ns * (uint32_t)sizeof(C);
        const T sy = sc * sg;
#pragma unroll
        for (int t = 0; t < R; t++) {
            if constexpr (BLUE) {
                const int p = k + t * ns;
                if (p < n) {
                    const C z = cmulc(buf_ld<C>(chirp, (uint32_t)p * (uint32_t)sizeof(C), 0), v[t]);
                    buf_st<C>(out, o, (uint32_t)t * step, cmk<C>(z.x * sc, z.y * sy));
                }
            } else {
                buf_st<C>(out, o, (uint32_t)t * step, cmk<C>(v[t].x * sc, v[t].y * sy));
            }
        }
    }
};

struct MixArgs {
    const void *in;
    void *out;
    long long nlines;
    long long in_dist, out_dist;
    MixPlan pl;
    const void *tw;           // L entries e^{-2 pi i q / L}
    int inverse;
    double scale;
    int n;                    // Bluestein: transform length
    const void *chirp, *H;    // Bluestein: n chirp entries, L filter entries (scaled 1 / L)
};

// Bound: one read and one write of the lines where a CU keeps two workgroups
// (up to 10240 FP32 / 5120 FP64 points by LDS, 16 waves at 128 VGPRs); beyond,
// one workgroup alternates loading, stages and storing.  2^26 points, before
// (mixed-radix lines with two LDS buffers up to 2048 points, Bluestein or a
// two-pass four-step) and now: FP32 N = 100 346 -> 213 us (5.0 TB/s), N =
// 1000 489 -> 261, N = 10^4 800 -> 223 (4.8 TB/s), N = 20000 982 -> 363; FP64
// N = 100 598 -> 435 us, N = 1000 709 -> 516, N = 10^4 1365 -> 527.
template <typename T, bool BLUE> __global__ void __launch_bounds__(mix_threads<T>()) k_mix_line(MixArgs a)
{
    using C = Cx<T>;
    extern __shared__ char smem[];
    const long long l0 = (long long)blockIdx.x * a.pl.G;
    const long long rem = a.nlines - l0;
    MixIoLine<T, BLUE> io;
    io.in = buf_rsrc((const C *)a.in + l0 * a.in_dist);
    io.out = buf_rsrc((C *)a.out + l0 * a.out_dist);
    io.idist = (uint32_t)a.in_dist * (uint32_t)sizeof(C);
    io.odist = (uint32_t)a.out_dist * (uint32_t)sizeof(C);
    io.glast = (int)(rem < a.pl.G ? rem : a.pl.G) - 1;
    io.n = a.n;
    io.sg = a.inverse ? (T)-1 : (T)1;
    io.sc = (T)a.scale;
    io.chirp = buf_rsrc(a.chirp);
    io.H = buf_rsrc(a.H);
    mix_lines<T, BLUE>(a.pl, (C *)smem, a.tw, io);
}

}  // namespace nfft
