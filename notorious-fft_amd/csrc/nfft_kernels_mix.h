// nfft_kernels_mix.h -- one-pass mixed-radix lines: 7-smooth lengths, and
// Bluestein over a 7-smooth convolution length, in one workgroup.
//
// A line of L = 2^a 3^b 5^c 7^d points is transformed by a self-sorting
// Stockham sequence of large register butterflies (radices up to 32, mostly
// 16 to 32, so that three stages cover up to 20480 points), one runtime
// schedule per length.  Stage s of radix R and stride Ns maps butterfly j
// (jq = j / Ns, k = j mod Ns) from points j + t L/R to points
// jq Ns R + k + t Ns.  What moves:
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
//     entries (two where an FP32 transform has FP64 entries) and products.
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
    int gfast;  // neighbouring lanes take neighbouring lines (else neighbouring butterflies)
};
struct MixPlan {
    int L = 0;
    int stages = 0, steps = 0;  // steps: stages, or 2 stages - 1 for Bluestein
    int blue = 0;               // Bluestein: step stages - 1 is the middle one
    int G = 1;                  // lines per workgroup
    float inG = 1.0f;           // its reciprocal for fdiv
    int nth = 0;                // threads per workgroup
    int lp = 0;                 // LDS points per line, padding included
    int tw64 = 0;               // lines: FP64 twiddle table (FP64 lines: always)
    MixStep st[kMixMaxSteps];
};

// Threads the kernels are compiled for, and butterflies of radix R a thread
// may hold: 32 points (FP32: 64 VGPRs of data under the 128 of a
// 1024-thread workgroup; FP64: 128 under the 256 of 512 threads).
template <typename T> __host__ __device__ constexpr int mix_threads() { return sizeof(T) == 4 ? 1024 : 512; }
__host__ __device__ constexpr int mix_reps(int R) { return 32 / R; }

// Buffer view of `bytes` bytes: loads beyond them return zero, stores beyond
// them are dropped, and kMixNone is beyond them.
constexpr uint32_t kMixNone = 0xfffffff0u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mix_rsrc(const void *base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

// w^t, t < R, applied to v: entry e of the table is e^{-2 pi i e / L}, w the
// entry `e`.  Powers t = Q h + l as products of the entries of l and Q h.
// W: type of the table entries.
// ONCE, FP32 transforms with FP64 entries (mix_plan says which lines have
// them, tiles do): the entries of w and w^Q alone, powers formed and
// applied in FP64 and rounded once.  With the powers rounded and applied in
// FP32 lengths were up to 5 % further off than with a table entry and four
// passes (N = 20000 1.42e-7 -> 1.49e-7; now 1.43e-7; N = 288 1.039e-7 ->
// 1.075e-7; now 1.030e-7), and the loads cost as much as the FP64 products
// (2^26 points: N = 20000 394 -> 359 us, 12000 375 -> 344, 288 202 -> 211, 480
// 202 -> 216, tiles of 10^6 636 -> 664).  Not the tiles of Bluestein, whose
// error is the convolution's (N = 33333 1533 -> 1632).
template <typename W, int R, bool ONCE, typename C>
__device__ __forceinline__ void mix_twiddle(C (&v)[R], __amdgpu_buffer_rsrc_t tw, int e)
{
    static_assert(!ONCE || sizeof(W) > sizeof(C), "FP32 transform, FP64 entries");
    constexpr int Q = R <= 5 ? R : R <= 9 ? 3 : R <= 16 ? 4 : R <= 25 ? 5 : 6;
    constexpr int NH = (R - 1) / Q;
    const uint32_t eb = (uint32_t)e * (uint32_t)sizeof(W);
    auto product = [](W a, W b) -> W {
        if constexpr (sizeof(a.x) == 8) return dmul(a, b);
        else return cmul(a, b);
    };
    W lo[Q], hi[NH + 1];
#pragma unroll
    for (int l = 1; l < Q; l++) lo[l] = ONCE && l > 1 ? product(lo[l / 2], lo[l - l / 2]) : buf_ld<W>(tw, eb * (uint32_t)l, 0);
#pragma unroll
    for (int h = 1; h <= NH; h++) hi[h] = ONCE && h > 1 ? product(hi[h / 2], hi[h - h / 2]) : buf_ld<W>(tw, eb * (uint32_t)(Q * h), 0);
#pragma unroll
    for (int t = 1; t < R; t++) {
        const int h = t / Q, l = t % Q;
        const W w = h == 0 ? lo[l] : l == 0 ? hi[h] : product(hi[h], lo[l]);
        if constexpr (ONCE) {
            const double2 z = dmul(make_double2(v[t].x, v[t].y), w);
            v[t] = cmk<C>((float)z.x, (float)z.y);
        } else {
            v[t] = cmul(v[t], cmk<C>((decltype(C::x))w.x, (decltype(C::x))w.y));
        }
    }
}

// One step of all the lines of a workgroup.  Every thread must call it.  PL:
// MixPlan, in any address space (kernel arguments or constant memory).
template <typename T, int R, bool BLUE, class PL, class IO>
__device__ __forceinline__ void mix_step(const PL &pl, int s, Cx<T> *lds, __amdgpu_buffer_rsrc_t tw, const IO &io)
{
    using C = Cx<T>;
    constexpr int B = mix_reps(R);
    const auto &ps = pl.st[s];
    const MixStep st{ps.radix, ps.pad, ps.nb, ps.ns, ps.q, ps.inb, ps.ins, ps.gfast};
    const int total = pl.G * st.nb, nth = blockDim.x;
    const bool first = s == 0, last = s + 1 == pl.steps, mid = BLUE && pl.blue && s + 1 == pl.stages;
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
            int g, j;
            if (st.gfast) {
                j = fdiv(idx, pl.inG);
                g = idx - __mul24(j, pl.G);
            } else {
                g = fdiv(idx, st.inb);
                j = idx - __mul24(g, st.nb);
            }
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
                mix_twiddle<typename IO::W, R, IO::kOnce>(v[i], tw, __mul24(k, st.q));
            }
            dft_any<R, -1>(v[i]);
            if constexpr (BLUE) {
                if (mid) {
                    io.template middle<R>(v[i], g, j, st.ns);
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

template <typename T, bool BLUE, class PL, class IO>
__device__ __forceinline__ void mix_lines(const PL &pl, Cx<T> *lds, const void *tw, const IO &io)
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

// Lines in global memory, points contiguous.  BLUE: n < L points per line,
// times the chirp on both sides, the filter spectrum between the two
// transforms; the inverse of the convolution is conj(FFT(conj(.))), folded
// into the products.  OFFS gives the byte offset of a line from the base of
// `in` / `out`.
template <typename T, bool BLUE, class OFFS, class TW = Cx<T>> struct MixIoLine {
    using C = Cx<T>;
    using W = TW;  // twiddle table entries
    static constexpr bool kOnce = sizeof(W) > sizeof(C);
    __amdgpu_buffer_rsrc_t in, out, chirp, H;  // in, out, chirp end with their last point
    OFFS offs;
    int glast;  // last line of this workgroup
    int n;      // BLUE: points per line
    T sg, sc;   // sign of the imaginary parts (-1: inverse), output scale

    template <int R> __device__ __forceinline__ void load(C (&v)[R], int g, int j, int nb) const
    {
        const uint32_t off = offs.in(min(g, glast));
        const uint32_t o = off + (uint32_t)j * (uint32_t)sizeof(C);
        const uint32_t step = (uint32_t)nb * (uint32_t)sizeof(C);
        if constexpr (BLUE) {
#pragma unroll
            for (int t = 0; t < R; t++) {
                const int p = j + t * nb;
                C x = buf_ld<C>(in, p < n ? o + (uint32_t)t * step : kMixNone, 0);
                x.y *= sg;
                v[t] = cmul(x, buf_ld<C>(chirp, (uint32_t)p * (uint32_t)sizeof(C), 0));
            }
        } else {
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = buf_ld<C>(in, o, (uint32_t)t * step);
#pragma unroll
            for (int t = 0; t < R; t++) v[t].y *= sg;
        }
    }
    // v (points j + t ns of the spectrum) -> conj(v H)
    template <int R> __device__ __forceinline__ void middle(C (&v)[R], int, int j, int ns) const
    {
#pragma unroll
        for (int t = 0; t < R; t++)
            v[t] = cconj(cmul(v[t], buf_ld<C>(H, (uint32_t)j * (uint32_t)sizeof(C),
                                              (uint32_t)(t * ns) * (uint32_t)sizeof(C))));
    }
    template <int R> __device__ __forceinline__ void store(const C (&v)[R], int g, int k, int ns) const
    {
        if (g > glast) return;
        const uint32_t o = offs.out(g) + (uint32_t)k * (uint32_t)sizeof(C);
        const uint32_t step = (uint32_t)ns * (uint32_t)sizeof(C);
        const T sy = sc * sg;
#pragma unroll
        for (int t = 0; t < R; t++) {
            if constexpr (BLUE) {
                const int p = k + t * ns;
                const C z = cmulc(buf_ld<C>(chirp, (uint32_t)p * (uint32_t)sizeof(C), 0), v[t]);
                buf_st<C>(out, p < n ? o + (uint32_t)t * step : kMixNone, 0, cmk<C>(z.x * sc, z.y * sy));
            } else {
                buf_st<C>(out, o, (uint32_t)t * step, cmk<C>(v[t].x * sc, v[t].y * sy));
            }
        }
    }
};

// lines at a fixed distance
struct MixDist {
    uint32_t idist, odist;  // bytes
    __device__ __forceinline__ uint32_t in(int g) const { return (uint32_t)g * idist; }
    __device__ __forceinline__ uint32_t out(int g) const { return (uint32_t)g * odist; }
};
// lines at offsets of their own, the first one the lowest
template <typename C> struct MixOffs {
    const long long *offs;  // elements
    long long base;
    __device__ __forceinline__ uint32_t in(int g) const { return (uint32_t)(offs[g] - base) * (uint32_t)sizeof(C); }
    __device__ __forceinline__ uint32_t out(int g) const { return in(g); }
};

struct MixArgs {
    const void *in;
    void *out;
    long long nlines;
    long long in_dist, out_dist;
    MixPlan pl;
    const void *tw;           // L entries e^{-2 pi i q / L}, FP64 where pl.tw64
    int inverse;
    double scale;
    int n;                    // Bluestein: transform length
    const void *chirp, *H;    // Bluestein: n chirp entries, L filter entries (scaled 1 / L)
    int flat = 0;             // mix_flat
};

// Lines of one butterfly, next to each other on both sides: copied through LDS
// in their order in memory, a line per thread in between.  Loaded straight, the
// lanes' lines lie R points apart (2^24 points, straight / copied in us: FP32 N = 7
// 71.5 / 42, 30 100 / 44, FP64 3 150 / 98, 30 153 / 98).
template <int R> __host__ __device__ constexpr int mix_flat_pitch() { return R % 2 ? R : R + 1; }
template <typename T, int R>
__device__ __forceinline__ void mix_flat(__amdgpu_buffer_rsrc_t in, __amdgpu_buffer_rsrc_t out, int cnt, T sg, T sc, Cx<T> *lds)
{
    using C = Cx<T>;
    constexpr int P = mix_flat_pitch<R>();
    const int total = cnt * R;
    auto at = [](int i) { return i / R * (P - R) + i; };
    for (int i0 = threadIdx.x; i0 < total; i0 += 8 * blockDim.x) {
        C x[8];
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = buf_ld<C>(in, (uint32_t)(i0 + k * blockDim.x) * (uint32_t)sizeof(C), 0);
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (i0 + k * (int)blockDim.x < total) lds[at(i0 + k * blockDim.x)] = x[k];
    }
    __syncthreads();
    for (int g = threadIdx.x; g < cnt; g += blockDim.x) {
        C v[R];
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = lds[g * P + t];
#pragma unroll
        for (int t = 0; t < R; t++) v[t].y *= sg;
        dft_any<R, -1>(v);
#pragma unroll
        for (int t = 0; t < R; t++) lds[g * P + t] = cmk<C>(v[t].x * sc, v[t].y * (sc * sg));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < total; i += blockDim.x) buf_st<C>(out, (uint32_t)i * (uint32_t)sizeof(C), 0, lds[at(i)]);
}

// Bound: one read and one write of the lines where a CU keeps two workgroups
// (up to 10240 FP32 / 5120 FP64 points by LDS, 16 waves at 128 VGPRs); beyond,
// one workgroup alternates loading, stages and storing.  2^26 points, before
// (mixed-radix lines with two LDS buffers up to 2048 points, Bluestein or a
// two-pass four-step) and now: FP32 N = 100 346 -> 212 us (5.1 TB/s), N =
// 1000 489 -> 253, N = 10^4 800 -> 222 (4.8 TB/s), N = 20000 982 -> 357; FP64
// N = 100 598 -> 435 us, N = 1000 709 -> 516, N = 10^4 1365 -> 527.  Counters
// of FP32 N = 10^4, and of Bluestein lines of 10007 points (15 waves a CU, 54 %
// vector issue, 69 % of their time waiting): profiles/mixed_radix_pmc.md.
template <typename T, bool BLUE, class TW> __global__ void __launch_bounds__(mix_threads<T>()) k_mix_line(MixArgs a)
{
    using C = Cx<T>;
    extern __shared__ char smem[];
    const long long l0 = (long long)blockIdx.x * a.pl.G;
    const long long rem = a.nlines - l0;
    const int cnt = (int)(rem < a.pl.G ? rem : a.pl.G);
    const MixDist d{(uint32_t)a.in_dist * (uint32_t)sizeof(C), (uint32_t)a.out_dist * (uint32_t)sizeof(C)};
    const uint32_t len = (uint32_t)(BLUE ? a.n : a.pl.L) * (uint32_t)sizeof(C);
    const MixIoLine<T, BLUE, MixDist, TW> io{mix_rsrc((const C *)a.in + l0 * a.in_dist, (uint32_t)(cnt - 1) * d.idist + len),
                                         mix_rsrc((C *)a.out + l0 * a.out_dist, (uint32_t)(cnt - 1) * d.odist + len),
                                         mix_rsrc(a.chirp, len),
                                         buf_rsrc(a.H),
                                         d,
                                         cnt - 1,
                                         a.n,
                                         a.inverse ? (T)-1 : (T)1,
                                         (T)a.scale};
    if constexpr (!BLUE) {
        if (a.flat) {
            switch (a.pl.L) {
#define NFFT_MIX_CASE(R) case R: mix_flat<T, R>(io.in, io.out, cnt, io.sg, io.sc, (C *)smem); break;
                NFFT_MIX_RADICES(NFFT_MIX_CASE)
#undef NFFT_MIX_CASE
            }
            return;
        }
    }
    mix_lines<T, BLUE>(a.pl, (C *)smem, a.tw, io);
}

// ---------------------------------------------------------------------------
// Tiles: G lines of an array with any line and point strides, the passes of
// transforms longer than one workgroup.
//   N = N1 x N2 (both 7-smooth), element n1 N2 + n2:
//     phase 1, columns [c0, c0 + G): FFT_N1, times w_N^{k1 c}, to scratch
//     phase 2, rows of the scratch: FFT_N2, stored transposed (k1 + N1 k2)
//   Bluestein over M = M1 x M2 >= 2N - 1 (both 7-smooth):
//     phase 1, columns: times the chirp, FFT_M1, times w_M^{k1 c}
//     phase 2, rows: FFT_M2, times the filter, conjugate, FFT_M2, times
//              w_M^{k1 c}, in place: the conjugate of the inverse's first half
//     phase 3, columns: FFT_M1, conjugate, times the chirp
// ---------------------------------------------------------------------------
enum { MIX_CHIRP_IN = 1, MIX_CHIRP_OUT = 2, MIX_TW = 4, MIX_HEAD = 8, MIX_TAIL = 16 };
struct MixPhase {
    MixPlan pl;
    const void *tw;            // L entries e^{-2 pi i q / L}: FP64, groups of Bluestein lines of the transform's type
    Tw2 tw2;                   // MIX_TW: two-level table of the whole length
    const void *chirp, *H;     // chirp entries below nv; filter in the layout of the rows
    int ig, ip, og, op;        // element distances of lines and points, input and output
    int lines;                 // lines of the phase (tiles of pl.G)
    int nv;                    // Bluestein: points of the transform
    int flags;                 // MIX_HEAD / MIX_TAIL: reads the input / writes the output of the transform
};

// Phases and items in constant memory: read through the scalar cache, and not
// again after every store.
typedef const MixPhase __attribute__((address_space(4))) MixPhaseK;

// v[t] *= w^{e0 + t es} (w = e^{-2 pi i / N}).  FP32: two table entries and
// two chains of FP64 products, rounded once.  FP64: the entries of every t (a
// chain would add an ulp per product).
template <int R, typename C>
__device__ __forceinline__ void mix_tw2(C (&v)[R], const Tw2 &tab, uint32_t e0, uint32_t es)
{
    if constexpr (sizeof(v[0].x) == 4) {
        double2 st = tw2_get(tab, es), b[2];
        b[0] = tw2_get(tab, e0);
        b[1] = dmul(b[0], st);
        st = dmul(st, st);
#pragma unroll
        for (int t = 0; t < R; t++) {
            v[t] = ctw64<-1>(v[t], b[t % 2]);
            if (t + 2 < R) b[t % 2] = dmul(b[t % 2], st);
        }
    } else {
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = ctw64<-1>(v[t], tw2_get(tab, e0 + (uint32_t)t * es));
    }
}

// PH: MixPhase, as a kernel argument or in constant memory.  ONCE: as
// mix_twiddle's.
template <typename T, class PH, bool ONCE> struct MixIoTile {
    using C = Cx<T>;
    using W = double2;  // twiddle table entries
    static constexpr bool kOnce = ONCE;
    const PH &ph;
    __amdgpu_buffer_rsrc_t in, out, chirp, H;  // in / out / H at line c0 (chirped sides: at the transform)
    int c0, glast;
    T sg, sc;                                  // inverse: -1 and the scale of the result

    template <int R> __device__ __forceinline__ void load(C (&v)[R], int g, int j, int nb) const
    {
        const int gc = min(g, glast), step = nb * ph.ip;
        if (ph.flags & MIX_CHIRP_IN) {  // `in` and `chirp` end with point nv - 1
            const uint32_t o = (uint32_t)((c0 + gc) * ph.ig + j * ph.ip) * (uint32_t)sizeof(C);
#pragma unroll
            for (int t = 0; t < R; t++) {
                C x = buf_ld<C>(in, o + (uint32_t)(t * step) * (uint32_t)sizeof(C), 0);
                x.y *= sg;
                v[t] = cmul(x, buf_ld<C>(chirp, o + (uint32_t)(t * step) * (uint32_t)sizeof(C), 0));
            }
            return;
        }
        const uint32_t o = (uint32_t)(gc * ph.ig + j * ph.ip) * (uint32_t)sizeof(C);
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = buf_ld<C>(in, o, (uint32_t)(t * step) * (uint32_t)sizeof(C));
        if (ph.flags & MIX_HEAD) {
#pragma unroll
            for (int t = 0; t < R; t++) v[t].y *= sg;
        }
    }
    template <int R> __device__ __forceinline__ void middle(C (&v)[R], int g, int j, int ns) const
    {
        const uint32_t o = (uint32_t)(min(g, glast) * ph.ig + j) * (uint32_t)sizeof(C);
#pragma unroll
        for (int t = 0; t < R; t++)
            v[t] = cconj(cmul(v[t], buf_ld<C>(H, o, (uint32_t)(t * ns) * (uint32_t)sizeof(C))));
    }
    template <int R> __device__ __forceinline__ void store(C (&v)[R], int g, int k, int ns) const
    {
        if (g > glast) return;
        if (ph.flags & MIX_TW) mix_tw2<R>(v, Tw2{ph.tw2.hi, ph.tw2.lo, ph.tw2.sh, ph.tw2.mask}, (uint32_t)(c0 + g) * (uint32_t)k, (uint32_t)(c0 + g) * (uint32_t)ns);
        const int step = ns * ph.op;
        if (ph.flags & MIX_CHIRP_OUT) {  // `out` and `chirp` end with point nv - 1
            const uint32_t o = (uint32_t)((c0 + g) * ph.og + k * ph.op) * (uint32_t)sizeof(C);
            const T sy = sc * sg;
#pragma unroll
            for (int t = 0; t < R; t++) {
                const uint32_t ot = o + (uint32_t)(t * step) * (uint32_t)sizeof(C);
                const C z = cmulc(buf_ld<C>(chirp, ot, 0), v[t]);
                buf_st<C>(out, ot, 0, cmk<C>(z.x * sc, z.y * sy));
            }
            return;
        }
        const uint32_t o = (uint32_t)(g * ph.og + k * ph.op) * (uint32_t)sizeof(C);
        if (ph.flags & MIX_TAIL) {
            const T sy = sc * sg;
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = cmk<C>(v[t].x * sc, v[t].y * sy);
        }
#pragma unroll
        for (int t = 0; t < R; t++) buf_st<C>(out, o, (uint32_t)(t * step) * (uint32_t)sizeof(C), v[t]);
    }
};

// Lines [c0, c0 + cnt) of phase `ph` of one transform (cnt <= ph.pl.G); src
// and dst at the transform (or its scratch).
template <typename T, bool ONCE, class PH>
__device__ __forceinline__ void mix_tile(const PH &ph, const Cx<T> *src, Cx<T> *dst, int c0, int cnt, int inverse,
                                         T scale, Cx<T> *lds)
{
    using C = Cx<T>;
    const uint32_t nb = (uint32_t)ph.nv * (uint32_t)sizeof(C);
    const MixIoTile<T, PH, ONCE> io{ph,
                    ph.flags & MIX_CHIRP_IN ? mix_rsrc(src, nb) : buf_rsrc(src + (long long)c0 * ph.ig),
                    ph.flags & MIX_CHIRP_OUT ? mix_rsrc(dst, nb) : buf_rsrc(dst + (long long)c0 * ph.og),
                    mix_rsrc(ph.chirp, nb),
                    buf_rsrc((const C *)ph.H + (long long)c0 * ph.ig),
                    c0,
                    cnt - 1,
                    inverse ? (T)-1 : (T)1,
                    scale};
    mix_lines<T, true>(ph.pl, lds, ph.tw, io);
}

// Item of workgroup b: kTileRun neighbouring items go to one XCD (workgroup b
// runs on XCD b mod 8), since tiles whose edges share 128-byte lines then
// share an L2 (the ragged batch of nfft_ragged.hip: 1.54 -> 1.42 ms, with
// its groups after the tiles and FP32 twiddles).
constexpr int kTileRun = 16;
__device__ __forceinline__ long long mix_item(long long b, long long nitems)
{
    const long long w = b % (8 * kTileRun);
    return b < nitems / (8 * kTileRun) * (8 * kTileRun) ? b - w + (w & 7) * kTileRun + (w >> 3) : b;
}

// One phase of a batch of transforms of one length.
struct MixTileArgs {
    const void *in;
    void *out;
    long long in_dist, out_dist;  // elements between transforms on either side
    long long ntrans;
    int inverse, blue;            // blue: a phase of Bluestein
    double scale;
    MixPhase ph;
};
// Bound: memory, as the ragged tiles (four workgroups of 4096 points per CU in
// FP32, two in FP64).  2^26 points, before (two LDS buffers per tile, radices
// up to 10; Bluestein over the next power of two) and now: FP32 N = 20736 1134
// -> 444 us, 196608 1225 -> 441, 10^6 1589 (Bluestein) -> 676, 33333 2496 ->
// 1580; FP64 20736 1810 -> 839, 196608 1969 -> 923, 33331 4441 -> 3697.
template <typename T, bool ONCE> __global__ void __launch_bounds__(mix_threads<T>()) k_mix_tile(MixTileArgs a)
{
    using C = Cx<T>;
    extern __shared__ char smem[];
    const int G = a.ph.pl.G, tiles = (a.ph.lines + G - 1) / G;
    const long long i = mix_item(blockIdx.x, a.ntrans * tiles), t = i / tiles;
    const int c0 = (int)(i - t * tiles) * G;
    mix_tile<T, ONCE>(a.ph, (const C *)a.in + t * a.in_dist, (C *)a.out + t * a.out_dist, c0, min(G, a.ph.lines - c0),
                a.inverse, (T)a.scale, (C *)smem);
}

// ---------------------------------------------------------------------------
// Ragged batches (nfft_ragged.hip): one launch per phase over a list of
// items, an item a tile of one long transform, or a group of same-size short
// transforms at any offsets.
// ---------------------------------------------------------------------------
struct RagItem {
    int phase;           // index of its MixPhase
    int c0, cnt;         // tiles: lines [c0, c0 + cnt); groups: cnt transforms
    int first;           // groups: first entry of the offset list
    long long src, dst;  // tiles: element offsets of the transform (or its scratch)
    int n;               // transform length
    int pow2;            // inverse not scaled
    int in_place;        // tiles: written back to the scratch
};
typedef const RagItem __attribute__((address_space(4))) RagItemK;
struct RagArgs {
    const void *in;
    void *out;
    const MixPhase *phases;
    const RagItem *items;
    int nitems;
    int inverse;
    const long long *offs;  // groups: element offset of each transform
    void *alt;              // tiles: scratch, the output of in-place items
};

template <typename T> __device__ __forceinline__ T rag_scale(const RagArgs &a, RagItemK &it)
{
    return a.inverse && !it.pow2 ? (T)1 / (T)it.n : (T)1;
}

// Groups of short transforms.  Lines have FP64 twiddle entries at every length
// (FP32 ones: 2 % further off on average than an entry per twiddle, N = 3136
// 1.20e-7 -> 1.29e-7, 14000 1.34e-7 -> 1.42e-7; now 4 % nearer, 1.19e-7 and
// 1.33e-7, for 1 to 3 % of the batch's time).  Bluestein lines, whose error is
// the convolution's, have entries of their type.
template <typename T, bool BLUE> __global__ void __launch_bounds__(mix_threads<T>()) k_rag_group(RagArgs a)
{
    using C = Cx<T>;
    extern __shared__ char smem[];
    RagItemK &it = ((RagItemK *)a.items)[blockIdx.x];
    MixPhaseK &ph = ((MixPhaseK *)a.phases)[it.phase];
    const long long *offs = a.offs + it.first;
    const long long base = offs[0];
    const C *in = (const C *)a.in + base;
    C *out = (C *)a.out + base;
    if (ph.pl.steps == 0) {  // one-point transforms
        for (int i = threadIdx.x; i < it.cnt; i += blockDim.x) out[offs[i] - base] = in[offs[i] - base];
        return;
    }
    const uint32_t len = (uint32_t)it.n * (uint32_t)sizeof(C);
    const uint32_t end = (uint32_t)(offs[it.cnt - 1] - base) * (uint32_t)sizeof(C) + len;
    using W = typename std::conditional<BLUE, C, double2>::type;
    const MixIoLine<T, BLUE, MixOffs<C>, W> io{mix_rsrc(in, end), mix_rsrc(out, end), mix_rsrc(ph.chirp, len),
                                            buf_rsrc(ph.H),    MixOffs<C>{offs, base}, it.cnt - 1,
                                            it.n,              a.inverse ? (T)-1 : (T)1, rag_scale<T>(a, it)};
    mix_lines<T, BLUE>(ph.pl, (C *)smem, ph.tw, io);
}

// Tiles of long transforms.
constexpr int kTileThreads = 256;
template <typename T> __global__ void __launch_bounds__(kTileThreads, (sizeof(T) == 4 ? 4 : 2)) k_rag_tile(RagArgs a)
{
    using C = Cx<T>;
    extern __shared__ char smem[];
    for (int b = blockIdx.x; b < a.nitems; b += gridDim.x) {
        const int i = (int)mix_item(b, a.nitems);
        RagItemK &it = ((RagItemK *)a.items)[i];
        MixPhaseK &ph = ((MixPhaseK *)a.phases)[it.phase];
        mix_tile<T, sizeof(T) == 4>(ph, (const C *)a.in + it.src, (C *)(it.in_place ? a.alt : a.out) + it.dst, it.c0, it.cnt, a.inverse, rag_scale<T>(a, it),
                    (C *)smem);
        __syncthreads();  // the next tile overwrites the buffer
    }
}

}  // namespace nfft
