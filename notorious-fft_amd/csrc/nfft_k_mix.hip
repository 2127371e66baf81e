// nfft_k_mix.hip -- schedules and launchers of the one-pass mixed-radix lines.
#include "nfft_internal.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <map>
#include <tuple>

namespace nfft {

// instantiated in nfft_k_mix_f32.hip / nfft_k_mix_f64.hip
extern template __global__ void k_mix_line<float, false, float2>(MixArgs);
extern template __global__ void k_mix_line<float, false, double2>(MixArgs);
extern template __global__ void k_mix_line<float, true, float2>(MixArgs);
extern template __global__ void k_mix_line<double, false, double2>(MixArgs);
extern template __global__ void k_mix_line<double, true, double2>(MixArgs);
extern template __global__ void k_mix_tile<float, false>(MixTileArgs);
extern template __global__ void k_mix_tile<float, true>(MixTileArgs);
extern template __global__ void k_mix_tile<double, false>(MixTileArgs);

namespace {

constexpr int kRadices[] = {32, 30, 28, 27, 25, 24, 21, 20, 18, 16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// VALU instructions per point of a radix-r butterfly (two-level radices: both
// levels and the inner twiddles)
double dft_ops(int r)
{
    switch (r) {
    case 2: return 2;
    case 3: return 4.7;
    case 4: return 4;
    case 5: return 7.2;
    case 7: return 9.4;
    case 8: return 6.5;
    case 16: return 10.5;
    }
    static const int two[][2] = {{2, 3}, {3, 3}, {2, 5}, {4, 3}, {3, 5}, {4, 5}, {5, 5}, {2, 7}, {2, 9},
                                 {3, 7}, {3, 8}, {3, 9}, {4, 7}, {5, 6}, {4, 8}};
    for (auto &t : two)
        if (t[0] * t[1] == r) return dft_ops(t[0]) + dft_ops(t[1]) + 4.0 * (t[0] - 1) * (t[1] - 1) / r;
    return 20;
}

int gcd_int(int a, int b) { return b ? gcd_int(b, a % b) : a; }

float rcp_up_host(int d) { return (1.0f / (float)d) * 1.00000095367431640625f; }

// Fill the steps of radices r[0..ns) (execution order) for G lines; false if
// the lines do not fit the LDS.  Returns in *conflict the expected extra LDS
// cycles factor of the first stage's writes.
bool fill(MixPlan &p, int prec, int L, const int *r, int ns, bool blue, int G, MixLanes lanes, size_t lds_max,
          double *conflict)
{
    const size_t cb = prec == 0 ? 8 : 16;
    const int banks = prec == 0 ? 32 : 16;  // elements per LDS row of banks
    p.L = L;
    p.stages = ns;
    p.steps = blue ? 2 * ns - 1 : ns;
    p.blue = blue ? 1 : 0;
    p.G = G;
    p.inG = rcp_up_host(G);
    *conflict = 1.0;
    for (int pads = 2; pads >= 0; pads--) {
        long long lp = p.steps > 1 ? L : 0;
        int Ns = 1;
        for (int s = 0; s < p.steps; s++) {
            MixStep &t = p.st[s];
            const bool mid = blue && s == ns - 1;
            t.radix = s < ns ? r[s] : r[2 * (ns - 1) - s];
            t.ns = Ns;
            t.nb = L / t.radix;
            t.q = t.nb / Ns;
            t.inb = rcp_up_host(t.nb);
            t.ins = rcp_up_host(Ns);
            const int so = mid ? 1 : Ns, U = so * t.radix;
            t.pad = 0;
            t.gfast = lanes == MIX_LANES_LINES || (lanes == MIX_LANES_TRANSPOSE && s > 0 && s + 1 == p.steps) ? 1 : 0;
            if (s + 1 < p.steps) {
                if (so == 1) {
                    if (pads >= 1 && U % 2 == 0) t.pad = 1;
                    if (t.pad == 0) *conflict = std::max(*conflict, (double)gcd_int(U, banks) / 2);
                } else if (pads >= 2) {
                    const int w = ((so - U) % banks + banks) % banks;
                    if ((long long)(L / U) * w <= L / 16) t.pad = w;
                }
                lp = std::max(lp, (long long)(L / U) * (U + t.pad));
            }
            Ns = mid ? t.radix : Ns * t.radix;
        }
        if (lanes != MIX_LANES_POINTS && lp > 0) {
            // neighbouring lanes on neighbouring lines: line distance such that
            // G lines and the butterflies beside them fall on different banks
            int w = 1;
            while (w < G && w < banks) w <<= 1;
            lp += (((long long)(banks / w) - lp) % banks + banks) % banks;
        }
        p.lp = (int)lp;
        if ((size_t)lp * G * cb <= lds_max) return true;
        *conflict = 1.0;
    }
    return false;
}

// Estimated cost per line: instructions issued per wave and stage, scaled by
// how many waves a CU keeps to hide latencies with.
double cost_of(const MixPlan &p, int prec, double conflict)
{
    const size_t cb = prec == 0 ? 8 : 16;
    const size_t lds = std::max<size_t>((size_t)p.lp * p.G * cb, 1024);
    const int wv = p.nth / 64, vgpr_waves = prec == 0 ? 16 : 8;
    const int wg = std::max(1, std::min((int)(kMixLds / lds), vgpr_waves / wv));
    double c = 0;
    for (int s = 0; s < p.steps; s++) {
        const int total = p.G * p.st[s].nb, R = p.st[s].radix;
        const bool mid = p.blue && s == p.stages - 1;
        double waves = 0;
        for (int i = 0; i * p.nth < total; i++) waves += std::min(wv, (total - i * p.nth + 63) / 64);
        // a whole round of the workgroup takes as long as its busiest SIMD
        double simd = 0;
        for (int i = 0; i * p.nth < total; i++) simd += (std::min(wv, (total - i * p.nth + 63) / 64) + 3) / 4;
        const double per = R * (dft_ops(R) * (mid ? 2 : 1) + 16 + (s == 0 && R > 1 ? 4 * (conflict - 1) : 0)) + 50;
        c += (wg > 1 ? waves / 4 * 0.7 + simd * 0.3 : simd) * per + 60;
    }
    return c / p.G * (1.0 + 6.0 / (wg * wv));
}

// Time of one workgroup that has its CU to itself, in issue slots: the rounds
// of its busiest SIMD, and per stage a trip through LDS, a table load and a
// barrier.  The same in both precisions, whose instructions issue at one rate
// (weighing FP64's half as much again took smaller radices: mean over 24
// lengths from 480 to 196608 points, up to 40 lines, 4 % longer).
double latency_of(const MixPlan &p)
{
    double c = 0;
    for (int s = 0; s < p.steps; s++) {
        const int total = p.G * p.st[s].nb, R = p.st[s].radix, reps = (total + p.nth - 1) / p.nth;
        const int waves = (std::min(p.nth, total) + 63) / 64;
        const bool mid = p.blue && s == p.stages - 1;
        c += reps * ((waves + 3) / 4) * (R * (dft_ops(R) * (mid ? 2 : 1) + 16) + 50) + 350;
    }
    return c;
}

struct Search {
    int prec, L;
    bool blue;
    MixShape shape;
    double best = 1e300;
    MixPlan plan;
    int r[kMixMaxStages];

    void consider(int ns)
    {
        const int tmax = std::min(shape.nth_max, prec == 0 ? mix_threads<float>() : mix_threads<double>());
        // an odd radix first, if there is one: its writes need no padding
        int ord[kMixMaxStages];
        std::copy(r, r + ns, ord);
        for (int i = 0; i < ns; i++)
            if (ord[i] % 2) {
                std::rotate(ord, ord + i, ord + i + 1);
                break;
            }
        for (int G = shape.g_min; G <= shape.g_max; G = G < 8 ? G + 1 : G + G / 4) {
            MixPlan p;
            double conflict;
            if (!fill(p, prec, L, ord, ns, blue, G, shape.lanes, shape.lds_max, &conflict)) break;
            for (int nth = shape.nth_min; nth <= tmax; nth += 64) {
                bool ok = true;
                int most = 0;
                for (int s = 0; s < ns && ok; s++) {
                    const int total = G * (L / ord[s]);
                    ok = total <= nth * mix_reps(ord[s]);
                    most = std::max(most, total);
                }
                if (!ok) continue;
                if (nth > shape.nth_min && nth - 64 >= most) break;  // only idle waves beyond
                p.nth = nth;
                const double c = shape.few ? latency_of(p) : cost_of(p, prec, conflict);
                if (c < best) {
                    best = c;
                    plan = p;
                }
            }
        }
    }
    // every multiset of radices, in falling order, of at most `stages` stages
    void split(int left, int depth, int maxr, int stages)
    {
        if (left == 1) {
            if (depth) consider(depth);
            return;
        }
        if (depth == stages) return;
        for (int q : kRadices)
            if (q <= maxr && left % q == 0 && std::pow((double)q, stages - depth) >= left) {
                r[depth] = q;
                split(left / q, depth + 1, q, stages);
            }
    }
};

struct Found {
    double cost;
    MixPlan plan;
};
typedef std::tuple<int, int, int, int, int, int, int, int, size_t, bool> Key;
std::mutex g_mix_mu;
std::map<Key, Found> g_mix_plans;  // schedules are searched once per process

const Found &find(int prec, int L, bool blue, const MixShape &sh)
{
    const Key key(L, prec, blue ? 1 : 0, sh.g_min, sh.g_max, sh.nth_min, sh.nth_max, (int)sh.lanes, sh.lds_max, sh.few);
    std::lock_guard<std::mutex> lk(g_mix_mu);
    auto it = g_mix_plans.find(key);
    if (it == g_mix_plans.end()) {
        Search se;
        se.prec = prec;
        se.L = L;
        se.blue = blue;
        se.shape = sh;
        // the fewest stages possible and one more (few workgroups: two more)
        for (int stages = 1, found = 0; stages <= kMixMaxStages && found < (sh.few ? 3 : 2); stages++) {
            se.split(L, 0, 32, stages);
            if (se.best < 1e299) found++;
        }
        it = g_mix_plans.emplace(key, Found{se.best, se.plan}).first;
    }
    return it->second;
}

MixShape line_shape(int L)
{
    MixShape sh;
    sh.g_max = L >= 4096 ? 1 : std::min(256, 8192 / L);
    return sh;
}

}  // namespace

bool smooth7(long long v)
{
    if (v < 1) return false;
    for (int q : {2, 3, 5, 7})
        while (v % q == 0) v /= q;
    return v == 1;
}

int mix_max(int prec) { return (int)(kMixLds / (prec == F32 ? 8 : 16)); }

bool mix_fit(int prec, long long n, bool blue, const MixShape &sh, MixPlan *p, double *cost)
{
    if (n < 2 || n > mix_max(prec) || !smooth7(n)) return false;
    const Found &f = find(prec, (int)n, blue, sh);
    if (f.cost >= 1e299) return false;
    *p = f.plan;
    if (cost) *cost = f.cost;
    return true;
}

bool mix_plan(int prec, long long n, long long lines, MixPlan *p)
{
    MixShape sh = line_shape((int)n);
    // Small batches end with their longest workgroup: few lines in each, radices
    // around 10 (us, large batches' schedule / this / two LDS buffers: FP32 N = 1200
    // x 40 9.6 / 6.2 / 8.7, 10^4 x 20 13 / 11 / 16; FP64 720 x 40 10.2 / 6.2 / 6.5, 2000 x
    // 60 11.2 / 7.1 / 12.5, 720 x 729 11.2 / 8.0 / 9.1, 1000 x 1049 10.9 / 12.4 / 12.7, 480 x
    // 3277 12.6 / 11.3 / 18.3).  The kernels' registers leave room for four
    // workgroups a CU in FP32, two in FP64.  FP64 lines of up to 128 points gain
    // from it in larger batches, in groups of about 4096 points (100 x 31458 26.5 /
    // 22.5 / 24.7, x 83887 58.2 / 49.2 / 55.3; 360 x 11651 26.7 / 28.8 / 39.4).
    const long long points = lines * n, most = prec == F32 ? (n > 512 ? 1 << 19 : 1 << 20) : (n > 512 ? 9 << 16 : 5 << 19);
    const int groups = prec == F32 ? 1024 : 512;
    if (lines > 0 && points <= most) {
        sh.g_min = sh.g_max = (int)std::min<long long>(sh.g_max, (lines + groups - 1) / groups);
        sh.few = true;
    } else if (lines > 0 && prec == F64 && n > 32 && n <= 128 && points <= 9 << 20) {
        sh.g_min = sh.g_max = (int)(4096 / n);
        sh.few = true;
    }
    if (n < 2 || !mix_fit(prec, n, false, sh, p)) return false;
    // FP32 twiddle tables where Bluestein's error was the larger before (from
    // 513 to 10000 points; N = 1000 2.1e-7 -> 1.2e-7).  Shorter lines and those
    // beyond 10000 points would lose up to 3 % to products of two rounded
    // entries (N = 480 1.055e-7 -> 1.084e-7, 10125 1.413e-7 -> 1.459e-7, 10240
    // 1.259e-7 -> 1.293e-7; 10000 gains, 1.466e-7 -> 1.446e-7) and have the FP64
    // table (2^26 points: N = 10080 304 -> 323 us).
    p->tw64 = prec == F64 || n <= 512 || n > 10000 || sh.few;
    return true;
}

bool mix_blue_fit(int prec, long long n, MixShape sh, MixPlan *p)
{
    // 7-smooth lengths from 2n - 1 up to a quarter more: the cheapest
    const long long lo = 2 * n - 1, hi = std::min<long long>(mix_max(prec), lo + std::max<long long>(lo / 4, 4));
    const int points = sh.g_max;
    double best = 1e300;
    for (long long m = lo; m <= hi; m++) {
        MixPlan q;
        double c;
        sh.g_max = std::max<long long>(1, points / m);
        if (mix_fit(prec, m, true, sh, &q, &c) && c < best) {
            best = c;
            *p = q;
        }
    }
    return best < 1e299;
}

bool mix_blue_plan(int prec, long long n, MixPlan *p)
{
    MixShape sh;
    sh.g_max = 2 * n - 1 >= 4096 ? 4096 : 8192;  // points per workgroup
    return mix_blue_fit(prec, n, sh, p);
}

template <typename T, bool BLUE, class TW> static hipError_t mix_go(const MixArgs &a0, hipStream_t s)
{
    static const bool attr = [] {  // once per instantiation and process
        (void)hipFuncSetAttribute((const void *)k_mix_line<T, BLUE, TW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)kMixLds);
        (void)hipGetLastError();
        return true;
    }();
    (void)attr;
    if (a0.nlines < 1) return hipSuccess;
    MixArgs a = a0;
    // lines of a workgroup are addressed by 32-bit byte offsets
    const long long far = std::max(a.in_dist, a.out_dist);
    if ((far * (a.pl.G - 1) + a.pl.L) * (long long)sizeof(Cx<T>) >= (1LL << 32)) a.pl.G = 1;
    a.flat = !BLUE && a.pl.steps == 1 && a.in_dist == a.pl.L && a.out_dist == a.pl.L;
    if (a.flat && a.nlines * a.pl.L >= 1 << 21) {
        // 2048 points on 256 threads where that makes 1024 workgroups (2^24 points in us,
        // 1024 / 2048 / 4096: FP64 N = 3 115 / 98 / 103, 30 151 / 97 / 104, FP32 7 46 / 42 / 44)
        a.pl.G = 2048 / a.pl.L;
        a.pl.nth = 256;
    }
    const long long grid = (a.nlines + a.pl.G - 1) / a.pl.G;
    const size_t lds = (size_t)a.pl.G * (a.flat ? a.pl.L | 1 : a.pl.lp) * sizeof(Cx<T>);
    if (grid > 0x7fffffffLL || lds > kMixLds || a.pl.nth < 64 || a.pl.nth > mix_threads<T>()) return hipErrorInvalidValue;
    for (int i = 0; i < a.pl.steps && !a.flat; i++)  // every butterfly has its place in a thread
        if (a.pl.G * a.pl.st[i].nb > a.pl.nth * mix_reps(a.pl.st[i].radix)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_mix_line<T, BLUE, TW>), dim3((unsigned)grid), dim3(a.pl.nth), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_mix(int prec, const MixArgs &a, hipStream_t s)
{
    const bool blue = a.pl.blue != 0;
    if (blue && (!a.chirp || !a.H)) return hipErrorInvalidValue;
    const int slot = prof_on() ? prof_begin(s) : -1;
    const hipError_t e = prec == F32 ? (blue          ? mix_go<float, true, float2>(a, s)
                                        : a.pl.tw64 ? mix_go<float, false, double2>(a, s)
                                                    : mix_go<float, false, float2>(a, s))
                                     : (blue ? mix_go<double, true, double2>(a, s) : mix_go<double, false, double2>(a, s));
    if (slot >= 0)
        prof_end(slot, s, blue ? "k_mix_line(bluestein)" : "k_mix_line", prec, a.pl.L,
                 2.0 * (double)a.nlines * (blue ? a.n : a.pl.L) * (prec == F32 ? 8.0 : 16.0));
    return e;
}

// lines of L points, in tiles; strided lanes: neighbouring lines are the ones
// contiguous in memory, so a tile should span a segment of them
const TileFit &TileFits::get(int L, MixLanes lanes, bool blue)
{
    auto it = seen.find({L, (int)lanes, blue ? 1 : 0});
    if (it != seen.end()) return it->second;
    TileFit best;
    auto consider = [&](int g, int nth_min, size_t lds_max) {
        MixShape sh;
        sh.g_min = sh.g_max = g;
        sh.nth_min = nth_min;
        sh.nth_max = nth_max;
        sh.lanes = lanes;
        sh.lds_max = lds_max;
        sh.few = few;
        TileFit f;
        f.ok = mix_fit(prec, L, blue, sh, &f.plan, &f.cost);
        // a point read and written takes half an issue slot of its CU's share
        // of the memory bandwidth (few workgroups: a whole tile's in FP64), more
        // where a tile covers part of a segment
        if (f.ok && !(few && prec == F32))
            f.cost += 0.5 * (prec == F32 ? 1 : 2) * L * (few ? f.plan.G : 1) *
                      (lanes == MIX_LANES_POINTS ? 1.0 : std::max(1.0, (double)seg() / f.plan.G));
        if (f.ok && (!best.ok || f.cost < best.cost)) best = f;
        return f.ok;
    };
    int g = std::max(1, points / L);
    if (lanes != MIX_LANES_POINTS && g > seg()) g -= g % seg();
    g = std::min(g, 64);
    // as many workgroups of kTileThreads per CU as their registers allow (4 / 2)
    const size_t part = points <= 16 * kTileThreads ? (prec == F32 ? kMixLds / 4 : kMixLds / 2) : kMixLds;
    for (int h = g; h >= 1 && !consider(h, kTileThreads, part); h = h > 1 ? (h + 1) / 2 : 0) {}
    if (nth_max > kTileThreads && (!best.ok || (lanes != MIX_LANES_POINTS && g < seg())))
        for (int h = seg(); h >= 1; h /= 2) consider(h, kTileThreads, kMixLds);
    return seen.emplace(std::make_tuple(L, (int)lanes, blue ? 1 : 0), best).first->second;
}

TileStatus tile_plan(TileFits &fits, long long n, bool blue, TilePlan *p)
{
    // cost of all lines of a phase
    auto phase = [&](const TileFit &f, int lines) {
        if (fits.few) return f.ok ? f.cost : 1e300;  // all tiles at a time
        return f.ok ? f.cost * f.plan.G * ((lines + f.plan.G - 1) / f.plan.G) : 1e300;
    };
    const long long lo = 2 * n - 1;
    const int amax = fits.nth_max > kTileThreads ? 1280 : 1024, bmax = fits.nth_max > kTileThreads ? 4096 : 2048;
    double best = 1e299;
    int n1 = 0, n2 = 0;
    for (int a = 32; a <= amax; a++) {
        if (!smooth7(a) || (!blue && n % a)) continue;
        long long b = blue ? (lo + a - 1) / a : n / a;
        int tries = blue ? 2 : 1;
        for (; tries > 0 && b <= bmax; b++) {
            // Bluestein: rows of whole segments, so that tiles of columns are aligned
            if (!smooth7(b) || (blue && b % fits.seg())) continue;
            tries--;
            if (b < 32) continue;
            double c = phase(fits.get(a, MIX_LANES_LINES, false), (int)b);
            if (c >= best) continue;
            if (blue) c = 2 * c + phase(fits.get((int)b, MIX_LANES_POINTS, true), a);
            else c += phase(fits.get((int)b, MIX_LANES_TRANSPOSE, false), a);
            if (c < best) {
                best = c;
                n1 = a;
                n2 = (int)b;
            }
        }
    }
    if (best >= 1e299) return TILE_NONE;
    Tw2 tw2;
    const void *t1 = phase_table(F64, n1, 1, 0, n1), *t2 = phase_table(F64, n2, 1, 0, n2);
    if (!t1 || !t2 || !tw2_table((long long)n1 * n2, &tw2)) return TILE_FAILED;
    // the scratch holds rows of whole segments
    const int pitch = (n2 + fits.seg() - 1) / fits.seg() * fits.seg();
    p->n1 = n1;
    p->n2 = n2;
    p->elems = (long long)n1 * pitch;
    MixPhase cols{};
    cols.pl = fits.get(n1, MIX_LANES_LINES, false).plan;
    cols.tw = t1;
    cols.tw2 = tw2;
    cols.ig = cols.og = 1;
    cols.ip = n2;
    cols.op = pitch;
    cols.lines = n2;
    cols.nv = (int)n;
    cols.flags = MIX_HEAD | MIX_TW | (blue ? MIX_CHIRP_IN : 0);
    MixPhase rows = cols;
    rows.pl = fits.get(n2, blue ? MIX_LANES_POINTS : MIX_LANES_TRANSPOSE, blue).plan;
    rows.tw = t2;
    rows.ig = pitch;
    rows.ip = 1;
    rows.lines = n1;
    p->ph[0] = cols;
    if (blue) {
        rows.og = pitch;
        rows.op = 1;
        rows.flags = MIX_TW;
        cols.flags = MIX_TAIL | MIX_CHIRP_OUT;
        p->ph[2] = cols;
    } else {
        rows.og = 1;
        rows.op = n1;
        rows.flags = MIX_TAIL;
    }
    p->ph[1] = rows;
    p->phases = blue ? 3 : 2;
    return TILE_OK;
}

template <typename T, bool ONCE> static hipError_t mix_tile_go(const MixTileArgs &a, hipStream_t s)
{
    static const bool attr = [] {  // once per instantiation and process
        (void)hipFuncSetAttribute((const void *)k_mix_tile<T, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMixLds);
        (void)hipGetLastError();
        return true;
    }();
    (void)attr;
    const MixPlan &pl = a.ph.pl;
    if (a.ntrans < 1) return hipSuccess;
    const long long grid = a.ntrans * ((a.ph.lines + pl.G - 1) / pl.G);
    const size_t lds = (size_t)pl.G * pl.lp * sizeof(Cx<T>);
    if (grid > 0x7fffffffLL || lds > kMixLds || pl.nth < 64 || pl.nth > mix_threads<T>()) return hipErrorInvalidValue;
    if ((pl.blue && !a.ph.H) || ((a.ph.flags & (MIX_CHIRP_IN | MIX_CHIRP_OUT)) && !a.ph.chirp)) return hipErrorInvalidValue;
    for (int i = 0; i < pl.steps; i++)  // every butterfly has its place in a thread
        if (pl.G * pl.st[i].nb > pl.nth * mix_reps(pl.st[i].radix)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_mix_tile<T, ONCE>), dim3((unsigned)grid), dim3(pl.nth), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_mix_tile(int prec, const MixTileArgs &a, hipStream_t s)
{
    const int slot = prof_on() ? prof_begin(s) : -1;
    const hipError_t e = prec == F64 ? mix_tile_go<double, false>(a, s)
                         : a.blue ? mix_tile_go<float, false>(a, s) : mix_tile_go<float, true>(a, s);
    if (slot >= 0)
        prof_end(slot, s, "k_mix_tile", prec, a.ph.pl.L,
                 2.0 * (double)a.ntrans * a.ph.lines * a.ph.pl.L * (prec == F32 ? 8.0 : 16.0));
    return e;
}

}  // namespace nfft
