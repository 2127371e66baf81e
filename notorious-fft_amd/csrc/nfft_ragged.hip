// nfft_ragged.hip -- ragged batches of mixed-size 1D complex transforms in
// one HIP graph launch.
//
// The reference has no batch API at all (src/07_legacy.h:29-57); a caller
// with many transforms of different sizes loops over plans on the CPU.  Here
// the host sorts the transforms by what one workgroup holds
// (nfft_kernels_mix.h) and the whole batch is a handful of launches:
//   - short transforms, in groups of one size: lines of any 7-smooth length
//     (powers of two among them) up to 20480 points (FP32) / 10240 (FP64),
//     and Bluestein lines whose M >= 2N - 1 is as short, the power of two up
//     to 4096 points and 7-smooth beyond; one launch per workgroup size and
//     form;
//   - long transforms, in tiles: 7-smooth N = N1 x N2 in two phases (columns,
//     rows), Bluestein over M = M1 x M2 in three (columns, rows, columns); one
//     launch per phase over the tiles of all of them, the intermediate of each
//     in a scratch region of its own.
// The phases follow each other by the order of the stream: no tile waits for
// another inside a kernel; the short transforms run beside them on a second
// branch of the graph (1.42 -> 1.36 ms on the batch below, with FP32 twiddles).
// Batches whose intermediates exceed the scratch budget (NFFT_RAGGED_MB) run in
// several such sequences.
//
// One persistent launch with queued tiles and dependency waits, over the
// power-of-two lines and two-buffer mixed-radix tiles, took 2.43 ms (FP32) for
// 10,000 sizes log-uniform in [16, 65536], 40 % of them primes (80.5 M
// points); this form takes 1.41 ms (1.35 with FP32 twiddles; FP64 5.0 -> 3.0
// ms).  What changed with it: M beyond 4096 points is 7-smooth instead of the
// next power of two, transforms of up to 20480 points cross memory once, and a
// tile's stages run in registers.
// The tile launches wait for memory: 16 waves a CU, 70 to 72 % of their time
// waiting, 3.3 to 3.7 TB/s over 128-byte segments, vector issue 29 to 40 %
// (profiles/mixed_radix_pmc.md).
// Inverse transforms follow the reference's normalisation: unnormalised for
// powers of two, 1/N for other lengths (src/05_algorithms.h:315-333).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/notorious_fft_hip.h"
#include "nfft_internal.h"

namespace nfft {
// instantiated in nfft_k_rag_f32.hip / nfft_k_rag_f64.hip
extern template __global__ void k_rag_group<float, false>(RagArgs);
extern template __global__ void k_rag_group<float, true>(RagArgs);
extern template __global__ void k_rag_tile<float>(RagArgs);
extern template __global__ void k_rag_group<double, false>(RagArgs);
extern template __global__ void k_rag_group<double, true>(RagArgs);
extern template __global__ void k_rag_tile<double>(RagArgs);
}  // namespace nfft

using namespace nfft;

namespace {
bool is_pow2(long long n) { return n > 0 && (n & (n - 1)) == 0; }
int env_int_rg(const char *name, int dflt)
{
    const char *v = getenv(name);
    return v && *v ? atoi(v) : dflt;
}
// Tile size (points per thread of a tile) and scratch budget (quarters of the
// default) of the batch being created: set by the autotuner around its
// candidate builds and from a tuning record (0: the defaults).
struct RagShape {
    int gpt = 0, lag4 = 0;
};
thread_local RagShape t_rag_shape;

// Workgroups of the short transforms.  FP32: four of 256 threads, two of 512
// or one of 1024 share a CU (16 waves of 128 VGPRs; a quarter, half or all of
// the LDS); FP64: two of 256 or one of 512.
struct GroupClass {
    int nth;
    size_t lds;
};
const GroupClass kClass32[] = {{256, 40 * 1024}, {512, 80 * 1024}, {1024, 160 * 1024}};
const GroupClass kClass64[] = {{256, 80 * 1024}, {512, 160 * 1024}};
constexpr int kClasses = 3;
int n_classes(int prec) { return prec == F32 ? 3 : 2; }
const GroupClass &group_class(int prec, int c) { return prec == F32 ? kClass32[c] : kClass64[c]; }

struct GraphKey {
    const void *in;
    void *out;
    int inv;
    bool operator<(const GraphKey &o) const
    {
        if (in != o.in) return in < o.in;
        if (out != o.out) return out < o.out;
        return inv < o.inv;
    }
};

struct Range {
    int first = 0, count = 0;
};
}  // namespace

struct nfft_ragged {
    int prec = 0;
    int count = 0;
    long long total = 0;
    void *d_phases = nullptr, *d_items = nullptr, *d_offs = nullptr, *d_h = nullptr;
    void *scratch = nullptr;               // intermediates of one sequence of long transforms
    std::vector<Range> tiles;              // 3 per sequence: the phases' items
    Range groups[kClasses][2];             // short transforms: items by class, plain / Bluestein
    size_t tile_lds = 0, group_lds[kClasses][2] = {};
    int tile_grid = 0;                     // workgroups of a tile launch (0: one per item)
    hipStream_t cap = nullptr, side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    std::map<GraphKey, std::pair<hipGraph_t, hipGraphExec_t>> graphs;
};

template <typename T> static hipError_t launch_parts(const nfft_ragged *r, int inverse, const void *in, void *out, hipStream_t s)
{
    RagArgs a{in, out, (const MixPhase *)r->d_phases, nullptr, 0, inverse, (const long long *)r->d_offs};
    const RagItem *items = (const RagItem *)r->d_items;
    // the short transforms run beside the tiles, on a second branch
    hipError_t e = hipEventRecord(r->fork, s);
    if (e == hipSuccess) e = hipStreamWaitEvent(r->side, r->fork, 0);
    if (e != hipSuccess) return e;
    for (size_t i = 0; i < r->tiles.size(); i++) {
        if (!r->tiles[i].count) continue;
        // phase 1 reads the input, the last one of a transform writes the output
        const int ph = (int)(i % 3);
        a.in = ph == 0 ? in : r->scratch;
        a.out = ph == 0 ? r->scratch : out;
        a.alt = r->scratch;
        a.items = items + r->tiles[i].first;
        a.nitems = r->tiles[i].count;
        const int grid = r->tile_grid > 0 ? std::min(r->tile_grid, a.nitems) : a.nitems;
        hipLaunchKernelGGL((k_rag_tile<T>), dim3(grid), dim3(kTileThreads), r->tile_lds, s, a);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    a.in = in;
    a.out = out;
    for (int c = kClasses - 1; c >= 0; c--)
        for (int b = 0; b < 2; b++) {
            const Range &g = r->groups[c][b];
            if (!g.count) continue;
            a.items = items + g.first;
            a.nitems = g.count;
            const dim3 grid(g.count), block(group_class(r->prec, c).nth);
            if (b) hipLaunchKernelGGL((k_rag_group<T, true>), grid, block, r->group_lds[c][b], r->side, a);
            else hipLaunchKernelGGL((k_rag_group<T, false>), grid, block, r->group_lds[c][b], r->side, a);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    e = hipEventRecord(r->join, r->side);
    return e == hipSuccess ? hipStreamWaitEvent(s, r->join, 0) : e;
}

static int launch_ragged(nfft_ragged *r, int inverse, const void *in, void *out, hipStream_t s)
{
    const hipError_t e = r->prec == F32 ? launch_parts<float>(r, inverse, in, out, s) : launch_parts<double>(r, inverse, in, out, s);
    return e == hipSuccess ? NFFT_OK : NFFT_E_HIP;
}

template <typename T> static void lds_attr()
{
    static const bool done = [] {  // once per precision and process
        const void *f[] = {(const void *)k_rag_tile<T>, (const void *)k_rag_group<T, false>, (const void *)k_rag_group<T, true>};
        for (const void *p : f) (void)hipFuncSetAttribute(p, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMixLds);
        (void)hipGetLastError();
        return true;
    }();
    (void)done;
}

static void ragged_free(nfft_ragged *r)
{
    for (auto &kv : r->graphs) {
        (void)hipGraphExecDestroy(kv.second.second);
        (void)hipGraphDestroy(kv.second.first);
    }
    void *ptrs[] = {r->d_phases, r->d_items, r->d_offs, r->d_h, r->scratch};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (r->fork) (void)hipEventDestroy(r->fork);
    if (r->join) (void)hipEventDestroy(r->join);
    if (r->side) (void)hipStreamDestroy(r->side);
    if (r->cap) (void)hipStreamDestroy(r->cap);
    delete r;
}

// Tuning records are keyed by precision and size list: "ragged p<prec>
// c<count> h2:<hash> <form>", 1 for a workgroup per tile, 2 to 4 for a resident
// grid of so many workgroups per CU, and "ragged-gl ... <points per thread of a
// tile x 100 + quarters of the scratch budget>".  Those of the persistent
// kernel, whose numbers meant other things, have h and not h2: in their keys.
static std::string tune_key(int prec, const std::vector<int> &sizes)
{
    unsigned long long h = 1469598103934665603ULL;
    for (int v : sizes) h = (h ^ (unsigned long long)v) * 1099511628211ULL;
    char b[96];
    snprintf(b, sizeof b, "ragged p%d c%zu h2:%016llx", prec, sizes.size(), h);
    return b;
}

static int tune_lookup(const std::string &key)
{
    const char *path = getenv("NFFT_TUNE_CACHE");
    if (!path || !*path) return 0;
    FILE *f = fopen(path, "r");
    if (!f) return 0;
    char line[256];
    int found = 0;
    const size_t kl = key.size();
    while (fgets(line, sizeof line, f)) {
        if (strncmp(line, key.c_str(), kl) == 0 && line[kl] == ' ') found = atoi(line + kl + 1);
    }
    fclose(f);
    return found;
}

static void tune_store(const std::string &key, int val)
{
    const char *path = getenv("NFFT_TUNE_CACHE");
    if (!path || !*path) return;
    FILE *f = fopen(path, "a");
    if (!f) return;
    fprintf(f, "%s %d\n", key.c_str(), val);
    fclose(f);
}

// Status of a failed table / engine setup: NFFT_E_ALLOC when a device
// allocation failed since `fails0` (alloc_failures()), else NFFT_E_HIP.
static int setup_fail(long long fails0) { return alloc_failures() > fails0 ? NFFT_E_ALLOC : NFFT_E_HIP; }

namespace {
enum Kind { K_GROUP, K_GROUP_BLUE, K_TWO, K_THREE };
struct Size {
    Kind kind = K_GROUP;
    int cls = 0;           // groups: workgroup class
    int phase = 0;         // first of its phases
    int n1 = 0, n2 = 0;    // long transforms
    long long elems = 0;   // their scratch
    long long h = 0;       // Bluestein: filter offset in d_h
    int m = 0;             // Bluestein length
    std::vector<int> ids;  // its transforms
};
}  // namespace

// Filters of the Bluestein sizes, in FP64 on the device: one engine per M,
// the buffers shared in stream order.
static bool build_filters(nfft_ragged *r, const std::map<int, Size> &sizes, long long h_elems)
{
    const size_t cb = cx_bytes(r->prec);
    if (!h_elems) return true;
    if (dev_malloc(&r->d_h, (size_t)h_elems * cb) != hipSuccess) return false;
    std::map<int, C2C> engines;
    long long mmax = 0, smax = 0;
    bool ok = true;
    for (auto &kv : sizes) {
        const int m = kv.second.m;
        if (!m || engines.count(m)) continue;
        C2C e;
        ok = e.init(m, F64, 1, 0);
        if (!ok) e.release();
        else engines[m] = e;
        if (!ok) break;
        mmax = std::max<long long>(mmax, m);
        smax = std::max(smax, e.scratch_per_line);
    }
    void *hb = nullptr, *Hb = nullptr, *sb = nullptr;
    ok = ok && dev_malloc(&hb, (size_t)mmax * 16) == hipSuccess && dev_malloc(&Hb, (size_t)mmax * 16) == hipSuccess &&
         (smax == 0 || dev_malloc(&sb, (size_t)smax * 16) == hipSuccess);
    for (auto &kv : sizes) {
        const Size &z = kv.second;
        if (!z.m || !ok) continue;
        const double2 *chirp64 = nullptr;
        ok = chirp_table(r->prec, kv.first, &chirp64) && chirp64 &&
             launch_blue_filter((double2 *)hb, chirp64, kv.first, z.m, r->cap) == hipSuccess &&
             engines[z.m].run(hb, Hb, 1, z.m, z.m, -1, 1.0, sb, 1, r->cap) == hipSuccess &&
             launch_blue_hprep((const double2 *)Hb, (char *)r->d_h + (size_t)z.h * cb, r->prec, z.m,
                               z.kind == K_THREE ? z.n1 : 0, z.n2, 1.0 / (double)z.m, r->cap) == hipSuccess;
    }
    ok = hipStreamSynchronize(r->cap) == hipSuccess && ok;
    for (void *p : {hb, Hb, sb})
        if (p) (void)hipFree(p);
    for (auto &kv : engines) kv.second.release();
    return ok;
}

static int ragged_create_impl(nfft_ragged **out, int prec, int count, const int *sizes, int flags)
{
    clear_error();
    const long long fails0 = alloc_failures();
    if (!out || count < 1 || !sizes || (prec != NFFT_F32 && prec != NFFT_F64)) {
        set_error("invalid ragged arguments");
        return NFFT_E_INVALID;
    }
    *out = nullptr;
    // every size is checked before any device work
    for (int i = 0; i < count; i++) {
        if (sizes[i] < 1) {
            set_error("ragged sizes must be >= 1");
            return NFFT_E_SIZE;
        }
        if (sizes[i] > 65536) {
            set_error("ragged batches support N <= 65536");
            return NFFT_E_UNSUPPORTED;
        }
    }
    nfft_ragged *r = new (std::nothrow) nfft_ragged();
    if (!r) return NFFT_E_ALLOC;
    const auto fail = [&](const char *what) {
        const int st = setup_fail(fails0);
        set_error(what);
        ragged_free(r);
        return st;
    };
    r->prec = prec;
    r->count = count;
    const size_t cb = cx_bytes(prec);
    std::vector<long long> offs(count);
    std::map<int, Size> by_size;
    for (int i = 0; i < count; i++) {
        offs[i] = r->total;
        r->total += sizes[i];
        by_size[sizes[i]].ids.push_back(i);
    }
    if (hipStreamCreateWithFlags(&r->cap, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&r->side, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&r->fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&r->join, hipEventDisableTiming) != hipSuccess)
        return fail("ragged setup: no stream");
    if (prec == F32) lds_attr<float>();
    else lds_attr<double>();

    // schedules and tables of every size
    // 16 points per thread of a tile: four workgroups (FP32) share a CU
    const int gpt = std::max(1, env_int_rg("NFFT_RAGGED_GPT", t_rag_shape.gpt > 0 ? t_rag_shape.gpt : 16));
    TileFits fits{prec, std::min(gpt, 32) * kTileThreads, kTileThreads, {}};
    // Short transforms of small batches take the schedules that end first, a line or
    // a few to a workgroup (us, persistent kernel before / large batches' schedules /
    // these: FP32 sizes below 1000 x 30 24.5 / 28.7 / 22.5, x 200 26.0 / 30.2 / 23.7, x 400 27.1 /
    // 30.9 / 23.3, x 2000, 0.5 M points in all, 37.0 / 31.5 / 25.2; FP64 x 800, 0.2 M points,
    // 34.5 / 26.5 by the last two, but x 2000 36.3 / 38.1), but not Bluestein lines of
    // more than 4096 points (10007 x 1 143 / 37 / 44).
    const bool few = env_int_rg("NFFT_FEW", 1) != 0 && r->total <= (prec == F32 ? 1 << 19 : 1 << 18);
    std::vector<MixPhase> phases;
    long long h_elems = 0;
    for (auto &kv : by_size) {
        const int n = kv.first;
        Size &z = kv.second;
        z.phase = (int)phases.size();
        MixPhase ph{};
        ph.nv = n;
        if (n == 1) {  // copied: no steps
            ph.pl.G = 256;
            phases.push_back(ph);
            continue;
        }
        const bool blue = !smooth7(n);
        // Bluestein's M: the next power of two up to 4096, else the cheapest
        // 7-smooth length from 2n - 1 on.  The error falls with M / n, and a
        // 7-smooth M takes that away from lengths just above a power of two
        // (N = 1103, M = 4096 and a 7-smooth one from 2205 on: FP64 4.37e-16 and
        // 5.77e-16, FP32 1.81e-7 and 1.96e-7); beyond 4096 the one pass makes up for it (N = 2053
        // FP64 7.39e-16 in three passes over 8192 points, 5.81e-16 in one).
        int m2 = 1;
        while (m2 < 2 * n - 1) m2 <<= 1;
        bool one = false;
        for (int c = 0; c < n_classes(prec) && !one; c++) {
            const GroupClass &gc = group_class(prec, c);
            MixShape sh;
            sh.nth_min = sh.nth_max = gc.nth;
            sh.lds_max = gc.lds;
            sh.few = few && !(blue && m2 > 4096);
            const int points = 16 * gc.nth;
            sh.g_max = blue ? points : std::max(1, std::min(256, points / n));
            if (few && !blue) sh.g_min = sh.g_max = std::min(sh.g_max, (count + 1023) / 1024);
            if (blue && m2 <= 4096) {
                sh.g_max = std::max(1, points / m2);
                one = mix_fit(prec, m2, true, sh, &ph.pl);
            } else {
                one = blue ? mix_blue_fit(prec, n, sh, &ph.pl) : mix_fit(prec, n, false, sh, &ph.pl);
            }
            z.cls = c;
        }
        if (blue) {
            const double2 *chirp64 = nullptr;
            ph.chirp = chirp_table(prec, n, &chirp64);
            if (!ph.chirp) return fail("ragged setup: chirp table");
        }
        if (one) {
            z.kind = blue ? K_GROUP_BLUE : K_GROUP;
            if (blue) {
                z.m = ph.pl.L;
                z.h = h_elems;
                h_elems += z.m;
            }
            ph.tw = phase_table(blue ? prec : F64, ph.pl.L, 1, 0, ph.pl.L);
            if (!ph.tw) return fail("ragged setup: twiddle table");
            size_t &lds = r->group_lds[z.cls][blue ? 1 : 0];
            lds = std::max(lds, (size_t)ph.pl.lp * ph.pl.G * cb);
            phases.push_back(ph);
            continue;
        }
        TilePlan tp;
        const TileStatus ts = tile_plan(fits, n, blue, &tp);
        if (ts == TILE_FAILED) return fail("ragged setup: twiddle tables");
        if (ts == TILE_NONE) {
            set_error("ragged setup: no split");
            ragged_free(r);
            return NFFT_E_UNSUPPORTED;
        }
        z.kind = blue ? K_THREE : K_TWO;
        z.n1 = tp.n1;
        z.n2 = tp.n2;
        z.elems = tp.elems;
        if (blue) {
            z.m = tp.n1 * tp.n2;
            z.h = h_elems;
            h_elems += z.m;
        }
        for (int k = 0; k < tp.phases; k++) {
            tp.ph[k].chirp = ph.chirp;
            phases.push_back(tp.ph[k]);
        }
        for (size_t k = z.phase; k < phases.size(); k++)
            r->tile_lds = std::max(r->tile_lds, (size_t)phases[k].pl.lp * phases[k].pl.G * cb);
    }
    if (!build_filters(r, by_size, h_elems)) return fail("ragged setup: Bluestein filters");
    for (auto &kv : by_size)
        if (kv.second.m) phases[kv.second.phase + (kv.second.kind == K_THREE ? 1 : 0)].H = (char *)r->d_h + (size_t)kv.second.h * cb;

    // long transforms, longest first, in sequences whose intermediates fit
    // the scratch budget
    std::vector<RagItem> items;
    struct Long {
        int id, n;
        long long elems;
    };
    std::vector<Long> longs;
    for (auto &kv : by_size)
        if (kv.second.kind == K_TWO || kv.second.kind == K_THREE)
            for (int id : kv.second.ids) {
                longs.push_back({id, kv.first, kv.second.elems});
            }
    std::stable_sort(longs.begin(), longs.end(), [](const Long &a, const Long &b) { return a.elems > b.elems; });
    const long long dflt_mb = t_rag_shape.lag4 > 0 ? 1024LL * t_rag_shape.lag4 : 4096;
    const long long budget = (((long long)std::max(1, env_int_rg("NFFT_RAGGED_MB", (int)dflt_mb))) << 20) / (long long)cb;
    long long scratch = 0;
    for (size_t b = 0; b < longs.size();) {
        size_t e = b;
        long long used = 0;
        std::vector<long long> at;
        while (e < longs.size() && (e == b || used + longs[e].elems <= budget)) {
            at.push_back(used);
            used += longs[e++].elems;
        }
        scratch = std::max(scratch, used);
        for (int p = 0; p < 3; p++) {
            Range rg;
            rg.first = (int)items.size();
            for (size_t k = b; k < e; k++) {
                const Size &z = by_size[longs[k].n];
                if (p == 2 && z.kind != K_THREE) continue;
                const MixPhase &ph = phases[z.phase + p];
                RagItem it{};
                it.phase = z.phase + p;
                it.n = longs[k].n;
                it.pow2 = is_pow2(it.n) ? 1 : 0;
                it.src = p == 0 ? offs[longs[k].id] : at[k - b];
                it.dst = (p == 2 || (p == 1 && z.kind == K_TWO)) ? offs[longs[k].id] : at[k - b];
                it.in_place = p == 1 && z.kind == K_THREE ? 1 : 0;
                for (int c = 0; c < ph.lines; c += ph.pl.G) {
                    it.c0 = c;
                    it.cnt = std::min(ph.pl.G, ph.lines - c);
                    items.push_back(it);
                }
            }
            rg.count = (int)items.size() - rg.first;
            r->tiles.push_back(rg);
        }
        b = e;
    }
    // short transforms, longest groups first
    std::vector<long long> goffs;
    for (int c = 0; c < kClasses; c++)
        for (int bl = 0; bl < 2; bl++) {
            Range &g = r->groups[c][bl];
            g.first = (int)items.size();
            for (auto &kv : by_size) {
                const Size &z = kv.second;
                if (z.kind != (bl ? K_GROUP_BLUE : K_GROUP) || z.cls != c) continue;
                const int per = phases[z.phase].pl.G;
                for (size_t k = 0; k < z.ids.size();) {
                    RagItem it{};
                    it.phase = z.phase;
                    it.n = kv.first;
                    it.pow2 = is_pow2(it.n) ? 1 : 0;
                    it.first = (int)goffs.size();
                    const long long base = offs[z.ids[k]];
                    // ids rise, so the first offset is the lowest; the others
                    // are addressed from it by 32-bit byte offsets
                    while (it.cnt < per && k < z.ids.size() &&
                           (offs[z.ids[k]] - base + kv.first) * (long long)cb < 0xf0000000LL) {
                        goffs.push_back(offs[z.ids[k++]]);
                        it.cnt++;
                    }
                    items.push_back(it);
                }
            }
            g.count = (int)items.size() - g.first;
            std::stable_sort(items.begin() + g.first, items.end(),
                             [](const RagItem &a, const RagItem &b) { return (long long)a.n * a.cnt > (long long)b.n * b.cnt; });
        }
    if (goffs.empty()) goffs.push_back(0);
    int dev = 0, ncu = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    const std::string key = tune_key(prec, std::vector<int>(sizes, sizes + count));
    // a workgroup per tile, or, by a record or the autotuner, a resident grid
    const auto grid_of = [&](int form) { return form > 1 ? ncu * form : 0; };
    const int record = tune_lookup(key);
    const bool recorded = record > 0;
    r->tile_grid = grid_of(record);
    const bool ok = dev_malloc(&r->d_items, items.size() * sizeof(RagItem)) == hipSuccess &&
                    dev_malloc(&r->d_offs, goffs.size() * sizeof(long long)) == hipSuccess &&
                    dev_malloc(&r->d_phases, phases.size() * sizeof(MixPhase)) == hipSuccess &&
                    (scratch == 0 || dev_malloc(&r->scratch, (size_t)scratch * cb) == hipSuccess) &&
                    hipMemcpy(r->d_items, items.data(), items.size() * sizeof(RagItem), hipMemcpyHostToDevice) == hipSuccess &&
                    hipMemcpy(r->d_offs, goffs.data(), goffs.size() * sizeof(long long), hipMemcpyHostToDevice) == hipSuccess &&
                    hipMemcpy(r->d_phases, phases.data(), phases.size() * sizeof(MixPhase), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) return fail("ragged setup: device allocation or copy failed");
    if ((flags & 1) && !recorded) {
        // project-written autotuner: time the batch as it is and with a few
        // resident grids, at most what the kernel's registers keep resident, on
        // scratch data and keep the fastest (the batch as it is where anything fails)
        void *tin = nullptr, *tout = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        bool timed = dev_malloc(&tin, (size_t)r->total * cb) == hipSuccess &&
                     dev_malloc(&tout, (size_t)r->total * cb) == hipSuccess && hipEventCreate(&e0) == hipSuccess &&
                     hipEventCreate(&e1) == hipSuccess &&
                     launch_fill_uniform(tin, 2 * r->total, 7, 0, prec, r->cap) == hipSuccess;
        float best = 1e30f;
        int form = 1;
        for (int f = 1; f <= (prec == F32 ? 4 : 2) && timed; f++) {
            r->tile_grid = grid_of(f);
            float ms = 0;
            timed = launch_ragged(r, 0, tin, tout, r->cap) == NFFT_OK && hipEventRecord(e0, r->cap) == hipSuccess;
            for (int k = 0; k < 3 && timed; k++) timed = launch_ragged(r, 0, tin, tout, r->cap) == NFFT_OK;
            timed = timed && hipEventRecord(e1, r->cap) == hipSuccess && hipEventSynchronize(e1) == hipSuccess &&
                    hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
            if (timed && ms < best) {
                best = ms;
                form = f;
            }
        }
        r->tile_grid = grid_of(timed ? form : 1);
        if (timed) tune_store(key, form);
        else (void)hipGetLastError();
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (tin) (void)hipFree(tin);
        if (tout) (void)hipFree(tout);
    }
    *out = r;
    return NFFT_OK;
}

// Project-written autotuner for the tile size and the scratch budget: builds
// the batch with each candidate (16 points per thread and the default budget,
// half and twice either), times four launches of each on scratch data and
// keeps the fastest ("ragged-gl" record).
static int ragged_tune_shape(int prec, int count, const int *sizes, const std::string &key, RagShape *best)
{
    const size_t cb = cx_bytes(prec);
    long long total = 0;
    for (int i = 0; i < count; i++) total += sizes[i];
    void *tin = nullptr, *tout = nullptr;
    if (dev_malloc(&tin, (size_t)total * cb) != hipSuccess || dev_malloc(&tout, (size_t)total * cb) != hipSuccess) {
        if (tin) (void)hipFree(tin);
        return NFFT_E_ALLOC;
    }
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    bool ok = hipStreamCreateWithFlags(&st, hipStreamNonBlocking) == hipSuccess && hipEventCreate(&e0) == hipSuccess &&
              hipEventCreate(&e1) == hipSuccess && launch_fill_uniform(tin, 2 * total, 7, 0, prec, st) == hipSuccess;
    float best_ms = 1e30f;
    int fail = NFFT_E_HIP;
    const RagShape cands[] = {{16, 4}, {8, 4}, {32, 4}, {16, 2}, {16, 8}};
    for (const RagShape &c : cands) {
        if (!ok) break;
        t_rag_shape = c;
        nfft_ragged *r = nullptr;
        const int rc = ragged_create_impl(&r, prec, count, sizes, 0);
        t_rag_shape = RagShape{};
        if (rc != NFFT_OK) {
            if (rc == NFFT_E_ALLOC) continue;  // this shape's scratch did not fit
            fail = rc;
            ok = false;
            break;
        }
        float ms = 0;
        ok = launch_ragged(r, 0, tin, tout, st) == NFFT_OK && hipEventRecord(e0, st) == hipSuccess;
        for (int k = 0; k < 4 && ok; k++) ok = launch_ragged(r, 0, tin, tout, st) == NFFT_OK;
        ok = ok && hipEventRecord(e1, st) == hipSuccess && hipEventSynchronize(e1) == hipSuccess &&
             hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
        ragged_free(r);
        if (ok && ms < best_ms) {
            best_ms = ms;
            *best = c;
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
    (void)hipFree(tin);
    (void)hipFree(tout);
    if (!ok || best_ms >= 1e30f) {
        (void)hipGetLastError();
        return fail;
    }
    tune_store(key, best->gpt * 100 + best->lag4);
    return NFFT_OK;
}

extern "C" {

int nfft_ragged_create(nfft_ragged **out, int prec, int count, const int *sizes, int flags)
{
    clear_error();
    if (!out || count < 1 || !sizes || (prec != NFFT_F32 && prec != NFFT_F64))
        return ragged_create_impl(out, prec, count, sizes, flags);  // reports the argument error
    // tile size and budget: a tuning record, else measured with flags bit 0
    RagShape shape;
    const std::string key = "ragged-gl" + tune_key(prec, std::vector<int>(sizes, sizes + count)).substr(6);
    const int rec = tune_lookup(key);
    if (rec > 0) {
        shape.gpt = rec / 100;
        shape.lag4 = rec % 100;
    } else if (flags & 1) {
        // the sizes are validated by the first candidate build
        const int rc = ragged_tune_shape(prec, count, sizes, key, &shape);
        if (rc == NFFT_E_SIZE || rc == NFFT_E_UNSUPPORTED || rc == NFFT_E_INVALID) return rc;
        if (rc != NFFT_OK) shape = RagShape{};  // nothing measured: the defaults
        clear_error();
    }
    t_rag_shape = shape;
    const int rc = ragged_create_impl(out, prec, count, sizes, flags);
    t_rag_shape = RagShape{};
    return rc;
}

int nfft_ragged_execute(nfft_ragged *r, int inverse, const void *in, void *out, void *stream)
{
    clear_error();
    if (!r || !in || !out) {
        set_error("NULL ragged handle or buffer");
        return NFFT_E_INVALID;
    }
    GraphKey k{in, out, inverse ? 1 : 0};
    auto it = r->graphs.find(k);
    if (it == r->graphs.end()) {
        if (r->graphs.size() >= 8) {
            (void)hipGraphExecDestroy(r->graphs.begin()->second.second);
            (void)hipGraphDestroy(r->graphs.begin()->second.first);
            r->graphs.erase(r->graphs.begin());
        }
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        if (hipStreamBeginCapture(r->cap, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            set_error("graph capture failed to start");
            return NFFT_E_HIP;
        }
        const int st = launch_ragged(r, k.inv, in, out, r->cap);
        if (hipStreamEndCapture(r->cap, &g) != hipSuccess || st != NFFT_OK ||
            hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            set_error("graph capture of the ragged launch failed");
            return NFFT_E_HIP;
        }
        it = r->graphs.emplace(k, std::make_pair(g, ge)).first;
    }
    if (hipGraphLaunch(it->second.second, (hipStream_t)stream) != hipSuccess) {
        set_error("graph launch failed");
        return NFFT_E_HIP;
    }
    return NFFT_OK;
}

int nfft_ragged_destroy(nfft_ragged *r)
{
    if (r) ragged_free(r);
    return NFFT_OK;
}

long long nfft_ragged_total(const nfft_ragged *r) { return r ? r->total : 0; }

int nfft_ragged_check(nfft_ragged *r, void *stream)
{
    clear_error();
    if (!r) {
        set_error("NULL ragged handle");
        return NFFT_E_INVALID;
    }
    if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) {
        set_error("hipStreamSynchronize failed");
        return NFFT_E_HIP;
    }
    return NFFT_OK;
}

}  // extern "C"
