// nfft_kernels_team.h -- the whole FP64 four-step of a batch of 2^15- or
// 2^17-point transforms in one launch, the intermediate of a transform in one
// XCD's L2.
//
// A transform of N = N1 x N2 points is cut into TILES column tiles (LPB1
// adjacent columns, FFT of N1 points, inter-pass twiddle) and as many row
// tiles (LPB2 rows, FFT of N2 points, transposed store), 128 KiB each.  A
// workgroup takes a column tile, stores its result to the transform's slot,
// waits for the other TILES - 1 and runs the row tile of the same index: the
// workgroups that hold one transform work as a team, and the slot is read
// back within microseconds of being written, by the XCD that wrote it.
// k_four_xcd's two kinds of items off one queue need a lag of several
// transforms between them, and k_four_persist's intermediate always goes
// through the memory-side cache.
//
// Bound: the fabric, and the wait for the team.  2^26 points, against the
// path it replaces: N = 2^15 (TILES 4, six slots of 512 KiB per XCD) 690 ->
// 495 us (persistent four-step), 2^17 (TILES 16, two slots of 2 MiB) 770 ->
// 680 us (two launches).  All the slots' reads hit the L2; where the slots in
// use exceed about 3 MiB of its 4 MiB, every intermediate point is also
// written back (2^15: nine slots 688 us; with three the teams wait for each
// other, 678).  N = 2^16 (TILES 8) gains
// nothing (694 against 693 us): its four teams need four slots of 1 MiB.  Nor
// do the FP32 lengths 2^16 .. 2^18 (742 / 858 / 1025 us against 742 / 770 /
// 774 of the two launches): the FFTs of a tile take as long as its transfers,
// and one workgroup a CU runs them one after the other.  Tiles of 64 KiB, two
// workgroups a CU, have twice the team: 2^15 576, 2^16 708, 2^17 810 us.
//
// Tickets.  A workgroup takes tickets from the queue of the XCD that it runs
// on (XCC_ID, as k_four_xcd).  Queue q owns transforms q, q + nq, ... (its
// step s is transform s nq + q), ticket i is column tile i % TILES of step
// i / TILES.  A workgroup takes its next ticket before it waits for its
// current step; if that is of the same step, it runs that column tile first
// and owes its row tile too.  So when it waits, every ticket of the step has
// been taken, by workgroups that run their column tile without waiting for
// anything but earlier steps (the slot's previous user): the earliest
// unfinished step always proceeds, however many workgroups are resident.
// Waits are bounded by wall-clock time and raise an error flag that the host
// reads back; the last workgroup to leave checks that every tile was done.
//
// Within an XCD the L2 is the coherence point: plain stores, waited for
// before the step is counted, and agent-scope (sc1) loads, which pass by the
// reading CU's L1.  The next column tile's loads are issued before the wait
// for the team (after the row tile's loads: 2^15 610 us, 2^17 756).
#pragma once
#include "nfft_kernels_xcd.h"

namespace nfft {

template <typename T_, int N1_, int N2_, int LPB1_, int LPB2_> struct TeamShape {
    using T = T_;
    static constexpr int N1 = N1_, N2 = N2_, LPB1 = LPB1_, LPB2 = LPB2_;
    static constexpr int NT1 = Sched<N1>::NT, NT2 = Sched<N2>::NT;
    static constexpr int BT = NT1 * LPB1;
    static constexpr int TILES = N2 / LPB1;
    static constexpr int L1 = N1 * LPB1, L2 = rowT_lds<T, N2, LPB2>();
    static constexpr int LDS = L1 > L2 ? L1 : L2;
    static constexpr int TWA = N1 == N2 ? 1 : stage_tw_lds<T, N1>();
    static constexpr int TWB = stage_tw_lds<T, N2>();
    static constexpr long long LDS_BYTES = (long long)(LDS + TWA + TWB) * (long long)sizeof(Cx<T>) + 64;
    static constexpr bool ok = NT2 * LPB2 == BT && N1 / LPB2 == TILES && TILES <= 64 && N2 % LPB1 == 0 &&
                               N1 % LPB2 == 0 && Sched<N1>::R == 16 && Sched<N2>::R == 16 &&
                               LDS_BYTES <= 160 * 1024;
};

struct TeamArgs {
    const void *in;
    void *out;
    long long ntrans;
    long long in_dist, out_dist;  // per-transform distances (elements)
    void *scratch;                // nq queues x slots x N elements
    int slots;                    // intermediate slots per queue
    unsigned *ctr;                // counter block (team_ctr_words)
    const void *tw_a, *tw_b;      // FP64 stage tables of N1 and N2
    Tw2 tw2;                      // FP64 two-level table of w_N^e
    double scale;
    long long timeout;            // wall-clock ticks one wait may take
    int nq;                       // queues in use (1..kXcdQueues)
    signed char qmap[kXcdIds];    // XCC_ID -> queue (-1: not expected)
};

// Counter block (32-bit words): [1] error flag of this launch, [2] sticky
// error, [4, 6) completion word (as k_four_xcd's); then lines of kTeamLine
// words, one each for the queue heads and, per queue and step, the column
// tiles stored and the row tiles loaded.  Counters that are polled while their
// neighbours are added to must not share a 128-byte line: with k_four_xcd's
// packed block, and its poll of the error flag beside the heads, two
// workgroups a CU took 1900 us where they take 610 (N = 2^15, 64 KiB tiles).
// (k_four_xcd, whose items are rarely waited for, is 1 % slower with lines of
// their own.)
constexpr int kTeamLine = 32;
__host__ __device__ constexpr long long team_ctr_words(long long ntrans, int nq)
{
    return kTeamLine * (1 + kXcdQueues + 2 * (long long)nq * xcd_steps(ntrans, nq));
}

// Bounded spin of one thread until *c >= need (false: gave up, error raised).
// The error flag, one line for every workgroup, is read once in 256 polls.
__device__ __forceinline__ bool team_wait(const unsigned *c, unsigned need, unsigned *err, long long timeout)
{
    const unsigned long long t0 = wall_clock64();
    for (unsigned i = 1; __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need; i++) {
        if (i % 256 == 0) {
            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
            if ((long long)(wall_clock64() - t0) > timeout) {
                atomicOr(err, 1u);
                return false;
            }
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

template <class Sh, int DIR> __global__ void __launch_bounds__(Sh::BT, Sh::BT / 256) k_four_team(TeamArgs a)
{
    using T = typename Sh::T;
    using C = Cx<T>;
    constexpr int N1 = Sh::N1, N2 = Sh::N2, LPB1 = Sh::LPB1, LPB2 = Sh::LPB2, BT = Sh::BT, TILES = Sh::TILES;
    constexpr int R = 16, NT1 = Sh::NT1, NT2 = Sh::NT2;
    constexpr long long N = (long long)N1 * N2;
    constexpr int CPS = 2;  // input loads and output stores: non-temporal
    static_assert(Sh::ok, "team four-step shape");
    __shared__ C lds[Sh::LDS];
    __shared__ C ltwb[Sh::TWB];
    __shared__ C ltwa[Sh::TWA];
    __shared__ int s_next[2];  // step, tile
    const int nq = a.nq;
    const long long SM = xcd_steps(a.ntrans, nq);
    unsigned *err = a.ctr + 1;
    const unsigned id = xcc_id();
    const int q = id < (unsigned)kXcdIds ? (int)a.qmap[id] : -1;
    const bool lead = __builtin_amdgcn_readfirstlane(threadIdx.x) == 0;  // wave 0
    const bool lane0 = threadIdx.x == 0;
    if (q < 0 || q >= nq) {  // an XCD the host did not see when it mapped the device
        if (lane0) atomicOr(err, 4u);
        return;
    }
    const int steps = q < a.ntrans ? (int)((a.ntrans - q + nq - 1) / nq) : 0;
    unsigned *head = a.ctr + kTeamLine * (1 + q);
    unsigned *const counts = a.ctr + kTeamLine * (1 + kXcdQueues + 2 * (long long)q * SM);
    auto stored = [&](int st) { return counts + 2 * kTeamLine * (long long)st; };
    auto loaded = [&](int st) { return counts + kTeamLine * (2 * (long long)st + 1); };
    stage_tw_to_lds<T, N2>(ltwb, (const double2 *)a.tw_b);
    if constexpr (N1 != N2) stage_tw_to_lds<T, N1>(ltwa, (const double2 *)a.tw_a);
    const C *twa = N1 == N2 ? ltwb : ltwa;
    const T sc = (T)a.scale;
    constexpr uint32_t cqst = (uint32_t)(NT1 * N2) * (uint32_t)sizeof(C);
    constexpr uint32_t rqst = (uint32_t)NT2 * (uint32_t)sizeof(C);
    int tid = threadIdx.x;  // made opaque in each iteration: no address is kept through the loop

    auto publish = [&](unsigned i) {
        s_next[0] = (int)(i / (unsigned)TILES);
        s_next[1] = (int)(i % (unsigned)TILES);
    };
    auto slot_of = [&](int s) { return (C *)a.scratch + ((long long)q * a.slots + s % a.slots) * N; };
    auto load_col = [&](C (&v)[R], int s, int r) {
        const int cb = tid % LPB1, cj = tid / LPB1;
        const uint32_t off = (uint32_t)(cj * N2 + cb) * (uint32_t)sizeof(C);
        const auto rs = buf_rsrc((const C *)a.in + ((long long)s * nq + q) * a.in_dist + r * LPB1);
#pragma unroll
        for (int i = 0; i < R; i++) v[i] = buf_ld<C, CPS>(rs, off, i * cqst);
    };

    if (lead && lane0) publish(__hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    __syncthreads();
    int s = __builtin_amdgcn_readfirstlane(s_next[0]);
    int r = __builtin_amdgcn_readfirstlane(s_next[1]);
    C reg[R], nxt[R];
    if (s < steps) load_col(reg, s, r);
    unsigned long long owed = 0;  // row tiles of step s that this workgroup runs
    unsigned ncol = 0, nrow = 0;
    // every iteration takes a ticket, and the queue holds steps * TILES
    for (long long left = (long long)steps * TILES; s < steps; left--) {
        if (left < 0) {
            if (lane0) atomicOr(err, 2u);
            break;
        }
        asm volatile("" : "+v"(tid));
        __syncthreads();  // s_next is read, the LDS free
        unsigned ticket = 0;
        if (lead && lane0) ticket = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        {
            const int cb = tid % LPB1, cj = tid / LPB1;
            const uint32_t off = (uint32_t)(cj * N2 + cb) * (uint32_t)sizeof(C);
            line_fft_tw<T, N1, DIR>(reg, lds, LayCol<LPB1>{cb}, cj, StageTwLds<T>{twa});
            const uint32_t c = (uint32_t)(r * LPB1 + cb);
            apply_tw2_series<DIR>(reg, a.tw2, c * (uint32_t)cj, c * (uint32_t)NT1);
            if (lead && lane0) {
                publish(ticket);
                // the slot's previous user has loaded it
                if (s >= a.slots) (void)team_wait(loaded(s - a.slots), TILES, err, a.timeout);
            }
            __syncthreads();
            const auto rd = buf_rsrc(slot_of(s) + r * LPB1);
#pragma unroll
            for (int i = 0; i < R; i++) buf_st<C>(rd, off, i * cqst, reg[i]);
        }
        const int ns = __builtin_amdgcn_readfirstlane(s_next[0]);
        const int nr = __builtin_amdgcn_readfirstlane(s_next[1]);
        // this wave's stores have reached the L2 before the barrier that
        // precedes the count
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (lead && lane0) __hip_atomic_fetch_add(stored(s), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        owed |= 1ull << r;
        ncol++;
        if (ns == s) {  // fewer workgroups than tiles: this step's next column tile
            load_col(reg, ns, nr);
            r = nr;
            continue;
        }
        if (ns < steps) load_col(nxt, ns, nr);
        if (lead && lane0) (void)team_wait(stored(s), TILES, err, a.timeout);
        __syncthreads();
        while (owed) {
            const int r0 = __builtin_ctzll(owed) * LPB2;
            owed &= owed - 1;
            const int rb = tid / NT2, rj = tid % NT2;
            {
                const auto rs = buf_rsrc(slot_of(s) + (long long)r0 * N2);
                const uint32_t off = (uint32_t)(rb * N2 + rj) * (uint32_t)sizeof(C);
#pragma unroll
                for (int i = 0; i < R; i++) reg[i] = buf_ld<C, kCpAgent>(rs, off, i * rqst);
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (lead && lane0) __hip_atomic_fetch_add(loaded(s), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            line_fft_tw<T, N2, DIR>(reg, lds, LayLine<T, N2>{rb * lpadlen<T, N2>()}, rj, StageTwLds<T>{ltwb});
#pragma unroll
            for (int i = 0; i < R; i++) {
                C v = reg[i];
                if (sc != (T)1) v = cscale(v, sc);
                lds[(rj + NT2 * i) * (LPB2 + 1) + rb] = v;
            }
            __syncthreads();
            constexpr int KS = BT / LPB2;  // output points k advanced per sweep of the transposed store
            const int bb = tid % LPB2, k0 = tid / LPB2;
            const uint32_t soff = (uint32_t)(k0 * N1 + bb) * (uint32_t)sizeof(C);
            constexpr uint32_t ist = (uint32_t)(KS * N1) * (uint32_t)sizeof(C);
            const auto rd = buf_rsrc((C *)a.out + ((long long)s * nq + q) * a.out_dist + r0);
#pragma unroll
            for (int i = 0; i < N2 / KS; i++)
                buf_st<C, CPS>(rd, soff, i * ist, lds[(k0 + KS * i) * (LPB2 + 1) + bb]);
            nrow++;
            if (owed) __syncthreads();  // the LDS is free for the next row tile
        }
#pragma unroll
        for (int i = 0; i < R; i++) reg[i] = nxt[i];
        s = ns;
        r = nr;
    }
    if (lane0) {
        const unsigned long long mine = 1ull | ((unsigned long long)ncol << 20) | ((unsigned long long)nrow << 42);
        const unsigned long long all = __hip_atomic_fetch_add((unsigned long long *)(a.ctr + 4), mine, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT) +
                                       mine;
        constexpr unsigned long long m20 = (1ull << 20) - 1, m22 = (1ull << 22) - 1;
        const unsigned long long want = (unsigned long long)a.ntrans * TILES;
        if ((all & m20) == gridDim.x && (((all >> 20) & m22) != want || ((all >> 42) & m22) != want))
            atomicOr(err, 8u);
    }
}

}  // namespace nfft
