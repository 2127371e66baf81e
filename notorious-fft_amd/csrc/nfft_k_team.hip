// nfft_k_team.hip -- instantiations and launcher of the team four-step
// (k_four_team).
#include "nfft_internal.h"
#include "nfft_kernels_team.h"

namespace nfft {

namespace {

template <class Sh> hipError_t team_go(int dir, const TeamArgs &a, int grid, hipStream_t s)
{
    if (dir < 0) hipLaunchKernelGGL((k_four_team<Sh, -1>), dim3(grid), dim3(Sh::BT), 0, s, a);
    else hipLaunchKernelGGL((k_four_team<Sh, 1>), dim3(grid), dim3(Sh::BT), 0, s, a);
    return hipGetLastError();
}

template <class Sh> int team_occ()
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_four_team<Sh, -1>, Sh::BT, 0) != hipSuccess) return 0;
    return nb;
}

struct Entry {
    int prec, n1, n2, tiles;
    hipError_t (*go)(int, const TeamArgs &, int, hipStream_t);
    int (*occ)();
};
template <class Sh> constexpr Entry entry(int prec)
{
    return Entry{prec, Sh::N1, Sh::N2, Sh::TILES, &team_go<Sh>, &team_occ<Sh>};
}

const Entry kTeams[] = {
    entry<TeamShape<double, 256, 128, 32, 64>>(F64),
    entry<TeamShape<double, 512, 256, 16, 32>>(F64),
};

}  // namespace

bool team_find(int prec, long long n, TeamCfg *cfg)
{
    for (const Entry &e : kTeams) {
        if (e.prec != prec || (long long)e.n1 * e.n2 != n) continue;
        *cfg = TeamCfg{(int)(&e - kTeams), e.n1, e.n2, e.tiles, e.occ()};
        return cfg->per_cu > 0;
    }
    return false;
}

hipError_t launch_four_team(const TeamCfg &c, int dir, const TeamArgs &a, int grid, hipStream_t s)
{
    const Entry &e = kTeams[c.id];
    const int slot = prof_on() ? prof_begin(s) : -1;
    const hipError_t err = e.go(dir, a, grid, s);
    if (slot >= 0)
        prof_end(slot, s, "k_four_team", e.prec, e.n1 * e.n2,
                 2.0 * (double)a.ntrans * e.n1 * e.n2 * (e.prec == F32 ? 8.0 : 16.0));
    return err;
}

}  // namespace nfft
