// muca_team.hip -- the team update kernel's launch side: LDS layout,
// dispatch over the instantiations (compiled in muca_team_r{7,10}_{f32,f64}.hip
// so that the build can run them in parallel), and the
// batched engine's persistent team-tile kernel.
#include "team_run.h"

namespace muca {

#define MUCA_TEAM_EXTERN(R, FP64, KEYING)                                                \
    extern template hipError_t launch_team_r<R, FP64, KEYING>(hipStream_t, const McsArgs &, \
                                                              const TeamLayout &);
MUCA_TEAM_EXTERN(7, false, 0)
MUCA_TEAM_EXTERN(7, false, 1)
MUCA_TEAM_EXTERN(7, true, 0)
MUCA_TEAM_EXTERN(7, true, 1)
MUCA_TEAM_EXTERN(10, false, 0)
MUCA_TEAM_EXTERN(10, false, 1)
MUCA_TEAM_EXTERN(10, true, 0)
MUCA_TEAM_EXTERN(10, true, 1)
#undef MUCA_TEAM_EXTERN

// windows: ln W read from HBM and lattices left there whether or not they fit
static bool place(const McsArgs &a, int fp64, size_t lds_max, bool windows, TeamLayout &lay)
{
    if (a.L < 8 || a.L > 256) return false;
    const size_t row = (a.L + 1) / 2;   // the longest chunk
    auto al = [](size_t x) { return (x + 15) & ~(size_t)15; };
    lay.row = (uint32_t)row;
    // Philox ring: a chunk of a half-row (at most 64 attempts, starting at any
    // of a block's four words) touches (chunk + 6) / 4 blocks per key at most
    // and a generation pass may run up to 7 blocks ahead of them; then the
    // team's ln W window
    lay.ring = (uint32_t)(((row < 64 ? row : 64) + 6) / 4 + 8);
    lay.off_win = (uint32_t)al(2 * (size_t)lay.ring * 16);
    // per-D moments (produce path, FP64): the team's window of moment slots;
    // they replace the D histogram
    const bool moms = fp64 && a.moms != nullptr && a.joint == nullptr;
    const size_t mbytes = moms ? kMomLdsWords * kMomSlots * sizeof(uint64_t) : 0;
    const size_t fixed = 256 * sizeof(double) + 16;   // the acceptance-log table, FP64 bounds
    // ln W (FP64: its differences in FP32) in LDS when it fits (with the
    // guards), else read from HBM, where it stays in L2 (512 KB at L = 256 in
    // FP64), one window per team at a time.  FP64 differences would fit to
    // L = 192, but one workgroup per compute unit then does less than four
    // whose windows come from L2.
    const size_t wbytes = al((a.N + 1 + 2 * kGuard) * sizeof(float));
    lay.lnw_global =
        windows || al((lay.off_win + mbytes) * kTeams) + fixed + wbytes * (fp64 ? 2 : 1) > lds_max;
    lay.off_mom = (uint32_t)(lay.off_win + (lay.lnw_global ? al(kWinCache * sizeof(float)) : 0));
    lay.team_bytes = (uint32_t)(lay.off_mom + mbytes);
    size_t off = 0;
    lay.off_team = 0;
    off += al((size_t)lay.team_bytes * kTeams);
    lay.off_tab = (uint32_t)off;
    off += fixed;
    lay.off_w = (uint32_t)off;
    if (!lay.lnw_global) off += wbytes;
    // histogram and lattice in LDS when they fit (histogram first)
    const bool hist_fits = !moms && off + al((a.N + 1) * 4) <= lds_max;
    lay.lds_hist = hist_fits;
    lay.off_hist = (uint32_t)off;
    if (hist_fits) off += al((a.N + 1) * 4);
    lay.off_lat = (uint32_t)off;
    // walker-major lattices: the lanes of a team read sites two bytes apart
    // (one dword per two lanes); a per-walker stride of 8 (mod 32) dwords puts
    // the four teams of a wavefront on disjoint LDS banks.
    uint32_t stride = (uint32_t)((a.N + 3) & ~3u);
    while ((stride / 4) % 32 != 8) stride += 4;
    lay.lat_stride = stride;
    lay.lat_lds = !windows && off + al((size_t)stride * kTeams) <= lds_max;
    if (lay.lat_lds) off += al((size_t)stride * kTeams);
    lay.bytes = off;
    // Where the last round of a half-row would be at most half full, chunks of
    // whole rounds run on into the next row (lattices in LDS: those in HBM are
    // read a chunk ahead, row by row).
    const uint32_t hw = a.L / 2, rem = hw % 16;   // attempts from a site to its upper neighbour
    const bool flow = lay.lat_lds && hw >= 16 && rem <= 8 && (rem != 0 || a.L % 2);
    lay.order = a.L % 2 ? 1 : flow ? 2 : 0;
    const uint32_t nr = flow ? hw / 16 : (uint32_t)(row + 15) / 16;
    const uint32_t cap = lay.lnw_global ? (uint32_t)kLnwgRounds : 4u;
    lay.rounds = nr < cap ? nr : cap;
    if (a.L % 2 && !lay.lat_lds) return false;   // odd L: lattices in LDS only
    // lattices in HBM are addressed by a 32-bit offset within a row
    if (!lay.lat_lds && (uint64_t)a.L * a.W > 0xffffffffull) return false;
    return off <= lds_max;
}

bool team_layout(const McsArgs &a, int fp64, size_t lds_max, uint32_t cus, TeamLayout &lay)
{
    if (!place(a, fp64, lds_max, false, lay)) return false;
    // Per-D moments need no histogram, so with windows of ln W from HBM four
    // workgroups share a compute unit (128 VGPRs).  That leads as soon as there
    // are more walkers than the LDS layout keeps resident (attempts/ns on 256
    // compute units; L = 128:
    // 8192 walkers 55 -> 80, 65 536 54 -> 97; 4096 55 against 49; L = 72: 16 384
    // 57 -> 76; L = 96, two workgroups per compute unit: 16 384 82 -> 90, 8192
    // 78 against 75), but not where two workgroups with their lattices fit
    // (L = 48, 16 384: 89 against 80).  Odd L need their lattices in LDS.
    const uint64_t per_cu = lds_max / lay.bytes;
    const bool moms = fp64 && a.moms != nullptr && a.joint == nullptr;
    TeamLayout win;
    if (moms && a.L % 2 == 0 && !lay.lnw_global &&
        (per_cu == 1 || (!lay.lat_lds && per_cu < 4)) && a.W > (uint64_t)kTeams * cus * per_cu &&
        place(a, fp64, lds_max, true, win))
        lay = win;
    return true;
}

hipError_t launch_mcs_team(hipStream_t st, const Launch &cfg, const McsArgs &a,
                           const TeamLayout &lay)
{
    if (cfg.rounds == 10) {
        if (cfg.fp64)
            return cfg.keying ? launch_team_r<10, true, 1>(st, a, lay)
                              : launch_team_r<10, true, 0>(st, a, lay);
        return cfg.keying ? launch_team_r<10, false, 1>(st, a, lay)
                          : launch_team_r<10, false, 0>(st, a, lay);
    }
    if (cfg.fp64)
        return cfg.keying ? launch_team_r<7, true, 1>(st, a, lay)
                          : launch_team_r<7, true, 0>(st, a, lay);
    return cfg.keying ? launch_team_r<7, false, 1>(st, a, lay)
                      : launch_team_r<7, false, 0>(st, a, lay);
}

// ---------------------------------------------------------------------------
// batched engine, team tiles: a persistent grid (one workgroup per compute
// unit; each keeps ~100 KB of LDS) takes tiles of sixteen walkers from the
// per-XCD tile queues, largest lattices first, and runs one weight iteration
// of the tile's instance.  Converged instances are skipped.  Weight keying,
// Philox4x32-7, walker ids 0..W-1 within each instance, seed = instance seed.
// ---------------------------------------------------------------------------
// LM: the lattice placements this build of the kernel handles (1: LDS,
// 2: HBM, 3: both); NRS: the rounds per chunk of every instance (0: any), 8
// more where chunks run on from row to row.
// A batch of one placement (and one chunk size) launches the build for it
// alone, whose registers and schedule the other variants' code does not
// constrain.
template <bool FP64, int LM, int NRS>
__global__ __launch_bounds__(256) void k_batch_team(BatchArgs b)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ uint32_t s_tile;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_tile = batch_take(b);
        __syncthreads();
        const uint32_t t = s_tile;
        if (t >= b.ntiles) break;
        const BatchTile tile = b.tiles[t];
        const BatchInst *I = b.inst + tile.inst;
        if (I->converged) continue;
        const McsArgs a = batch_mcs_args(b, *I);
        const TeamLayout lay = I->lay;
        auto run = [&](auto nr, auto ord) {
            constexpr int NR = decltype(nr)::value, ORD = decltype(ord)::value;
            if (lay.lat_lds) {
                if constexpr ((LM & 1) != 0) {
                    if (lay.lds_hist)
                        team_run<7, FP64, 0, true, true, 0, false, NR, ORD>(a, lay, tile.wbase, lds);
                    else
                        team_run<7, FP64, 0, true, false, 0, false, NR, ORD>(a, lay, tile.wbase, lds);
                }
            } else if constexpr ((LM & 2) != 0 && ORD == 0) {
                if (lay.lds_hist)
                    team_run<7, FP64, 0, false, true, 0, false, NR, ORD>(a, lay, tile.wbase, lds);
                else
                    team_run<7, FP64, 0, false, false, 0, false, NR, ORD>(a, lay, tile.wbase, lds);
            }
        };
        std::integral_constant<int, 0> rows;
        std::integral_constant<int, 2> flow;
        if constexpr (NRS > 8) {
            run(std::integral_constant<int, NRS - 8>{}, flow);
        } else if constexpr (NRS != 0) {
            run(std::integral_constant<int, NRS>{}, rows);
        } else if (lay.order == 2) {
            if (lay.rounds == 1)
                run(std::integral_constant<int, 1>{}, flow);
            else
                run(std::integral_constant<int, 2>{}, flow);
        } else {
            switch (lay.rounds) {
            case 1: run(std::integral_constant<int, 1>{}, rows); break;
            case 2: run(std::integral_constant<int, 2>{}, rows); break;
            case 3: run(std::integral_constant<int, 3>{}, rows); break;
            default: run(std::integral_constant<int, 4>{}, rows); break;
            }
        }
    }
}

template <bool FP64>
static void (*batch_team_kernel(int lat_modes, int nrs))(BatchArgs)
{
    if (lat_modes == 1) {
        switch (nrs) {
        case 1: return k_batch_team<FP64, 1, 1>;
        case 2: return k_batch_team<FP64, 1, 2>;
        case 3: return k_batch_team<FP64, 1, 3>;
        case 4: return k_batch_team<FP64, 1, 4>;
        case 9: return k_batch_team<FP64, 1, 9>;
        case 10: return k_batch_team<FP64, 1, 10>;
        default: return k_batch_team<FP64, 1, 0>;
        }
    }
    // lattices in HBM, chunks of four rounds (L = 98 to 128): 15.5 ms for 8 iterations
    // of L = 128, 4096 walkers, against 15.75 in the build for any
    if (lat_modes == 2 && nrs == 4) return k_batch_team<FP64, 2, 4>;
    return lat_modes == 2 ? k_batch_team<FP64, 2, 0> : k_batch_team<FP64, 3, 0>;
}

hipError_t launch_batch_team(hipStream_t st, int fp64, const BatchArgs &b, uint32_t grid,
                             size_t lds_bytes, int lat_modes, int nrs)
{
    void (*k)(BatchArgs) = fp64 ? batch_team_kernel<true>(lat_modes, nrs)
                                : batch_team_kernel<false>(lat_modes, nrs);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kTeams * kTeam), lds_bytes, st, b);
    return hipGetLastError();
}

const void *batch_team_function(int fp64)
{
    return (const void *)(fp64 ? batch_team_kernel<true>(3, 0) : batch_team_kernel<false>(3, 0));
}

hipError_t prepare_batch_team(int fp64, size_t lds_bytes, int lat_modes, int nrs)
{
    void (*k)(BatchArgs) = fp64 ? batch_team_kernel<true>(lat_modes, nrs)
                                : batch_team_kernel<false>(lat_modes, nrs);
    return hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds_bytes);
}

}  // namespace muca
