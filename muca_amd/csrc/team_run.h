// team_run.h -- the team update kernel: sixteen lanes (one DPP row) per
// walker, four walkers per wavefront, sixteen per workgroup.
//
// Why: a walker is a strict serial chain, so with few walkers (4096 walkers
// fill only 64 wavefronts) one-lane-per-walker leaves most SIMDs idle and
// every attempt waits on a chain of dependent memory loads.  The reference's
// even-L site order is column-parity stripes (muca_delta_multigpu.cu:173):
// a half-row of L/2 same-parity sites contains no two neighbours, and every
// neighbour of a half-row was last written by an earlier half-row.  So per
// chunk of a half-row (up to 64 attempts) the team
//   A. computes in parallel, attempt j on lane j % 16 of round j / 16: the
//      Philox blocks, the proposed spin, dE, dDel, -dE*beta and the screened
//      log of r1, for all rounds of the chunk at once;
//   B. resolves the D chain round by round: for each of a window of 8 D values
//      around the one the round starts at, whether the attempt accepts there
//      (one byte each; the exact test only where the screen is inconclusive).
//      An attempt is then a map of window positions, eight bytes wide;
//      v_perm_b32 looks four of them up at once, so sixteen lanes' maps compose
//      in a prefix scan of four DPP steps.  Where D leaves the window, the steps
//      after that are done again around the D reached;
//   C. writes the accepted spins, sums dE and dM and fills the histogram.
// Bound by one wavefront's issue and latency (a dependent VALU instruction
// takes 8.6 cycles, an independent one 5.2, a branch 21 to 37; L = 72: 22 % of
// the cycles in the Philox passes, 13 in A, 50 in B, 8 in C).  Measured against
// a serial chain of one DPP broadcast, bit extract and add per attempt over
// masks made once per chunk, one chunk per half-row: L = 72, 4096 walkers, from
// ln W = 0: 255 us per launch against 381; L = 128, seeded, NUPDATES = N: 1.86
// against 2.51 ms; L = 72 thermalization in FP64: 0.38 against 0.96 ms; L = 256,
// 16 384 walkers: 12.9 against 26.1 ms, with moments 14.2 against 19.5.  The
// scan alone, over masks per chunk, gave 341 us, 2.19, 0.63, 15.5 and 15.8 ms:
// D leaves a window of 8 around a chunk's start 0.2 to 1.3 times a round (L = 72
// from ln W = 0; seeded L = 128), one around the round's start 0.03 to 0.6 times.
// Every acceptance is decided by the reference's operations and rounding:
//   diff = ((T)(-dE*beta) + lnW[D+dDel]) - lnW[D];  accept iff diff >= 0 or
//   acclog(r1) < diff.  Because acclog(r1) < 0 always, that is exactly
//   acclog(r1) < diff.  Results are bit-identical to the one-lane kernel.
// Requires 8 <= L <= 256, and walkers whose D is their lattice's (D indexes LDS and
// HBM unchecked).  A half-row need not be a whole number of Philox
// blocks: a chunk starts at word rs % 4 of its first block.  Odd L (ODD, while
// the lattices fit in LDS): the reference's order visits the even linear
// indices 0, 2, .., N-3 twice and then N-2 (muca_delta_multigpu.cu:173).  Two
// of them are neighbours only across a wrap: x = 0 and L-1 of an even row, and
// rows 0 and L-1.  Chunks end at x = L-3 of an even row and at x = L-2 of an
// odd one, which separates both, or are no longer than the (L - 1) / 2 attempts
// that lie between such neighbours.
//
// LDS (dynamic): per team a ring of Philox blocks [2 keys][(min(L/2, 64) + 6)/4 + 8][4]
// and, where ln W stays in HBM, a window of it; the acceptance-log table; ln W
// (FP64: its differences) with guard entries on each side; the D histogram (u32,
// when it fits); the workgroup's lattices [N][16] int8 (when they fit).
#pragma once
#include "kernels.h"

#include "acclog.h"
#include "moments.h"
#include "philox.h"
#include "proposal.h"

namespace muca {

namespace team_detail {

constexpr int kTeam = 16;
constexpr int kTeams = 16;   // per workgroup of 256 lanes
constexpr uint32_t kXcds = 8;   // accelerator dies of an MI355X, one L2 each
// D values per window (at most 8).  Narrower ones cut the mask work per pass and
// make D leave them more often: L = 128, seeded 1.85 ms per launch against 1.90
// with 6 and 2.03 with 4; FP64 production, L = 256, 12.9 against 13.4 with 6
// (with moments 14.3 and 14.2), L = 72 0.43 against 0.46.
constexpr int kWin = 8;
// Rounds per chunk where ln W is in HBM: those launches have 128 VGPRs (four
// wavefronts per SIMD), which two rounds' state fits without spills.  L = 256,
// 16 384 walkers, 65 536 attempts each, with moments / without: 15.8 / 15.5 ms
// with two rounds, 16.8 / 16.1 with three, 18.5 / 16.0 with four.
constexpr int kLnwgRounds = 2;
// ln W values (FP64: differences) per team in LDS where ln W is in HBM: 64 are
// loaded again more often (L = 256, 16 384 walkers 13.3 ms against 12.9), 256
// cost more per load (with moments 15.7 against 14.2)
constexpr int kWinCache = 128;
constexpr int kGuard = 24;   // ln W guard entries on each side (> kWin / 2 + 2)

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int32_t team_sum(int32_t v)
{
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, kTeam);
    return v;
}

// the word of x that holds its sign bit (bit 31)
__device__ __forceinline__ uint32_t sign_word(float x)
{
    return __float_as_uint(x);
}

// the smaller of two, NaN where either is (v_minimum3_f32)
__device__ __forceinline__ float min_or_nan(float x, float y)
{
    return __builtin_elementwise_minimum(x, y);
}

// value of lane L of this lane's 16-lane row (v_mov_b32_dpp row_newbcast:L;
// every lane of the row reads a valid source, so no old value is needed)
template <int L>
__device__ __forceinline__ int32_t row_bcast(int32_t v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x150 + L, 0xf, 0xf, false);
}

// The proposal byte of an attempt: bits 0-1 hold dDel + 1, 2-4 the spin change
// + 2, 5-6 the new spin + 1 (the six cases of proposal_index)
__device__ __forceinline__ uint32_t proposal_byte(uint32_t at)
{
    return __builtin_amdgcn_perm(0x00240651u, 0x00014e2cu, at);
}
// fields of an attempt's info word: a proposal byte and (dE + 8) << 8
__device__ __forceinline__ int32_t i_ddel(int32_t i)
{
    return (i & 3) - 1;
}
__device__ __forceinline__ int32_t i_ds(int32_t i)
{
    return ((i >> 2) & 7) - 2;
}
__device__ __forceinline__ int32_t i_new(int32_t i)
{
    return ((i >> 5) & 3) - 1;
}
__device__ __forceinline__ int32_t i_dE(int32_t i)
{
    return (i >> 8) - 8;
}

// ---- maps of window positions, KW <= 8 positions as bytes 0..3 (lo), 4..7 (hi)

// byte k of (lo, hi) = 0xff iff bit 31 of sg[k] is set, k < KW; other bytes 0.
// v_perm_b32(a, b, sel): selector bytes 0x00-0x03 take b's bytes, 0x0b and
// 0x09 replicate the sign of a and of b, 0x0c is 0x00
template <int KW>
__device__ __forceinline__ void sign_bytes(const uint32_t *sg, uint32_t &lo, uint32_t &hi)
{
    auto four = [&](int k0, int n) -> uint32_t {
        uint32_t v = n > 1 ? __builtin_amdgcn_perm(sg[k0 + 1], sg[k0], 0x0c0c0b09u)
                           : __builtin_amdgcn_perm(sg[k0], sg[k0], 0x0c0c0c09u);
        if (n > 2) v = __builtin_amdgcn_perm(sg[k0 + 2], v, 0x0c0b0100u);
        if (n > 3) v = __builtin_amdgcn_perm(sg[k0 + 3], v, 0x0b020100u);
        return v;
    };
    lo = four(0, KW < 4 ? KW : 4);
    hi = KW > 4 ? four(4, KW - 4) : 0u;
}

// the identity: byte k = k for k < KW, else 0xff
template <int KW>
__device__ __forceinline__ constexpr uint32_t window_id(int word)
{
    uint32_t v = 0;
    for (int k = 0; k < 4; k++) {
        const int q = 4 * word + k;
        v |= (q < KW ? (uint32_t)q : 0xffu) << (8 * k);
    }
    return v;
}

// the map of one attempt: k + dDel where its accept byte k is set, else k;
// 0xff outside 0..KW-1.  dp1 = dDel + 1 in its low two bits: the moved
// positions are the four bytes from dp1 on of ff 00 01 .. KW-1 ff ff
template <int KW>
__device__ __forceinline__ void window_map(uint32_t alo, uint32_t ahi, uint32_t dp1, uint32_t &lo,
                                           uint32_t &hi)
{
    auto seq = [](int i) -> uint32_t { return i >= 1 && i <= KW ? (uint32_t)(i - 1) : 0xffu; };
    auto word = [&](int i) { return seq(i) | seq(i + 1) << 8 | seq(i + 2) << 16 | seq(i + 3) << 24; };
    const uint32_t s = dp1 & 3u;
    const uint32_t mlo = __builtin_amdgcn_alignbyte(word(4), word(0), s);
    lo = (alo & mlo) | (~alo & window_id<KW>(0));
    if (KW > 4) {
        const uint32_t mhi = __builtin_amdgcn_alignbyte(word(8), word(4), s);
        hi = (ahi & mhi) | (~ahi & window_id<KW>(1));
    } else {
        hi = 0xffffffffu;
    }
}

// byte `at` of (lo, hi), 0xff for at = 0xff
__device__ __forceinline__ uint32_t window_at(uint32_t lo, uint32_t hi, uint32_t at)
{
    return __builtin_amdgcn_perm(hi, lo, at | 0x0c0c0c00u);
}

// one level of the inclusive prefix scan: the map of the lane DPP points at
// (row_shr), then this lane's; q holds the identity where there is no such lane
template <int KW, int DPP>
__device__ __forceinline__ void scan_level(uint32_t &lo, uint32_t &hi, uint32_t &ql, uint32_t &qh)
{
    ql = (uint32_t)__builtin_amdgcn_update_dpp((int)ql, (int)lo, DPP, 0xf, 0xf, false);
    const uint32_t l = __builtin_amdgcn_perm(hi, lo, ql);
    if (KW > 4) {
        qh = (uint32_t)__builtin_amdgcn_update_dpp((int)qh, (int)hi, DPP, 0xf, 0xf, false);
        hi = __builtin_amdgcn_perm(hi, lo, qh);
    }
    lo = l;
}

}  // namespace team_detail
using namespace team_detail;

// NR: rounds of 16 attempts per chunk; a half-row of L / 2 attempts runs in
// chunks of up to 16 NR (NR <= 4 keeps the registers of all rounds' attempts
// low enough for more wavefronts per SIMD)
// OBS: 0 the D histogram; 1 joint H(D,M) per walker block (produce2_multigpu.cu:489);
// 2 exact per-D moments per walker block (the D histogram is then their S0).
// LNWG: ln W read from HBM (it does not fit in LDS), one window per team.
// One workgroup's sixteen walkers wbase .. wbase+15 of the launch described
// by a (all 256 lanes of the workgroup call it together).
template <int R, bool FP64, int KEYING, bool LATLDS, bool LDSHIST, int OBS, bool LNWG, int NR,
          int ORD = 0>
__device__ __forceinline__ void team_run(const McsArgs &a, const TeamLayout &lay, uint64_t wbase,
                                         unsigned char *lds)
{
    constexpr int KW = kWin;
    constexpr bool ODD = ORD == 1, FLOW = ORD == 2;
    constexpr bool JOINT = OBS == 1, MOMS = OBS == 2, TRACKM = OBS >= 1;
    __syncthreads();   // LDS may still be read by a previous call's flush
    // FP32: ln W.  FP64: ln W[D + 1] - ln W[D] in FP32, for the screening of
    // `pass`; its exact test reads ln W from HBM.  Valid for [-kGuard, N + kGuard]
    float *wt = (float *)(lds + lay.off_w) + kGuard;
    uint32_t *hist = (uint32_t *)(lds + lay.off_hist);
    int8_t *latl = (int8_t *)(lds + lay.off_lat);
    double *logtab = (double *)(lds + lay.off_tab);
    const int tid = threadIdx.x, team = tid >> 4, tl = tid & 15;
    const uint32_t N = a.N, L = a.L, Rw = lay.row;
    unsigned char *tbase = lds + lay.off_team + (size_t)team * lay.team_bytes;
    uint32_t *rng = (uint32_t *)tbase;                          // [2][ring][4]
    float *winb = (float *)(tbase + lay.off_win);               // LNWG: wt[wb .. wb + kWinCache - 1]
    // wt's value at any D from HBM (only positions a walker cannot be at read
    // one from outside [0, N]); FP64: `bound` grows to the error that the
    // screening has to allow for it, 2^-22 |value| for the FP32 arithmetic and
    // 2^-50 |ln W| for the rounding of the exact FP64 difference.  Where one bound
    // serves all D, walls around an excluded range must not set it (L = 64,
    // 32 768 walkers: 3.6 ms per launch with walls of 10^6 and of 10^300, 9.8 and
    // 12.1 ms when they did): a value of `plain` or more needs no allowance, since
    // with |thi| < 17 and |beta dE| <= 8 |beta| it decides the sign of e by 2^22
    // times its error, and a value between ln W whose rounding would need more than
    // 2^-16 is NaN, which `pass` takes to the exact test.  A window's own bound
    // (LNWG) needs neither, and the selects cost its loads 15 % (L = 256, 4096
    // walkers).
    const float plain = 2.0f * (8.0f * fabsf((float)a.beta) + 17.0f);
    auto lnw_at = [&](int32_t i, float &bound) -> float {
        const int32_t c = min(max(i, 0), (int32_t)a.N - (FP64 ? 1 : 0));
        if (!FP64) return a.lnw32[c];
        const double from = a.lnw64[c], to = a.lnw64[c + 1];
        const float g = (float)(to - from), size = (float)(fabs(from) + fabs(to));
        const bool screened = LNWG || size <= 0x1p34f;
        const float need = (LNWG || fabsf(g) < plain ? fabsf(g) * 0x1p-22f : 0.0f) + size * 0x1p-50f;
        bound = fmaxf(bound, screened ? need : 0.0f);
        return screened ? g : NAN;
    };
    float gbound = 0.0f;   // FP64: the largest bound of wt (LNWG: of the team's window)
    float *const wave_bound = (float *)(lds + lay.off_tab + 256 * sizeof(double));

    const uint64_t W = a.W;
    const uint64_t w = wbase + team;
    const bool active = w < W;

    if (!LNWG) {
#pragma unroll 4
        for (int i = (int)tid - kGuard; i <= (int)N + kGuard; i += blockDim.x)
            wt[i] = lnw_at(i, gbound);
        if (FP64) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) gbound = fmaxf(gbound, __shfl_xor(gbound, off));
            if ((tid & 63) == 0) wave_bound[tid >> 6] = gbound;
        }
    }
    // MOMS: this team's moment slots, word k of slot s at msl[k * kMomSlots + s]
    uint64_t *msl = (uint64_t *)(tbase + lay.off_mom);
    if (MOMS)
        for (int k = 0; k < kMomLdsWords; k++) msl[k * kMomSlots + tl] = 0;
    if (LDSHIST)
        for (uint32_t i = tid; i <= N; i += blockDim.x) hist[i] = a.hist_preload;
    acclog_table_to_lds(logtab, tid, blockDim.x);
    // LATLDS: the tile's lattices move between the site-major layout in HBM
    // and walker-major LDS rows.  For sixteen whole walkers on 16-byte
    // aligned rows, a lane moves four consecutive sites at a time: four
    // 16-byte global accesses (one per site: the tile's walkers), a 4x4 byte
    // transpose per four walkers, sixteen dword LDS accesses (one per
    // walker); a lane's four loads are all in flight before the first is
    // used.  Otherwise, and for the last N % 4 sites, lane tl of a team moves
    // walker tl's byte of every sixteenth site, four loads in flight (eight take the
    // kernel's small builds past 128 VGPRs).  L = 64, 10 007 walkers 0.58 ms per
    // launch against 0.83 one at a time; L = 16, 30 003 walkers 0.086 against 0.093.
    const bool lat_vec = LATLDS && W % kTeams == 0 && wbase + kTeams <= W &&
                         ((uintptr_t)a.lat & 15) == 0;
    if (LATLDS) {
        if (lat_vec) {
            for (uint32_t q = tid; q < N / 4; q += blockDim.x) {
                uint32_t s4[4][4];   // [site 4q+j][walkers 4c .. 4c+3]
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint4 v = *(const uint4 *)(a.lat + (uint64_t)(4 * q + j) * W + wbase);
                    s4[j][0] = v.x;
                    s4[j][1] = v.y;
                    s4[j][2] = v.z;
                    s4[j][3] = v.w;
                }
#pragma unroll
                for (int t = 0; t < kTeams; t++) {
                    const int c = t >> 2, sh = (t & 3) * 8;
                    *(uint32_t *)(latl + t * lay.lat_stride + 4 * q) =
                        ((s4[0][c] >> sh) & 0xffu) | (((s4[1][c] >> sh) & 0xffu) << 8) |
                        (((s4[2][c] >> sh) & 0xffu) << 16) | (((s4[3][c] >> sh) & 0xffu) << 24);
                }
            }
        }
        int t = tid;   // a copy of its own here and below, so that nothing made of it
        asm volatile("" : "+v"(t));   // stays in registers between the two
        const uint32_t wl = t & 15;
        const int8_t *const g = a.lat + wbase + (wbase + wl < W ? wl : 0);
        int8_t *const l = latl + wl * lay.lat_stride;
#pragma unroll 4
        for (uint32_t site = (lat_vec ? N & ~3u : 0u) + ((uint32_t)t >> 4); site < N; site += kTeams)
            l[site] = g[(uint64_t)site * W];
    }
    __syncthreads();
    if (FP64 && !LNWG)
        gbound = fmaxf(fmaxf(wave_bound[0], wave_bound[1]), fmaxf(wave_bound[2], wave_bound[3]));

    if (active) {
        // The walker's spin at x of a row: the row's address is the same in
        // every lane where lattices are in HBM (one 32-bit offset per lane and
        // x, site x W + w of a row; team_layout checks that it fits)
        const uint32_t xw = LATLDS ? 1u : (uint32_t)W;
        const uint32_t x0 = LATLDS ? team * lay.lat_stride : (uint32_t)w;
        auto row_at = [&](uint32_t yy) -> int8_t * {
            return LATLDS ? latl + yy * L : a.lat + (uint64_t)yy * ((uint64_t)L * W);
        };
        const uint32_t wid = a.w_offset + (uint32_t)w;
        const uint32_t k1a = KEYING == 0 ? 2u * wid : wid;
        const uint32_t k1b = 0xdecafbadu;
        const uint32_t k3a = KEYING == 0 ? 2u * wid + 50000u : wid + 40000u;
        const uint32_t k3b = KEYING == 0 ? 0x11cafeadu : 0xdecafeadu;
        int32_t d = a.D[w], e = a.E[w], m = a.M[w];
        // loaded before the loop, which would otherwise wait for them (and for
        // every load after them) where it uses d
        asm volatile("" : "+v"(d), "+v"(e), "+v"(m));
        uint64_t *jbase = nullptr;
        if (JOINT) jbase = a.joint + (w / a.block_walkers) * a.joint_stride;
        // MOMS: the walker's production attempts are summed per D in the
        // team's LDS slots for D = mwb .. mwb + kMomSlots - 1 (mwb the same in
        // every lane of the team) and added to the block's moments in HBM when
        // D leaves that window and at the end
        const uint64_t mstride = (uint64_t)N + 1;
        uint64_t *mbase = nullptr;
        if (MOMS) mbase = a.moms + (w / a.block_walkers) * (uint64_t)kMomWords * mstride;
        int32_t mwb = -(1 << 30);   // no window yet
        // lane tl moves slot tl (D = mwb + tl) to HBM and clears it
        auto flush_slot = [&]() {
            uint64_t v[kMomLdsWords];
#pragma unroll
            for (int k = 0; k < kMomLdsWords; k++) v[k] = msl[k * kMomSlots + tl];
            if (v[0]) {
                const uint64_t dd = (uint64_t)(mwb + (int32_t)tl);   // a visited D, in [0, N]
                atomicAdd((unsigned long long *)&mbase[dd], (unsigned long long)v[0]);
                atomicAdd((unsigned long long *)&mbase[mstride + dd], (unsigned long long)v[1]);
                atomic_add_limbs(&mbase[2 * mstride + dd], &mbase[3 * mstride + dd],
                                 &mbase[4 * mstride + dd], v[2], 0);
                // sum M^4 = v3 + v4 2^32 + v5 2^64 (limb sums) as a 128-bit value
                const uint64_t lo = v[3] + (v[4] << 32);
                const uint64_t hi = v[5] + (v[4] >> 32) + (lo < v[3] ? 1u : 0u);
                atomic_add_limbs(&mbase[5 * mstride + dd], &mbase[6 * mstride + dd],
                                 &mbase[7 * mstride + dd], lo, hi);
#pragma unroll
                for (int k = 0; k < kMomLdsWords; k++) msl[k * kMomSlots + tl] = 0;
            }
        };
        // FP64: the part of the screening's limit that is the same for all
        // attempts (|beta dE| <= 8 |beta|)
        const float limc = (8.0f * fabsf((float)a.beta) + 1.0f) * 0x1p-22f;
        uint32_t c0base = 0;
        const uint32_t RB = lay.ring;
        uint32_t gen = 0, gen_slot = 0, cur_slot = 0;   // next block to make, its slot, block blk0's slot
        // PF (lattices in HBM, ln W in LDS): the spins a chunk reads are
        // loaded while the chunk before it runs its D chain, so the loads'
        // latency is hidden.  pf_* hold, per round, the next chunk's site,
        // its right, left and upper neighbours and the lower neighbour as
        // read from memory; with pf_fwd the lower neighbour is instead this
        // lane's own site of the chunk before (same round and lane, the row
        // below), whose final spin fin[] phase C keeps (-9: none).
        constexpr bool PF = !LATLDS && !LNWG;
        int32_t pf_s[NR], pf_r[NR], pf_l[NR], pf_u[NR], pf_d[NR], fin[NR];
        bool pf_have = false, pf_fwd = false;
        int32_t de_lane = 0, dm_lane = 0;
        // wt[dc - KW/2 + k] at [k], k = -1 .. KW.  LNWG: from the team's
        // window of kWinCache values in LDS, staged again around dc when it
        // does not hold them
        int32_t wb = -(1 << 30);
        auto window = [&](int32_t dc) -> const float * {
            if (!LNWG) return wt + dc - KW / 2;
            if (dc - KW / 2 - 1 < wb || dc + KW / 2 >= wb + kWinCache) {
                wb = dc - kWinCache / 2;
                gbound = 0.0f;
#pragma unroll 4
                for (int i = 0; i < kWinCache / kTeam; i++)
                    winb[kTeam * i + tl] = lnw_at(wb + kTeam * i + (int32_t)tl, gbound);
                if (FP64)
#pragma unroll
                    for (int off = 8; off > 0; off >>= 1)
                        gbound = fmaxf(gbound, __shfl_xor(gbound, off, kTeam));
                wave_sync();
            }
            return winb + (dc - KW / 2 - wb);
        };
        // the scan's shifted-in maps per level: the lanes that have no source
        // lane at a level keep the identity from here on
        uint32_t ql[4], qh[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            ql[k] = window_id<KW>(0);
            qh[k] = window_id<KW>(1);
        }
        // this lane's sites in a row for a chunk of half h from jb on, and
        // their right and left neighbours; they stay from row to row
        uint32_t sx[NR], sxr[NR], sxl[NR], sx_h = ~0u, sx_jb = ~0u;
        auto sites = [&](uint32_t sh, uint32_t sj) {
            const uint32_t last = min(Rw - sj, 16u * NR) - 1;
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const uint32_t x = 2 * (sj + min(16u * r + tl, last)) + sh;
                sx[r] = x0 + x * xw;
                sxr[r] = x0 + ((x + 1 == L) ? 0 : x + 1) * xw;
                sxl[r] = x0 + ((x == 0) ? L - 1 : x - 1) * xw;
            }
            sx_h = sh;
            sx_jb = sj;
        };
        // a workgroup adds at most 16 NUPDATES counts to one u32 bin
        const bool may_wrap = a.hist_preload != 0 || (uint64_t)kTeams * a.nup >= (1ull << 32);
        for (int phase = 0; phase < 2; phase++) {
            const uint64_t n = phase ? a.nup : a.therm;
            // A half-row is worked in chunks of up to 16 NR attempts (no two
            // sites of a half-row are neighbours, so any split of it is exact).
            // FLOW: chunks of 16 NR <= Rw attempts run on into the next row
            // (the lower neighbour of an attempt is Rw attempts back, every
            // other one of its half further): half-rows of 16 k + 1 .. 16 k + 8
            // attempts would leave half or more of their last round idle.
            // L = 72, 4096 walkers: 74 -> 82 attempts/ns (FP64 67 -> 76), with
            // 36 = 32 + 4 attempts in a row; at 16 k + 10 and more the shorter
            // chunks cost more than the lanes (L = 60: 81 -> 75).
            // Attempt rs of a phase is at sweep position rs mod N: half h
            // (x parity), row y, place jb in the half-row -- advanced chunk by
            // chunk from 0, without divisions.
            uint32_t h = 0, y = 0, jb = 0;
            // ODD: the next site (ox, oy), its place ot in its pair of rows
            // (L sites: (L - 1) / 2, then the even row's last and the odd
            // row's), and op: first or second visit of the even indices, or N-2
            uint32_t ox = 0, oy = 0, ot = 0, op = 0;
            // (of two neighbouring sites visited in one pass over the even indices
            // the later one comes hw attempts after the other or more: with
            // 16 NR <= hw a chunk may run on over the ends of rows)
            const uint32_t hw = (L - 1) / 2;
            for (uint64_t rs = 0; rs < n;) {
                const uint32_t odd_left = hw >= 16u * NR ? (N - 1 - oy * L - ox) / 2
                                          : ot < hw      ? hw - ot
                                                         : L - ot;
                const uint32_t most = ODD    ? (op == 2 ? 1u : odd_left)
                                      : FLOW ? Rw
                                             : Rw - jb;
                const uint32_t cmax = min(most, 16u * NR);
                const uint32_t cnt = (uint32_t)min((uint64_t)cmax, n - rs);
                // ---- A1: the walker's Philox stream (block b uses counter b + 1;
                // the stream runs on across chunks and phases) is generated
                // eight blocks x two keys per pass into a ring of `RB` blocks per
                // key, so no lane idles when a chunk's block count is not a
                // multiple of eight.  Blocks [blk0, blk0 + nblk) serve this
                // chunk; a pass may run up to 7 blocks ahead, and RB >= nblk + 8
                // keeps those from overwriting blocks still in use.
                const uint32_t wo = (uint32_t)rs & 3u, nblk = (wo + cnt + 3) / 4;
                const uint32_t blk0 = c0base + (uint32_t)(rs / 4);
                while (gen < blk0 + nblk) {
                    const uint32_t b = gen + (uint32_t)(tl >> 1), key = tl & 1;
                    const philox4 r = philox4x32<R>(b + 1, a.seed, a.iter, 0xBADC0DEDu,
                                                    key ? k3a : k1a, key ? k3b : k1b);
                    uint32_t slot = gen_slot + (uint32_t)(tl >> 1);
                    slot = slot >= RB ? slot - RB : slot;
                    uint32_t *dst = rng + (key * RB + slot) * 4;
                    dst[0] = r.v[0];
                    dst[1] = r.v[1];
                    dst[2] = r.v[2];
                    dst[3] = r.v[3];
                    gen += 8;
                    gen_slot = gen_slot + 8 >= RB ? gen_slot + 8 - RB : gen_slot + 8;
                }
                // ring slot of this chunk's first block; the next chunk starts
                // in this one's last block unless that is used up or the
                // phase ends (a phase starts with a block of its own)
                const uint32_t slot0 = cur_slot;
                cur_slot += rs + cnt == n ? nblk : (wo + cnt) / 4;
                cur_slot = cur_slot >= RB ? cur_slot - RB : cur_slot;
                wave_sync();
                // ---- A2: attempt j = 16 r + tl on this lane, everything in registers
                int8_t *const row = ODD || FLOW ? latl : row_at(y);
                // ring word of attempt j: s4 + j (mod ringw)
                const uint32_t s4 = slot0 * 4 + wo, ringw = RB * 4;
                // the proposal byte and dE + 8
                // in bits 8..12
                int32_t info[NR];
                // Every load of the chunk's spins and random words first, then
                // the proposals, without a branch between the rounds: one
                // wavefront per SIMD hides no latency of its own.
                // A lane past the end of the chunk works on an in-bounds
                // attempt and keeps nothing of it.
                if (!ODD && !FLOW && (LNWG || h != sx_h || jb != sx_jb)) sites(h, jb);
                uint32_t cx[NR];   // this chunk's sites (sx may move on to the next one's)
#pragma unroll
                for (int r = 0; r < NR; r++) cx[r] = sx[r];
                int32_t old_s[NR], nb[NR];
                uint32_t r1[NR], r3[NR];
                float thi[NR];   // the screened log of r1 (acclog_screen)
                if (ODD) {
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        uint32_t x = ox + 2 * min(16u * r + tl, cmax - 1), yy = oy;
                        if (x >= L) {
                            x -= L;
                            yy++;
                        }
                        const uint32_t c = x0 + yy * L + x;
                        cx[r] = c;
                        old_s[r] = row[c];
                        nb[r] = row[x + 1 == L ? c + 1 - L : c + 1] +
                                row[x == 0 ? c + L - 1 : c - 1] +
                                row[yy + 1 == L ? c + L - N : c + L] +
                                row[yy == 0 ? c + N - L : c - L];
                    }
                } else if (FLOW) {
                    // row y from jb on, then the next row (of the next half
                    // after the last) from its start
                    const uint32_t y1 = y + 1 == L ? 0 : y + 1, h1 = y + 1 == L ? h ^ 1u : h;
                    const uint32_t c0 = x0 + y * L + h, c1 = x0 + y1 * L + h1 - L;
                    const uint32_t up0 = y + 1 == L ? L - N : L, up1 = y1 + 1 == L ? L - N : L;
                    const uint32_t dn0 = y == 0 ? N - L : 0u - L, dn1 = y1 == 0 ? N - L : 0u - L;
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const uint32_t j2 = 2 * (jb + min(16u * r + tl, cmax - 1));
                        const bool nxt = j2 >= L;
                        const uint32_t c = j2 + (nxt ? c1 : c0), x = j2 + (nxt ? h1 - L : h);
                        cx[r] = c;
                        old_s[r] = row[c];
                        nb[r] = row[x + 1 == L ? c + 1 - L : c + 1] +
                                row[x == 0 ? c + L - 1 : c - 1] + row[c + (nxt ? up1 : up0)] +
                                row[c + (nxt ? dn1 : dn0)];
                    }
                } else if (PF && pf_have) {
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        old_s[r] = pf_s[r];
                        nb[r] = pf_r[r] + pf_l[r] + pf_u[r] +
                                ((pf_fwd && fin[r] != -9) ? fin[r] : pf_d[r]);
                    }
                } else {
                    const int8_t *up = row_at((y + 1 == L) ? 0 : y + 1);
                    const int8_t *dn = row_at((y == 0) ? L - 1 : y - 1);
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        old_s[r] = row[sx[r]];
                        nb[r] = row[sxr[r]] + row[sxl[r]] + up[sx[r]] + dn[sx[r]];
                    }
                }
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    uint32_t widx = s4 + 16 * r + tl;
                    widx = widx >= ringw ? widx - ringw : widx;
                    r1[r] = rng[widx];
                    r3[r] = rng[ringw + widx];
                }
                // FP32: -beta dE; FP64: the screened log less it
                float fde[NR];
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const uint32_t at = proposal_index(old_s[r], r3[r]);
                    const uint32_t pr = proposal_byte(at);
                    const int32_t mds = proposal_mds(at);
                    thi[r] = acclog_screen(r1[r]);
                    const int32_t dE = __mul24(mds, nb[r]);
                    info[r] = (int32_t)pr | ((dE + 8) << 8);
                    // past the chunk's end: accepted nowhere
                    const float f = (float)(-(double)dE * a.beta);
                    const bool in = 16 * r + (uint32_t)tl < cnt;
                    fde[r] = FP64 ? (in ? thi[r] - f : INFINITY) : (in ? f : -INFINITY);
                    // made here, not where the round uses them: that would put
                    // their latency into the chain
                    asm volatile("" : "+v"(info[r]), "+v"(fde[r]), "+v"(thi[r]));
                }
                wave_sync();
                if (PF) {
                    // The next chunk (the next phase's first after a phase's
                    // last) and whether its spins may be read now: this chunk
                    // writes sites jb .. jb + cnt - 1 of half-row (y, h) only.
                    // Reads of that half-row are safe when their sites lie
                    // outside it; the lower neighbours of the next row's
                    // chunk at the same jb come from fin[] (lanes within this
                    // chunk) or from memory (lanes past it: not written).
                    uint64_t rs_n = rs + cnt, n_n = n;
                    bool nx = rs_n < n;
                    uint32_t h_n = h, y_n = y, jb_n = jb + cnt;
                    if (jb_n == Rw) {
                        jb_n = 0;
                        if (++y_n == L) {
                            y_n = 0;
                            h_n ^= 1u;
                        }
                    }
                    if (!nx && phase == 0 && a.nup > 0) {
                        rs_n = 0;
                        n_n = a.nup;
                        nx = true;
                        h_n = y_n = jb_n = 0;
                    }
                    const uint32_t cnt_n = (uint32_t)min((uint64_t)min(Rw - jb_n, 16u * NR), n_n - rs_n);
                    const uint32_t yu_n = (y_n + 1 == L) ? 0 : y_n + 1;
                    const uint32_t yd_n = (y_n == 0) ? L - 1 : y_n - 1;
                    const bool ovl = jb_n < jb + cnt && jb < jb_n + cnt_n;
                    bool have = nx;
                    bool fwd = false;
                    if (y_n == y && h_n != h) have = false;          // neighbours in the written half-row
                    if (h_n == h && (y_n == y || yu_n == y) && ovl) have = false;
                    if (h_n == h && yd_n == y && ovl) {
                        if (jb_n == jb) fwd = true;
                        else have = false;
                    }
                    pf_have = have;
                    pf_fwd = fwd;
                    if (have) {
                        if (h_n != sx_h || jb_n != sx_jb) sites(h_n, jb_n);
                        const int8_t *row_n = row_at(y_n), *up_n = row_at(yu_n),
                                     *dn_n = row_at(yd_n);
#pragma unroll
                        for (int r = 0; r < NR; r++) {
                            pf_s[r] = row_n[sx[r]];
                            pf_r[r] = row_n[sxr[r]];
                            pf_l[r] = row_n[sxl[r]];
                            pf_u[r] = up_n[sx[r]];
                            pf_d[r] = dn_n[sx[r]];
                        }
                    }
                }
                // ---- B: the D chain, round by round.  A window of KW values
                // of D around the one the round starts at, dlo .. dlo + KW - 1:
                // attempt j maps the window position k = D - dlo before it to
                // the one after it, k + dDel where it accepts at dlo + k and
                // else k; a position outside the window is 0xff and stays so.
                // A map is eight bytes, and v_perm_b32 looks up four of them
                // at once (a selector of 0xff gives 0xff), so that two maps
                // compose in two instructions and sixteen lanes' maps in a
                // prefix scan of four levels.
                const uint32_t sh = (uint32_t)(tid & 48);    // this team's 16 lanes of a ballot
                const uint32_t upto = (2u << tl) - 1u;       // steps 0..tl of a round
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const uint32_t j0 = 16 * r;
                    if (PF) fin[r] = -9;
                    if (j0 >= cnt) continue;
                    const bool valid = j0 + tl < cnt;
                    // The window around D = dc before step `from` of the round;
                    // the steps before it are identities (accepted nowhere).
                    // Byte k of (lo, hi): accept at dlo + k, i.e.
                    // acclog(r1) < ((fde + lnW[dlo + k + dDel]) - lnW[dlo + k]),
                    // screened: the sign of e = thi - diff (the difference of two
                    // infinite floats is a NaN whose sign is clear: rejected);
                    // |e| < lim, in FP64 also an e that is NaN, needs the exact
                    // test.  FP64 screens with FP32 differences of ln W
                    // (lim allows for them): one load and one fma per position
                    // and half the LDS, against two loads and three additions of
                    // doubles (L = 72, 4096 walkers: thermalization launch 432 ->
                    // 380 us, joint 728 -> 673; L = 256 waits for memory: the same).
                    // o: the window position after this lane's step; before:
                    // the one before it; ok: accepted there.
                    auto pass = [&](int32_t dc, uint32_t from, uint32_t &o, uint32_t &before,
                                    bool &ok) {
                        const float *wc = window(dc);
                        const int32_t dd = i_ddel(info[r]);
                        uint32_t sg[8], lo, hi;
                        float emin = 1e30f, diff[KW];
                        float lim = acclog_screen_lim(thi[r]);
                        if constexpr (FP64) {
                            // thi - diff = (thi + beta dE) -+ the step's difference
                            const float *wq = wc + min(dd, 0), step = -(float)dd;
                            const float base = (uint32_t)tl >= from ? fde[r] : INFINITY;
                            lim += (limc - thi[r] * 0x1p-22f) + gbound;
#pragma unroll
                            for (int k = 0; k < KW; k++) {
                                const float e = __builtin_fmaf(step, wq[k], base);
                                sg[k] = sign_word(e);
                                emin = min_or_nan(emin, fabsf(e));
                            }
                        } else {
                            const float *wto = wc + dd;
                            const float fd = (uint32_t)tl >= from ? fde[r] : -INFINITY;
#pragma unroll
                            for (int k = 0; k < KW; k++) {
                                diff[k] = fd + wto[k];
                                diff[k] = diff[k] - wc[k];
                            }
#pragma unroll
                            for (int k = 0; k < KW; k++) {
                                const float e = thi[r] - diff[k];
                                sg[k] = sign_word(e);
                                emin = fminf(emin, fabsf(e));
                            }
                        }
                        sign_bytes<KW>(sg, lo, hi);
                        const bool amb = !(emin >= lim);
                        if (__builtin_amdgcn_ballot_w64(amb)) {   // rare
                            if (amb) {
                                uint32_t w1 = s4 + j0 + tl;
                                w1 = w1 >= ringw ? w1 - ringw : w1;
                                const float tlog = (float)acclog_u01_double_tab(rng[w1], logtab,
                                                                                logtab + 128);
                                if constexpr (FP64) {
                                    const double f = -(double)i_dE(info[r]) * a.beta;
                                    const bool live = valid && (uint32_t)tl >= from;
                                    uint64_t bytes = 0;
#pragma unroll 1
                                    for (int k = 0; k < KW; k++) {
                                        const int32_t at = dc - KW / 2 + k;
                                        const double x = f + a.lnw64[min(max(at + dd, 0), (int32_t)N)];
                                        if (live &&
                                            (double)tlog < x - a.lnw64[min(max(at, 0), (int32_t)N)])
                                            bytes |= 0xffull << (8 * k);
                                    }
                                    lo = (uint32_t)bytes;
                                    hi = (uint32_t)(bytes >> 32);
                                } else {
#pragma unroll
                                    for (int k = 0; k < KW; k++)
                                        sg[k] = tlog < diff[k] ? 0x80000000u : 0u;
                                    sign_bytes<KW>(sg, lo, hi);
                                }
                            }
                        }
                        uint32_t plo, phi;   // the map of steps 0..tl
                        window_map<KW>(lo, hi, (uint32_t)info[r], plo, phi);
                        scan_level<KW, 0x111>(plo, phi, ql[0], qh[0]);
                        scan_level<KW, 0x112>(plo, phi, ql[1], qh[1]);
                        scan_level<KW, 0x114>(plo, phi, ql[2], qh[2]);
                        scan_level<KW, 0x118>(plo, phi, ql[3], qh[3]);
                        o = window_at(plo, phi, KW / 2);
                        before = (uint32_t)__builtin_amdgcn_update_dpp(KW / 2, (int)o, 0x111, 0xf,
                                                                       0xf, false);
                        ok = window_at(lo, hi, before) != 0;
                    };
                    uint32_t o, before;
                    bool acc;   // this lane's attempt: accepted, and D (and M) after it
                    pass(d, 0, o, before, acc);
                    int32_t dlo = d - KW / 2, dv = dlo + (int32_t)o, mv = 0;
                    // D left the window at step k: steps 0..k stand (step k is
                    // accepted and moved D by its dDel), and the window moves
                    // to D after it for the later ones, until the round is
                    // done.  k grows by KW / 2 at least each time.
                    uint64_t outs;
                    bool out = o == 0xffu;
                    while ((outs = __builtin_amdgcn_ballot_w64(out)) != 0) {
                        const uint32_t mine = (uint32_t)(outs >> sh) & 0xffffu;
                        if (mine) {
                            const uint32_t k = (uint32_t)__builtin_ctz(mine);
                            const int32_t dk = dlo + (int32_t)before + i_ddel(info[r]);
                            if ((uint32_t)tl == k) dv = dk;
                            const int32_t dc = __shfl(dk, (int)k, kTeam);
                            dlo = dc - KW / 2;
                            bool ok;
                            pass(dc, k + 1, o, before, ok);
                            out = o == 0xffu;
                            if ((uint32_t)tl > k) {
                                acc = ok;
                                dv = dlo + (int32_t)o;
                            }
                        }
                    }
                    d = row_bcast<15>(dv);
                    if (TRACKM) {
                        // M after this lane's step: an inclusive scan over the
                        // team of the accepted spin changes
                        int32_t x = acc ? i_ds(info[r]) : 0;
                        x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
                        mv = m + x;
                        m += row_bcast<15>(x);
                    }
                    // ---- C: accepted spins, dE / dM sums, histogram of the round
                    const uint32_t left = min(cnt - j0, 16u);
                    const int32_t ns = i_new(info[r]), ds = i_ds(info[r]);   // the proposal
                    // the site's spin after this chunk
                    if (PF) fin[r] = valid ? (acc ? ns : ns - ds) : -9;
                    if (acc) {
                        // the new spin is known from phase A: no site of
                        // the chunk is written between its read and here
                        row[cx[r]] = (int8_t)ns;
                        de_lane += i_dE(info[r]);
                        dm_lane += ds;
                    }
                    // Attempt j records the (D, M) after its step.  Steps that are
                    // not accepted keep the state, so a round splits into
                    // segments that start at step 0 and at every accepted step
                    // and share one (D, M); the first lane of each adds its
                    // length.
                    bool lead = false;
                    uint32_t slen = 0;
                    if (TRACKM && phase) {
                        const uint32_t ab =
                            (uint32_t)(__builtin_amdgcn_ballot_w64(acc) >> sh) & 0xffffu;
                        const uint32_t later = ab & ~upto;
                        lead = tl < left && (tl == 0 || acc);
                        slen = (later ? (uint32_t)__builtin_ctz(later) : left) - (uint32_t)tl;
                    }
                    if (JOINT && lead) {
                        const int64_t mm = min(max(mv, -dv), dv);
                        atomicAdd((unsigned long long *)&jbase[(mm + (int64_t)dv * (dv + 2)) >> 1],
                                  (unsigned long long)slen);
                    }
                    if (phase && !MOMS) {
                        // The D histogram: a round's steps split into runs at one D,
                        // starting at step 0 and at every accepted step that
                        // changed D; the first lane of a run adds its length (one
                        // atomic per run instead of sixteen on the same bin)
                        const bool moved = acc && i_ddel(info[r]) != 0;
                        const uint32_t starts =
                            ((uint32_t)(__builtin_amdgcn_ballot_w64(moved) >> sh) & 0xffffu) | 1u;
                        const uint32_t later = starts & ~upto;
                        const uint32_t len =
                            (later ? (uint32_t)__builtin_ctz(later) : left) - (uint32_t)tl;
                        if (tl < left && ((starts >> tl) & 1u)) {
                            const int32_t dd = dv;
                            if (LDSHIST) {
                                if (may_wrap) {
                                    // a u32 bin that wraps carries 2^32 into HBM
                                    if (atomicAdd(&hist[dd], len) > 0xFFFFFFFFu - len)
                                        atomicAdd((unsigned long long *)&a.hist[dd], 1ull << 32);
                                } else {
                                    atomicAdd(&hist[dd], len);
                                }
                            } else {
                                atomicAdd((unsigned long long *)&a.hist[dd], (unsigned long long)len);
                            }
                        }
                    }
                    if (MOMS && phase) {
                        // a segment adds len x (1, |M|, M^2, M^4) to the slot of its D
                        const uint32_t len = slen;
                        const int32_t dd = dv;
                        int32_t slot = dd - mwb;
                        const bool past = lead && (uint32_t)slot >= (uint32_t)kMomSlots;
                        const uint64_t ob = __builtin_amdgcn_ballot_w64(past);
                        if (ob) {
                            if ((ob >> sh) & 0xffffu) {   // the whole team: new window
                                flush_slot();
                                mwb = row_bcast<0>(dd) - kMomSlots / 2;
                                slot = dd - mwb;
                            }
                        }
                        if (lead) {
                            const int32_t mm = min(max(mv, -dd), dd);
                            const uint64_t am = (uint64_t)(mm < 0 ? -mm : mm);
                            const uint64_t m2 = am * am;
                            const uint64_t q = m2 * m2, qh = __umul64hi(m2, m2);   // M^4
                            const uint64_t pl = q * len, ph = qh * len + __umul64hi(q, len);
                            const uint64_t v[kMomLdsWords] = {len, len * am, len * m2,
                                                              pl & 0xFFFFFFFFull, pl >> 32, ph};
                            if ((uint32_t)slot < (uint32_t)kMomSlots) {
                                // no test for zero words: a branch per word
                                // costs more than the add
#pragma unroll
                                for (int k = 0; k < kMomLdsWords; k++)
                                    atomicAdd((unsigned long long *)&msl[k * kMomSlots + slot],
                                              (unsigned long long)v[k]);
                            } else {
                                // D moved more than kMomSlots / 2 within the round
                                atomicAdd((unsigned long long *)&mbase[dd], (unsigned long long)v[0]);
                                atomicAdd((unsigned long long *)&mbase[mstride + dd],
                                          (unsigned long long)v[1]);
                                atomic_add_limbs(&mbase[2 * mstride + dd], &mbase[3 * mstride + dd],
                                                 &mbase[4 * mstride + dd], v[2], 0);
                                atomic_add_limbs(&mbase[5 * mstride + dd], &mbase[6 * mstride + dd],
                                                 &mbase[7 * mstride + dd], pl, ph);
                            }
                        }
                    }
                }
                if (!LATLDS) __threadfence_block();
                wave_sync();
                rs += cnt;
                if (ODD) {
                    ox += 2 * cnt;
                    ot += cnt;
                    while (ox >= L) {
                        ox -= L;
                        oy++;
                    }
                    if (ot == L) ot = 0;
                    if (op == 2) {
                        ox = oy = ot = op = 0;
                    } else if (oy == L - 1 && ox == L - 1) {   // N-1 is not visited
                        ox = op == 0 ? 0 : L - 2;
                        oy = op == 0 ? 0 : L - 1;
                        ot = 0;
                        op++;
                    }
                } else {
                    jb += cnt;
                    if (jb >= Rw) {
                        jb -= Rw;
                        if (++y == L) {
                            y = 0;
                            h ^= 1u;
                        }
                    }
                }
            }
            c0base += (uint32_t)((n + 3) / 4);
        }
        if (MOMS) flush_slot();
        // dE and dM of accepted moves were summed per lane; one reduction
        // over the team's sixteen lanes per launch.  In joint mode the
        // chain itself tracks M (it is needed per attempt).
        e += team_sum(de_lane);
        const int32_t dm_team = team_sum(dm_lane);
        if (!TRACKM) m += dm_team;
        if (tl == 0) {
            a.D[w] = d;
            a.E[w] = e;
            a.M[w] = m;
        }
    }
    __syncthreads();
    if (LDSHIST) {
        // counts since the start (modulo 2^32; a wrap was carried already)
        for (uint32_t i = tid; i <= N; i += blockDim.x) {
            const uint32_t c = hist[i];
            if (c != a.hist_preload)
                atomicAdd((unsigned long long *)&a.hist[i],
                          (unsigned long long)((int64_t)c - (int64_t)a.hist_preload));
        }
    }
    if (LATLDS) {
        if (lat_vec) {
            for (uint32_t q = tid; q < N / 4; q += blockDim.x) {
                uint32_t r[kTeams];   // walker t's spins at sites 4q .. 4q+3
#pragma unroll
                for (int t = 0; t < kTeams; t++)
                    r[t] = *(const uint32_t *)(latl + t * lay.lat_stride + 4 * q);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int sh = 8 * j;
                    uint32_t d[4];
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        d[c] = ((r[4 * c] >> sh) & 0xffu) | (((r[4 * c + 1] >> sh) & 0xffu) << 8) |
                               (((r[4 * c + 2] >> sh) & 0xffu) << 16) |
                               (((r[4 * c + 3] >> sh) & 0xffu) << 24);
                    *(uint4 *)(a.lat + (uint64_t)(4 * q + j) * W + wbase) =
                        make_uint4(d[0], d[1], d[2], d[3]);
                }
            }
        }
        int t = tid;
        asm volatile("" : "+v"(t));
        const uint32_t wl = t & 15;
        if (wbase + wl < W) {
            int8_t *const g = a.lat + wbase + wl;
            const int8_t *const l = latl + wl * lay.lat_stride;
            for (uint32_t site = (lat_vec ? N & ~3u : 0u) + ((uint32_t)t >> 4); site < N; site += kTeams)
                g[(uint64_t)site * W] = l[site];
        }
    }
}

// LNWG launches are those of large lattices (FP64 from L = 138, with moments from
// 132; FP32 from 194) and, with moments, of more walkers than LDS keeps resident
// (from L = 54): they are held to 128 VGPRs, four wavefronts per SIMD
template <int R, bool FP64, int KEYING, bool LATLDS, bool LDSHIST, int OBS, bool LNWG, int NR,
          int ORD = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LNWG ? 4 : 1))) void
k_mcs_team(McsArgs a, TeamLayout lay)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    // Workgroups go to the eight XCDs round-robin, and eight consecutive
    // groups of 16 walkers share each 128-byte line of the site-major
    // lattice: workgroup b takes group (b mod 8) (G / 8) + b / 8, so that
    // XCD x runs the consecutive groups x G / 8 .. (x + 1) G / 8 - 1 and the
    // eight sharers of a line use one L2
    const uint32_t G = gridDim.x;
    uint32_t g = blockIdx.x;
    if (G % kXcds == 0) g = (g % kXcds) * (G / kXcds) + g / kXcds;
    team_run<R, FP64, KEYING, LATLDS, LDSHIST, OBS, LNWG, NR, ORD>(a, lay, (uint64_t)g * kTeams, lds);
}

template <int R, bool FP64, int KEYING, int NR, int ORD>
hipError_t launch_team_nr(hipStream_t st, const McsArgs &a, const TeamLayout &lay)
{
    const dim3 grid((unsigned)((a.W + kTeams - 1) / kTeams)), block(kTeams * kTeam);
    const bool joint = a.joint != nullptr;
    // per-D moments (the produce path, FP64) replace the D histogram
    const bool moms = FP64 && a.moms != nullptr && !joint;
    constexpr int MO = FP64 ? 2 : 0;
    void (*k)(McsArgs, TeamLayout) = nullptr;
    if constexpr (ORD != 0) {
        // lattices in LDS
        k = moms ? k_mcs_team<R, FP64, KEYING, true, false, MO, false, NR, ORD>
            : lay.lds_hist
                ? joint ? k_mcs_team<R, FP64, KEYING, true, true, 1, false, NR, ORD>
                        : k_mcs_team<R, FP64, KEYING, true, true, 0, false, NR, ORD>
            : joint ? k_mcs_team<R, FP64, KEYING, true, false, 1, false, NR, ORD>
                    : k_mcs_team<R, FP64, KEYING, true, false, 0, false, NR, ORD>;
    } else if (lay.lnw_global) {
        // ln W read through windows: lattices and histogram stay in HBM as well
        if constexpr (NR == kLnwgRounds) {
            k = moms ? k_mcs_team<R, FP64, KEYING, false, false, MO, true, NR>
                : joint ? k_mcs_team<R, FP64, KEYING, false, false, 1, true, NR>
                        : k_mcs_team<R, FP64, KEYING, false, false, 0, true, NR>;
        } else {
            return hipErrorInvalidValue;
        }
    } else if (moms) {
        k = lay.lat_lds ? k_mcs_team<R, FP64, KEYING, true, false, MO, false, NR>
                        : k_mcs_team<R, FP64, KEYING, false, false, MO, false, NR>;
    } else {
#define MUCA_TEAM_PICK(LL, LH)                                                  \
    k = joint ? k_mcs_team<R, FP64, KEYING, LL, LH, 1, false, NR>               \
              : k_mcs_team<R, FP64, KEYING, LL, LH, 0, false, NR>;
        if (lay.lat_lds && lay.lds_hist) {
            MUCA_TEAM_PICK(true, true)
        } else if (lay.lat_lds) {
            MUCA_TEAM_PICK(true, false)
        } else if (lay.lds_hist) {
            MUCA_TEAM_PICK(false, true)
        } else {
            MUCA_TEAM_PICK(false, false)
        }
#undef MUCA_TEAM_PICK
    }
    hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lay.bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, grid, block, lay.bytes, st, a, lay);
    e = hipGetLastError();
    if (e == hipSuccess && moms && a.nup > 0)
        e = launch_hist_from_moments(st, a.moms, a.N, a.joint_blocks, a.hist);
    return e;
}

template <int R, bool FP64, int KEYING>
hipError_t launch_team_r(hipStream_t st, const McsArgs &a, const TeamLayout &lay)
{
    if (lay.lnw_global) return launch_team_nr<R, FP64, KEYING, kLnwgRounds, 0>(st, a, lay);
    if (lay.order == 1) {
        if (lay.rounds == 1) return launch_team_nr<R, FP64, KEYING, 1, 1>(st, a, lay);
        if (lay.rounds == 2) return launch_team_nr<R, FP64, KEYING, 2, 1>(st, a, lay);
        return launch_team_nr<R, FP64, KEYING, 3, 1>(st, a, lay);
    }
    if (lay.order == 2) {
        if (lay.rounds == 1) return launch_team_nr<R, FP64, KEYING, 1, 2>(st, a, lay);
        return launch_team_nr<R, FP64, KEYING, 2, 2>(st, a, lay);
    }
    if (lay.rounds == 1) return launch_team_nr<R, FP64, KEYING, 1, 0>(st, a, lay);
    if (lay.rounds == 2) return launch_team_nr<R, FP64, KEYING, 2, 0>(st, a, lay);
    if (lay.rounds == 3) return launch_team_nr<R, FP64, KEYING, 3, 0>(st, a, lay);
    return launch_team_nr<R, FP64, KEYING, 4, 0>(st, a, lay);
}

}  // namespace muca
