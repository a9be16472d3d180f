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
//   A. computes in parallel, attempt j on lane j % 16: the Philox blocks,
//      the proposed spin, dE, dDel, (T)(-dE*beta) and, for each of a window
//      of 8 (weight path) or 6 (produce path) D values around the D the chunk
//      starts from, whether the attempt accepts there (one byte each),
//      screened with the hardware log (the exact log only where the screen
//      is inconclusive);
//   B. resolves the D chain: an attempt is a map of window positions, eight
//      bytes wide, and v_perm_b32 looks four of them up at once, so sixteen
//      lanes' maps compose in a prefix scan of four DPP steps and only one
//      lookup per round of sixteen attempts depends on the D before it.  A
//      round that starts outside the window, or leaves it, gets the masks of
//      its undecided attempts recomputed around the D reached;
//   C. writes the accepted spins, sums dE and dM and fills the histogram.
// What the scan measured against a serial chain of one DPP broadcast, bit
// extract and add per attempt: L = 72, 4096 walkers, from ln W = 0: 341 us per
// launch against 381; L = 128, seeded, NUPDATES = N: 2.19 against 2.51 ms;
// L = 72 thermalisation in FP64: 0.63 against 0.96 ms; L = 256, 16 384
// walkers with moments: 15.8 against 19.5 ms.
// Every acceptance is computed with the reference's operations and rounding:
//   diff = ((T)(-dE*beta) + lnW[D+dDel]) - lnW[D];  accept iff diff >= 0 or
//   acclog(r1) < diff.  Because acclog(r1) < 0 always, that is exactly
//   acclog(r1) < diff.  Results are bit-identical to the one-lane kernel.
// Requires L % 8 == 0 (whole Philox blocks per half-row) and L <= 256.
//
// LDS (dynamic): per team a ring of Philox blocks [2 keys][min(L/2, 64)/4 + 8][4]; the
// acceptance-log table; (T)(-dE*beta) for dE = -8..8; ln W with guard entries
// on each side; the D histogram (u32, when it fits); the workgroup's lattices
// [N][16] int8 (when they fit).
#pragma once
#include "kernels.h"

#include "acclog.h"
#include "moments.h"
#include "philox.h"

namespace muca {

namespace team_detail {

constexpr int kTeam = 16;
constexpr int kTeams = 16;   // per workgroup of 256 lanes
constexpr uint32_t kXcds = 8;   // accelerator dies of an MI355X, one L2 each
// D values per acceptance mask (the most any launch uses).  Narrower
// windows cut the mask work per attempt and make rounds in which D leaves
// the window more frequent.  The weight path (D moves fast in the early
// iterations from ln W = 0) uses 8: L = 72, 4096 walkers, 40.7 attempts/ns
// per weight-loop step against 39.8 with 6.  The produce path (D drifts
// slowly under near-flat weights) uses 6: L = 256, 16 384 walkers, 50.3
// attempts/ns against 41.8 with 8.
constexpr int kWin = 8;
template <int KEYING>
constexpr int kWinFor = KEYING == 1 ? 6 : 8;
// Rounds per chunk where ln W is in HBM: those launches have 128 VGPRs (four
// wavefronts per SIMD), which two rounds' state fits without spills.  L = 256,
// 16 384 walkers, 65 536 attempts each, with moments / without: 15.8 / 15.5 ms
// with two rounds, 16.8 / 16.1 with three, 18.5 / 16.0 with four.
constexpr int kLnwgRounds = 2;
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
__device__ __forceinline__ uint32_t sign_word(double x)
{
    return (uint32_t)(__double_as_longlong(x) >> 32);
}

// value of lane L of this lane's 16-lane row (v_mov_b32_dpp row_newbcast:L;
// every lane of the row reads a valid source, so no old value is needed)
template <int L>
__device__ __forceinline__ int32_t row_bcast(int32_t v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x150 + L, 0xf, 0xf, false);
}

// a monotone FP32 image of |x|'s order: x itself, or the high word of a double
// read as a float (magnitudes above 2^1016 read as NaN, which a minimum skips)
__device__ __forceinline__ float mag_word(float x)
{
    return x;
}
__device__ __forceinline__ float mag_word(double x)
{
    return __uint_as_float((uint32_t)(__double_as_longlong(x) >> 32));
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
template <int R, bool FP64, int KEYING, bool LATLDS, bool LDSHIST, int OBS, bool LNWG, int NR>
__device__ __forceinline__ void team_run(const McsArgs &a, const TeamLayout &lay, uint64_t wbase,
                                         unsigned char *lds)
{
    typedef typename std::conditional<FP64, double, float>::type T;
    constexpr int KW = kWinFor<KEYING>;   // this launch's mask width (<= kWin)
    constexpr bool JOINT = OBS == 1, MOMS = OBS == 2, TRACKM = OBS >= 1;
    __syncthreads();   // LDS may still be read by a previous call's flush
    T *wt = (T *)(lds + lay.off_w) + kGuard;   // valid for [-kGuard, N + kGuard]
    uint32_t *hist = (uint32_t *)(lds + lay.off_hist);
    int8_t *latl = (int8_t *)(lds + lay.off_lat);
    double *logtab = (double *)(lds + lay.off_tab);
    T *fdet = (T *)(lds + lay.off_fde) + 8;    // fdet[dE] = (T)(-dE * beta), |dE| <= 8
    const int tid = threadIdx.x, team = tid >> 4, tl = tid & 15;
    const uint32_t N = a.N, L = a.L, Rw = lay.row;
    unsigned char *tbase = lds + lay.off_team + (size_t)team * lay.team_bytes;
    uint32_t *rng = (uint32_t *)tbase;                          // [2][ring][4]
    T *winb = (T *)(tbase + lay.off_win);                       // LNWG: lnW[dlo - 1 .. dlo + KW]
    // ln W at any D: from LDS, or from HBM (clamped into [0, N]; only
    // positions a walker cannot be at read a clamped value)
    auto lnw_at = [&](int32_t i) -> T {
        if (LNWG) {
            const int32_t c = min(max(i, 0), (int32_t)a.N);
            return FP64 ? (T)a.lnw64[c] : (T)a.lnw32[c];
        }
        return wt[i];
    };

    const uint64_t W = a.W;
    const uint64_t w = wbase + team;
    const bool active = w < W;

    if (!LNWG) {
#pragma unroll 4
        for (int i = (int)tid - kGuard; i <= (int)N + kGuard; i += blockDim.x) {
            T v = (T)0;
            if (i >= 0 && i <= (int)N) v = FP64 ? (T)a.lnw64[i] : (T)a.lnw32[i];
            wt[i] = v;
        }
    }
    // MOMS: this team's moment slots, word k of slot s at msl[k * kMomSlots + s]
    uint64_t *msl = (uint64_t *)(tbase + lay.off_mom);
    if (MOMS)
        for (int k = 0; k < kMomLdsWords; k++) msl[k * kMomSlots + tl] = 0;
    if (LDSHIST)
        for (uint32_t i = tid; i <= N; i += blockDim.x) hist[i] = a.hist_preload;
    acclog_table_to_lds(logtab, tid, blockDim.x);
    if (tid < 17) fdet[tid - 8] = (T)(-(double)(tid - 8) * a.beta);
    // LATLDS: the tile's lattices move between the site-major layout in HBM
    // and walker-major LDS rows.  For sixteen whole walkers on 16-byte
    // aligned rows, a lane moves four consecutive sites at a time: four
    // 16-byte global accesses (one per site: the tile's walkers), a 4x4 byte
    // transpose per four walkers, sixteen dword LDS accesses (one per
    // walker); a lane's four loads are all in flight before the first is
    // used.  Otherwise one byte per lane and step.
    const bool lat_vec = LATLDS && W % kTeams == 0 && wbase + kTeams <= W &&
                         ((uintptr_t)a.lat & 15) == 0;   // N % 64 == 0 (L % 8 == 0)
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
        } else {
            for (uint32_t e = tid; e < N * kTeams; e += blockDim.x) {
                const uint32_t site = e >> 4, t = e & 15;
                latl[t * lay.lat_stride + site] =
                    (wbase + t < W) ? a.lat[(uint64_t)site * W + wbase + t] : (int8_t)0;
            }
        }
    }
    __syncthreads();

    if (active) {
        auto sp = [&](uint32_t site) -> int8_t & {
            return LATLDS ? latl[team * lay.lat_stride + site] : a.lat[(uint64_t)site * W + w];
        };
        const uint32_t wid = a.w_offset + (uint32_t)w;
        const uint32_t k1a = KEYING == 0 ? 2u * wid : wid;
        const uint32_t k1b = 0xdecafbadu;
        const uint32_t k3a = KEYING == 0 ? 2u * wid + 50000u : wid + 40000u;
        const uint32_t k3b = KEYING == 0 ? 0x11cafeadu : 0xdecafeadu;
        int32_t d = a.D[w], e = a.E[w], m = a.M[w];
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
        // joint-histogram entries of this lane's attempts, counted for the bin
        // in use and the one before it and added with one atomic when a third
        // bin comes up (a walker stepping back and forth adds nothing)
        uint64_t jrun = 0, jprun = 0;
        int64_t jbin = -1, jpbin = -1;
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
        // the scan's shifted-in maps per level: the lanes that have no source
        // lane at a level keep the identity from here on
        uint32_t ql[4], qh[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            ql[k] = window_id<KW>(0);
            qh[k] = window_id<KW>(1);
        }
        // a workgroup adds at most 16 NUPDATES counts to one u32 bin
        const bool may_wrap = a.hist_preload != 0 || (uint64_t)kTeams * a.nup >= (1ull << 32);
        for (int phase = 0; phase < 2; phase++) {
            const uint64_t n = phase ? a.nup : a.therm;
            // A half-row is worked in chunks of up to 16 NR attempts (no two
            // sites of a half-row are neighbours, so any split of it is exact).
            // Attempt rs of a phase is at sweep position rs mod N: half h
            // (x parity), row y, place jb in the half-row -- advanced chunk by
            // chunk from 0, without divisions.
            uint32_t h = 0, y = 0, jb = 0;
            for (uint64_t rs = 0; rs < n;) {
                const uint32_t cnt = (uint32_t)min((uint64_t)min(Rw - jb, 16u * NR), n - rs);
                // ---- A1: the walker's Philox stream (block b uses counter b + 1;
                // the stream runs on across chunks and phases) is generated
                // eight blocks x two keys per pass into a ring of `RB` blocks per
                // key, so no lane idles when a chunk's block count is not a
                // multiple of eight.  Blocks [blk0, blk0 + nblk) serve this
                // chunk; a pass may run up to 7 blocks ahead, and RB >= nblk + 8
                // keeps those from overwriting blocks still in use.
                const uint32_t nblk = (cnt + 3) / 4;
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
                // ring slot of this chunk's first block (blocks are contiguous
                // from one chunk to the next, across the phase change too)
                const uint32_t slot0 = cur_slot;
                cur_slot = cur_slot + nblk >= RB ? cur_slot + nblk - RB : cur_slot + nblk;
                wave_sync();
                // ---- A2: attempt j = 16 r + tl on this lane, everything in registers
                int32_t dlo = d - KW / 2;           // mask bit k <-> D = dlo + k
                // lnW[dlo + k] at wcen[k], k = -1 .. KW (LNWG: staged in the
                // team's window from HBM)
                auto window = [&]() -> const T * {
                    if (LNWG) {
                        if (tl < KW + 2) winb[tl] = lnw_at(dlo - 1 + tl);
                        wave_sync();
                        return winb + 1;
                    }
                    return wt + dlo;
                };
                const T *wcen = window();
                T wfrom[KW];                        // lnW[dlo .. dlo + KW - 1]
#pragma unroll
                for (int k = 0; k < KW; k++) wfrom[k] = wcen[k];
                const int32_t dlo_a = dlo;            // the window of every mask made here
                const uint32_t yu = (y + 1 == L) ? 0 : y + 1, yd = (y == 0) ? L - 1 : y - 1;
                const uint32_t s4 = slot0 * 4, ringw = RB * 4;   // ring word of attempt j: s4 + j (mod ringw)
                // attempt j's accept bytes: byte k is 0xff iff it accepts at
                // D = dlo_a + k (bytes 0..3, 4..7)
                uint32_t alo[NR], ahi[NR];
                // (dDel + 1) | (dE + 8) << 2 | (new - old + 2) << 7 | (new + 1) << 10
                int32_t info[NR];
                // Byte k = 0..KW-1: accept at D = dlo + k, i.e. acclog(r1) <
                // ((fde + lnW[D + dDel]) - lnW[D]), screened with the hardware
                // log and its proven band: la + band < diff accepts, la - band
                // >= diff rejects.  Byte k is the sign of e = thi - diff (e is
                // -0 never, +0 iff thi == diff, which rejects); a diff with
                // tlo < diff <= thi, i.e. 0 <= e < thi - tlo, needs the exact
                // log -- flagged (with margin) by min |e| < 2 (thi - tlo).
                // The minimum is taken over mag_word (exact in FP32, the high
                // words in FP64, compared there with <=).  An attempt past the
                // chunk's end has fde = -inf and accepts nowhere.
                auto accept_bytes = [&](const T *wf, const T *wc, uint32_t r1, T fde,
                                        int32_t ddel, uint32_t &lo, uint32_t &hi) {
                    const T *wto = wc + ddel;
                    T diff[KW];
#pragma unroll
                    for (int k = 0; k < KW; k++) {
                        diff[k] = fde + wto[k];
                        diff[k] = diff[k] - wf[k];
                    }
                    const float la = acclog_fast_u01(r1);
                    const float band = acclog_fast_band(la);
                    const T thi = (T)(la + band), tlo = (T)(la - band);
                    uint32_t sg[8];
                    float emin = 1e30f;
#pragma unroll
                    for (int k = 0; k < KW; k++) {
                        const T e = thi - diff[k];
                        sg[k] = sign_word(e);
                        emin = fminf(emin, fabsf(mag_word(e)));
                    }
                    sign_bytes<KW>(sg, lo, hi);
                    const float lim = mag_word((thi - tlo) + (thi - tlo));
                    const bool amb = FP64 ? emin <= lim : emin < lim;
                    if (__builtin_amdgcn_ballot_w64(amb)) {   // rare: a diff within the band
                        if (amb) {
                            const T tlog =
                                (T)(float)acclog_u01_double_tab(r1, logtab, logtab + 128);
#pragma unroll
                            for (int k = 0; k < KW; k++) sg[k] = tlog < diff[k] ? 0x80000000u : 0u;
                            sign_bytes<KW>(sg, lo, hi);
                        }
                    }
                };
                // Branch-free over the rounds so that the loads of all rounds
                // can be in flight together: a lane past the end of the
                // chunk works on a clamped (in-bounds) attempt and keeps
                // nothing of it.
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const uint32_t j = 16 * r + tl;
                    const bool valid = j < cnt;
                    const uint32_t jc = valid ? j : cnt - 1;
                    const uint32_t x = 2 * (jb + jc) + h;
                    const uint32_t xr = (x + 1 == L) ? 0 : x + 1;
                    const uint32_t xl = (x == 0) ? L - 1 : x - 1;
                    int32_t old_s, nb;
                    if (PF && pf_have) {
                        old_s = pf_s[r];
                        nb = pf_r[r] + pf_l[r] + pf_u[r] + ((pf_fwd && fin[r] != -9) ? fin[r] : pf_d[r]);
                    } else {
                        old_s = sp(y * L + x);
                        nb = sp(y * L + xr) + sp(y * L + xl) + sp(yu * L + x) + sp(yd * L + x);
                    }
                    uint32_t widx = s4 + jc;
                    widx = widx >= ringw ? widx - ringw : widx;
                    const uint32_t r1 = rng[widx], r3 = rng[ringw + widx];
                    int32_t new_s = old_s + (r3 < 0x80000000u ? 1 : -1);
                    new_s = new_s == 2 ? -1 : (new_s == -2 ? 1 : new_s);
                    const int32_t ds = new_s - old_s;
                    const int32_t dE = -ds * nb;
                    const int32_t ddel = new_s * new_s - old_s * old_s;
                    // (T)(-dE * beta) by arithmetic (the same operations as
                    // the table in LDS, without a dependent LDS load)
                    const T fde = (T)(-(double)dE * a.beta);
                    accept_bytes(wfrom, wcen, r1, valid ? fde : -(T)INFINITY, ddel, alo[r], ahi[r]);
                    info[r] = (ddel + 1) | ((dE + 8) << 2) | ((ds + 2) << 7) | ((new_s + 1) << 10);
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
#pragma unroll
                        for (int r = 0; r < NR; r++) {
                            const uint32_t jn = min(16u * r + tl, cnt_n - 1);
                            const uint32_t x = 2 * (jb_n + jn) + h_n;
                            const uint32_t xr = (x + 1 == L) ? 0 : x + 1;
                            const uint32_t xl = (x == 0) ? L - 1 : x - 1;
                            pf_s[r] = sp(y_n * L + x);
                            pf_r[r] = sp(y_n * L + xr);
                            pf_l[r] = sp(y_n * L + xl);
                            pf_u[r] = sp(yu_n * L + x);
                            pf_d[r] = sp(yd_n * L + x);
                        }
                    }
                }
                // ---- B: the D chain.  Attempt j maps the window position k =
                // D - dlo before it to the one after it: k + dDel where byte k
                // of its accept bytes is set, else k; a position outside the
                // window is 0xff and stays so.  A map is eight bytes, and
                // v_perm_b32 looks up four of them at once (a selector of 0xff
                // gives 0xff), so that two maps compose in two instructions
                // and sixteen lanes' maps in a prefix scan of four levels.  The
                // scans of all rounds are independent of D and of each other;
                // only one lookup per round depends on the D the round before
                // ended at.
                const uint32_t sh = (uint32_t)(tid & 48);    // this team's 16 lanes of a ballot
                const uint32_t upto = (2u << tl) - 1u;       // steps 0..tl of a round
                // made ahead of the rounds where registers allow
                constexpr bool AHEAD = !LNWG;
                auto scan = [&](uint32_t lo, uint32_t hi, int32_t inf, uint32_t &plo,
                                uint32_t &phi) {
                    window_map<KW>(lo, hi, (uint32_t)inf, plo, phi);
                    if (!AHEAD)
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            ql[k] = window_id<KW>(0);
                            qh[k] = window_id<KW>(1);
                        }
                    scan_level<KW, 0x111>(plo, phi, ql[0], qh[0]);
                    scan_level<KW, 0x112>(plo, phi, ql[1], qh[1]);
                    scan_level<KW, 0x114>(plo, phi, ql[2], qh[2]);
                    scan_level<KW, 0x118>(plo, phi, ql[3], qh[3]);
                };
                // the maps of steps 0..tl of each round
                uint32_t plo[NR], phi[NR];
                if (AHEAD)
#pragma unroll
                    for (int r = 0; r < NR; r++) scan(alo[r], ahi[r], info[r], plo[r], phi[r]);
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const uint32_t j0 = 16 * r;
                    if (PF) fin[r] = -9;
                    if (j0 >= cnt) continue;
                    if (!AHEAD) scan(alo[r], ahi[r], info[r], plo[r], phi[r]);
                    const bool valid = j0 + tl < cnt;
                    // the window's accept bytes recomputed around dlo by all
                    // lanes of the team; steps below `from` are decided and
                    // become identities
                    auto remask = [&](uint32_t from) {
                        const T *wc = window();
                        T wf[KW];
#pragma unroll
                        for (int k = 0; k < KW; k++) wf[k] = wc[k];
                        uint32_t w1 = s4 + min(j0 + tl, cnt - 1);
                        w1 = w1 >= ringw ? w1 - ringw : w1;
                        const T fde = fdet[((info[r] >> 2) & 31) - 8];
                        accept_bytes(wf, wc, rng[w1], valid && tl >= from ? fde : -(T)INFINITY,
                                     (info[r] & 3) - 1, alo[r], ahi[r]);
                        scan(alo[r], ahi[r], info[r], plo[r], phi[r]);
                    };
                    // the window follows D from round to round: a round that
                    // starts outside the masks' window gets its masks
                    // recomputed around the current D (only this round's: the
                    // later rounds' stay relative to dlo_a)
                    dlo = dlo_a;
                    uint32_t off = (uint32_t)(d - dlo_a);
                    const bool shift = off >= (uint32_t)KW;
                    if (__builtin_amdgcn_ballot_w64(shift)) {
                        if (shift) {
                            dlo = d - KW / 2;
                            off = KW / 2;
                            remask(0);
                        }
                    }
                    uint32_t o = window_at(plo[r], phi[r], off);
                    uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(
                        (int)off, (int)o, 0x111, 0xf, 0xf, false);
                    // this lane's attempt: accepted, and D (and M) after it
                    bool acc = window_at(alo[r], ahi[r], before) != 0;
                    int32_t dv = dlo + (int32_t)o, mv = 0;
                    // Rare: D left the window at step k.  Steps 0..k stand (step
                    // k is accepted and moved D by its dDel); the masks of the
                    // later ones are recomputed around D there, and so on until
                    // the round is done.  k grows by KW / 2 at least each time.
                    uint64_t outs;
                    bool out = o == 0xffu;
                    while ((outs = __builtin_amdgcn_ballot_w64(out)) != 0) {
                        const uint32_t mine = (uint32_t)(outs >> sh) & 0xffffu;
                        if (mine) {
                            const uint32_t k = (uint32_t)__builtin_ctz(mine);
                            const int32_t dk = dlo + (int32_t)before + (info[r] & 3) - 1;
                            if ((uint32_t)tl == k) dv = dk;
                            dlo = __shfl(dk, (int)k, kTeam) - KW / 2;
                            remask(k + 1);
                            o = window_at(plo[r], phi[r], KW / 2);
                            before = (uint32_t)__builtin_amdgcn_update_dpp(
                                KW / 2, (int)o, 0x111, 0xf, 0xf, false);
                            out = o == 0xffu;
                            if ((uint32_t)tl > k) {
                                acc = window_at(alo[r], ahi[r], before) != 0;
                                dv = dlo + (int32_t)o;
                            }
                        }
                    }
                    d = row_bcast<15>(dv);
                    if (TRACKM) {
                        // M after this lane's step: an inclusive scan over the
                        // team of the accepted spin changes
                        int32_t x = acc ? ((info[r] >> 7) & 7) - 2 : 0;
                        x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
                        x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
                        mv = m + x;
                        m += row_bcast<15>(x);
                    }
                    // ---- C: accepted spins, dE / dM sums, histogram of the round
                    const uint32_t j = j0 + tl, left = min(cnt - j0, 16u);
                    const int32_t ns = ((info[r] >> 10) & 3) - 1;    // the proposed spin
                    const int32_t ds = ((info[r] >> 7) & 7) - 2;
                    // the site's spin after this chunk
                    if (PF) fin[r] = valid ? (acc ? ns : ns - ds) : -9;
                    if (acc) {
                        // the new spin is known from phase A: no site of
                        // the chunk is written between its read and here
                        sp(y * L + 2 * (jb + j) + h) = (int8_t)ns;
                        de_lane += ((info[r] >> 2) & 31) - 8;
                        dm_lane += ds;
                    }
                    if (JOINT && phase && valid) {
                        const int64_t dd = dv;
                        const int64_t mm = min(max((int64_t)mv, -dd), dd);
                        const int64_t jbn = (mm + dd * dd + 2 * dd) / 2;
                        if (jbn != jbin) {
                            if (jbn == jpbin) {
                                const uint64_t t = jrun;
                                jrun = jprun;
                                jprun = t;
                                jpbin = jbin;
                            } else {
                                if (jprun)
                                    atomicAdd((unsigned long long *)&jbase[jpbin], jprun);
                                jprun = jrun;
                                jpbin = jbin;
                                jrun = 0;
                            }
                            jbin = jbn;
                        }
                        jrun++;
                    }
                    if (phase && !MOMS) {
                        // The D histogram: a round's steps split into runs at one D,
                        // starting at step 0 and at every accepted step that
                        // changed D; the first lane of a run adds its length (one
                        // atomic per run instead of sixteen on the same bin)
                        const bool moved = acc && (info[r] & 3) != 1;
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
                        // Attempt j records the (D, M) after its step.  Steps that
                        // are not accepted keep the state, so a round splits into
                        // segments that start at step 0 and at every accepted step
                        // and share one (D, M); the first lane of each segment adds
                        // len x (1, |M|, M^2, M^4) to the slot of its D.
                        const uint32_t ab =
                            (uint32_t)(__builtin_amdgcn_ballot_w64(acc) >> sh) & 0xffffu;
                        const bool lead = tl < left && (tl == 0 || acc);
                        const uint32_t later = ab & ~upto;
                        const uint32_t len =
                            (later ? (uint32_t)__builtin_ctz(later) : left) - (uint32_t)tl;
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
                jb += cnt;
                if (jb == Rw) {
                    jb = 0;
                    if (++y == L) {
                        y = 0;
                        h ^= 1u;
                    }
                }
            }
            c0base += (uint32_t)((n + 3) / 4);
        }
        if (JOINT) {
            if (jrun) atomicAdd((unsigned long long *)&jbase[jbin], jrun);
            if (jprun) atomicAdd((unsigned long long *)&jbase[jpbin], jprun);
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
        } else {
            for (uint32_t e2 = tid; e2 < N * kTeams; e2 += blockDim.x) {
                const uint32_t site = e2 >> 4, t = e2 & 15;
                if (wbase + t < W) a.lat[(uint64_t)site * W + wbase + t] = latl[t * lay.lat_stride + site];
            }
        }
    }
}

// LNWG launches are the large lattices (L >= 136) with many walkers: they
// are held to 128 VGPRs, four wavefronts per SIMD
template <int R, bool FP64, int KEYING, bool LATLDS, bool LDSHIST, int OBS, bool LNWG, int NR>
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
    team_run<R, FP64, KEYING, LATLDS, LDSHIST, OBS, LNWG, NR>(a, lay, (uint64_t)g * kTeams, lds);
}

template <int R, bool FP64, int KEYING, int NR>
hipError_t launch_team_nr(hipStream_t st, const McsArgs &a, const TeamLayout &lay)
{
    const dim3 grid((unsigned)((a.W + kTeams - 1) / kTeams)), block(kTeams * kTeam);
    const bool joint = a.joint != nullptr;
    // per-D moments (the produce path, FP64) replace the D histogram
    const bool moms = FP64 && a.moms != nullptr && !joint;
    constexpr int MO = FP64 ? 2 : 0;
    void (*k)(McsArgs, TeamLayout) = nullptr;
    if (lay.lnw_global) {
        // ln W too large for LDS (L >= 136): lattices and histogram stay in
        // HBM as well
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
    const uint32_t rounds = (lay.row + 15) / 16;
    if (lay.lnw_global) return launch_team_nr<R, FP64, KEYING, kLnwgRounds>(st, a, lay);
    if (rounds <= 1) return launch_team_nr<R, FP64, KEYING, 1>(st, a, lay);
    if (rounds <= 2) return launch_team_nr<R, FP64, KEYING, 2>(st, a, lay);
    if (rounds <= 3) return launch_team_nr<R, FP64, KEYING, 3>(st, a, lay);
    return launch_team_nr<R, FP64, KEYING, 4>(st, a, lay);   // longer half-rows in chunks of 64
}

}  // namespace muca
