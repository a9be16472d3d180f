// muca_lane.hip -- the lane update kernel: one, two or four walkers per lane,
// for even L.
//
// For large walker counts (enough wavefronts to hide memory latency) the
// update is bound by VALU issue, about 60 instructions per attempt, a third of
// them Philox.  This kernel trims it:
//  - the reference's even-L site order (muca_delta_multigpu.cu:173: even
//    linear indices, then odd ones) is walked with scalar arithmetic instead
//    of the order/neighbour tables, and a lane's place among the walkers is
//    the 32-bit offset of every load;
//  - four walkers per lane load a dword per site, so that four independent
//    chains share one address and one memory instruction, and sum their
//    neighbours bytewise;
//  - ln W, the D histogram and (T)(-dE * beta) live in LDS, and lnW[D] is
//    carried from attempt to attempt;
//  - the five spins of an attempt are loaded four attempts ahead (PD; one ahead
//    with one walker per lane);
//  - proposals are looked up with v_perm_b32 (proposal.h);
//  - the acceptance "diff >= 0 or log(u) < diff" (equivalently log(u) <
//    diff, since log(u) < 0) is screened with the hardware log: outside a
//    band proven exhaustively around it, the decision needs no exact log;
//    inside, the correctly rounded acclog decides.
// Results are bit-identical to the generic kernel and the reference chain.
// L = 72, 524 288 walkers, therm = N: 4.6 ms (590 attempts/ns) against 9.85 ms
// for one walker per lane with byte loads one attempt ahead; four walkers per
// lane with loads one attempt ahead 5.0 ms, and 5.2 with a test of the phase's
// end between the attempts, which makes the waits at its joins drain them.
#include "kernels.h"

#include "acclog.h"
#include "philox.h"
#include "proposal.h"

namespace muca {

template <bool FP64>
using lane_t = typename std::conditional<FP64, double, float>::type;   // of ln W and diff

// V walkers' spins of one site: a dword, a half-word or a byte
template <int V>
__device__ __forceinline__ uint32_t load_spins(const uint8_t *p)
{
    if (V == 4) return *(const uint32_t *)p;
    if (V == 2) return *(const uint16_t *)p;
    return *p;
}
template <int V>
__device__ __forceinline__ void store_spins(uint8_t *p, uint32_t v)
{
    if (V == 4)
        *(uint32_t *)p = v;
    else if (V == 2)
        *(uint16_t *)p = (uint16_t)v;
    else
        *p = (uint8_t)v;
}

// The walkers wbase .. wbase + V blockDim.x - 1 of the launch described by a,
// V per lane (every lane of the workgroup calls it together; W % V == 0 and
// the lattice is V-aligned).
// OBS: 0 the D histogram; 1 joint H(D,M) per walker block as well.
// fde_tab: 17 entries in LDS, the kernel's (a variable of this function would
// be one per variant that a kernel calls).
template <int R, bool FP64, int KEYING, bool LDSHIST, int OBS, int V, int PD>
__device__ __forceinline__ void lane_run(const McsArgs &a, uint32_t lds_w, uint64_t wbase,
                                         unsigned char *lds, lane_t<FP64> *fde_tab)
{
    typedef lane_t<FP64> T;
    constexpr bool JOINT = OBS == 1;
    __syncthreads();   // LDS may still be read by a previous call's flush
    T *wt = (T *)lds, *fdet = fde_tab + 8;   // fdet[dE] = (T)(-dE * beta), |dE| <= 8
    uint32_t *hist = (uint32_t *)(lds + lds_w);
    const uint32_t N = a.N, L = a.L, Rw = L / 2;
    if (threadIdx.x < 17) fdet[(int)threadIdx.x - 8] = (T)(-(double)((int)threadIdx.x - 8) * a.beta);
    for (uint32_t i = threadIdx.x; i <= N; i += blockDim.x) {
        wt[i] = FP64 ? (T)a.lnw64[i] : (T)a.lnw32[i];
        if (LDSHIST) hist[i] = a.hist_preload;
    }
    __syncthreads();
    const uint64_t w0 = wbase + (uint64_t)threadIdx.x * V;
    if (w0 < a.W) {
        const uint64_t W = a.W;
        const uint32_t wl = (uint32_t)w0;   // walker counts are 32-bit
        uint8_t *const lat = (uint8_t *)a.lat;
        int32_t e[V], d[V], m[V];
        T wc[V];            // lnW[d]
        int32_t acc_em[V];  // accepted (dE << 16) - dM since the last widening
        uint64_t *jbase[V];
        uint32_t jrun[V], jprun[V];
        int32_t jbin[V], jpbin[V];
#pragma unroll
        for (int v = 0; v < V; v++) {
            e[v] = a.E[w0 + v];
            d[v] = a.D[w0 + v];
            m[v] = a.M[w0 + v];
            wc[v] = wt[d[v]];
            acc_em[v] = 0;
            // joint entries are counted for the bin in use and the one before
            // it and added with one atomic when a third comes up
            jrun[v] = jprun[v] = 0;
            jbin[v] = jpbin[v] = 0;
            jbase[v] = JOINT ? a.joint + ((w0 + v) / a.block_walkers) * a.joint_stride : nullptr;
        }
        auto widen = [&]() {
#pragma unroll
            for (int v = 0; v < V; v++) {
                const int32_t low = (int32_t)(int16_t)(uint16_t)acc_em[v];
                e[v] += (acc_em[v] - low) >> 16;
                if (!JOINT) m[v] -= low;
                acc_em[v] = 0;
            }
        };
        // The site and its four neighbours are the same in every lane: their
        // addresses are scalars, and a walker's place wl is the lane's offset.
        // A Cursor walks the site order (half h, row y, place xi).
        const uint64_t rowb = (uint64_t)L * W;
        struct Cursor {
            uint32_t h, y, xi;
            uint8_t *s;   // the site
        };
        auto next = [&](Cursor &c) {
            if (++c.xi == Rw) {
                c.xi = 0;
                if (++c.y == L) {
                    c.y = 0;
                    c.h ^= 1u;
                }
                c.s = lat + (uint64_t)c.y * rowb + (uint64_t)c.h * W;
            } else {
                c.s += 2 * W;
            }
        };
        uint32_t c0 = 0;
        // a workgroup adds at most V blockDim NUPDATES counts to one u32 bin
        const bool may_wrap =
            a.hist_preload != 0 || (uint64_t)V * blockDim.x * a.nup >= (1ull << 32);
        for (int phase = 0; phase < 2; phase++) {
            const uint64_t n = phase ? a.nup : a.therm;
            if (n == 0) continue;
            // An attempt's spins (site, right, left, upper and lower neighbour)
            // are loaded PD attempts ahead.  Exact while the PD attempts
            // before it change none of them: the right and left neighbours
            // belong to the other half, the upper one comes later, and the
            // lower one is the site of the attempt Rw before (PD < Rw).
            // The loads are made without a branch, past the phase's end too
            // (sites of the sweep that are then not used), so that a wait for
            // one attempt's spins leaves the later ones in flight.
            uint32_t sp[PD], rp[PD], lp[PD], up[PD], dp[PD];
            Cursor ahead{0, 0, 0, lat}, cur{0, 0, 0, lat};
            auto fetch = [&](int q) {
                const Cursor &c = ahead;
                const bool first = !c.h && c.xi == 0, last = c.h && c.xi == Rw - 1;
                const uint64_t wrap = (L - 1) * W, wrapy = (L - 1) * rowb;
                sp[q] = load_spins<V>(c.s + wl);
                rp[q] = load_spins<V>((last ? c.s - wrap : c.s + W) + wl);
                lp[q] = load_spins<V>((first ? c.s + wrap : c.s - W) + wl);
                up[q] = load_spins<V>((c.y + 1 == L ? c.s - wrapy : c.s + rowb) + wl);
                dp[q] = load_spins<V>((c.y == 0 ? c.s + wrapy : c.s - rowb) + wl);
                next(ahead);
            };
#pragma unroll
            for (int q = 0; q < PD; q++) fetch(q);
            philox4 r1[V], r3[V];
            auto draw = [&]() {
                ++c0;
#pragma unroll
                for (int v = 0; v < V; v++) {
                    const uint32_t wid = a.w_offset + wl + v;
                    r1[v] = philox4x32<R>(c0, a.seed, a.iter, 0xBADC0DEDu,
                                          KEYING == 0 ? 2u * wid : wid, 0xdecafbadu);
                    r3[v] = philox4x32<R>(c0, a.seed, a.iter, 0xBADC0DEDu,
                                          KEYING == 0 ? 2u * wid + 50000u : wid + 40000u,
                                          KEYING == 0 ? 0x11cafeadu : 0xdecafeadu);
                }
            };
            // attempt i0 + j, word j of the block drawn
            auto attempt = [&](auto jc) {
                constexpr int j = decltype(jc)::value;
                constexpr int kMask = PD - 1;
                const int q = j & kMask;
                // a copy, so that the next load of this place can go into the
                // register that the loop keeps for it (a register copied at the
                // loop's end would wait for its load there)
                uint32_t s4;
                asm volatile("v_mov_b32 %0, %1" : "=&v"(s4) : "v"(sp[q]));
                // neighbour sums modulo 16 per byte: -4 .. 4 as four bits
                const uint32_t nib = 0x0f0f0f0fu;
                uint32_t nb4 = (rp[q] & nib) + (lp[q] & nib) + (up[q] & nib) + (dp[q] & nib);
                asm volatile("" : "+v"(nb4) : : "memory");
                uint8_t *const pc = cur.s;
                next(cur);
                fetch(q);
                uint32_t at[V];
                int32_t dE[V], dd[V];
                T wn[V], diff[V];
                bool ok[V], amb[V], any_amb = false;
#pragma unroll
                for (int v = 0; v < V; v++) {
                    const int32_t old_s = (int32_t)(s4 << (24 - 8 * v)) >> 24;
                    const int32_t nb = (int32_t)(nb4 << (28 - 8 * v)) >> 28;
                    at[v] = proposal_index(old_s, r3[v].v[j]);
                    dd[v] = proposal_ddel(at[v]);
                    dE[v] = __mul24(proposal_mds(at[v]), nb);
                    wn[v] = wt[d[v] + dd[v]];
                    diff[v] = fdet[dE[v]] + wn[v];
                    diff[v] = diff[v] - wc[v];
                    const float thi = acclog_screen(r1[v].v[j]);
                    const T x = (T)thi - diff[v];
                    ok[v] = x < (T)0;
                    amb[v] = fabs(x) < (T)acclog_screen_lim(thi);
                    any_amb = any_amb || amb[v];
                }
                if (__builtin_amdgcn_ballot_w64(any_amb)) {   // rare
#pragma unroll
                    for (int v = 0; v < V; v++)
                        if (amb[v]) ok[v] = (T)acclog_u01(r1[v].v[j]) < diff[v];
                }
                // selects, not branches: some lane accepts nearly always
                uint32_t new4 = s4;
#pragma unroll
                for (int v = 0; v < V; v++) {
                    const int32_t mds = proposal_mds(at[v]);
                    const uint32_t put = __builtin_amdgcn_perm(
                        proposal_new(at[v]), new4,
                        (0x03020100u & ~(0xffu << (8 * v))) | (0x04u << (8 * v)));
                    new4 = ok[v] ? put : new4;
                    d[v] += ok[v] ? dd[v] : 0;
                    wc[v] = ok[v] ? wn[v] : wc[v];
                    acc_em[v] += ok[v] ? (dE[v] << 16) + mds : 0;
                    if (JOINT) m[v] -= ok[v] ? mds : 0;
                }
                if (new4 != s4) store_spins<V>(pc + wl, new4);
                if (phase) {
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        if (LDSHIST) {
                            if (may_wrap) {
                                // a u32 bin that wraps carries 2^32 into HBM
                                if (atomicAdd(&hist[d[v]], 1u) == 0xFFFFFFFFu)
                                    atomicAdd((unsigned long long *)&a.hist[d[v]],
                                              1ull << 32);
                            } else {
                                atomicAdd(&hist[d[v]], 1u);
                            }
                        } else {
                            atomicAdd((unsigned long long *)&a.hist[d[v]], 1ull);
                        }
                        if (JOINT) {
                            // (M + D^2 + 2 D) / 2 < 2^31: ln W in LDS needs L <= 202
                            const int32_t mm = min(max(m[v], -d[v]), d[v]);
                            const int32_t jb =
                                (int32_t)(((int64_t)mm + (int64_t)d[v] * (d[v] + 2)) >> 1);
                            if (jb != jbin[v]) {
                                if (jb == jpbin[v]) {
                                    const uint32_t t = jrun[v];
                                    jrun[v] = jprun[v];
                                    jprun[v] = t;
                                    jpbin[v] = jbin[v];
                                } else {
                                    if (jprun[v])
                                        atomicAdd((unsigned long long *)&jbase[v][jpbin[v]],
                                                  (unsigned long long)jprun[v]);
                                    jprun[v] = jrun[v];
                                    jpbin[v] = jbin[v];
                                    jrun[v] = 0;
                                }
                                jbin[v] = jb;
                            }
                            // a run stays below 2^32: it is added when full
                            if (++jrun[v] == 0xFFFFFFFFu) {
                                atomicAdd((unsigned long long *)&jbase[v][jb],
                                          (unsigned long long)jrun[v]);
                                jrun[v] = 0;
                            }
                        }
                    }
                }
            };
            using J0 = std::integral_constant<int, 0>;
            using J1 = std::integral_constant<int, 1>;
            using J2 = std::integral_constant<int, 2>;
            using J3 = std::integral_constant<int, 3>;
            // whole blocks without a test between their attempts: a join of
            // paths with and without a load would wait for it
            uint64_t i0 = 0;
            for (; i0 + 4 <= n; i0 += 4) {
                draw();
                if ((i0 & 1023u) == 0) widen();   // |sum dE| <= 8 x 1024, |sum dM| <= 2 x 1024
                attempt(J0());
                attempt(J1());
                attempt(J2());
                attempt(J3());
            }
            if (i0 < n) {
                draw();
                attempt(J0());
                if (i0 + 1 < n) attempt(J1());
                if (i0 + 2 < n) attempt(J2());
            }
            widen();
        }
#pragma unroll
        for (int v = 0; v < V; v++) {
            if (JOINT && jrun[v])
                atomicAdd((unsigned long long *)&jbase[v][jbin[v]], (unsigned long long)jrun[v]);
            if (JOINT && jprun[v])
                atomicAdd((unsigned long long *)&jbase[v][jpbin[v]], (unsigned long long)jprun[v]);
            a.E[w0 + v] = e[v];
            a.D[w0 + v] = d[v];
            a.M[w0 + v] = m[v];
        }
    }
    if (LDSHIST) {
        __syncthreads();
        // counts since the start (modulo 2^32; a wrap was carried already)
        for (uint32_t i = threadIdx.x; i <= N; i += blockDim.x) {
            const uint32_t c = hist[i];
            if (c != a.hist_preload)
                atomicAdd((unsigned long long *)&a.hist[i],
                          (unsigned long long)((int64_t)c - (int64_t)a.hist_preload));
        }
    }
}

template <int R, bool FP64, int KEYING, bool LDSHIST, int OBS, int V, int PD>
__global__ __launch_bounds__(V > 1 ? 512 : 1024) void k_mcs_lane(McsArgs a, uint32_t lds_w)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ lane_t<FP64> fde_tab[17];
    static_assert(sizeof(fde_tab) <= kStaticLds, "static LDS");
    lane_run<R, FP64, KEYING, LDSHIST, OBS, V, PD>(a, lds_w, (uint64_t)blockIdx.x * blockDim.x * V,
                                               lds, fde_tab);
}

// Four walkers per lane need one and a half wavefronts per SIMD to lead: 524 288
// walkers (two) at L = 72 590 attempts/ns against 335 with one walker per lane;
// 262 144 (one) 364 and 335 in the thermalisation, but 287 and 314 while the
// histogram is filled.
int lane_walkers(uint32_t L, uint64_t W, uint32_t cus)
{
    return L > 8 && W % 4 == 0 && W >= 1536ull * cus ? 4 : 1;
}

// A workgroup has the lanes that were asked for: four walkers per lane are built
// for up to 512, which leave a lane twice the registers that 1024 do (L = 64, 524 288
// walkers, 8192 attempts each: 7.7 ms with 256 or 512 lanes, 13.1 with 1024).
LaneShape lane_shape(uint32_t L, uint64_t W, uint32_t cus, int block)
{
    return {block, block <= 512 ? lane_walkers(L, W, cus) : 1};
}

bool lane_eligible(const McsArgs &a, int fp64, size_t lds_max)
{
    const size_t tsz = fp64 ? 8 : 4;
    return a.L % 2 == 0 && a.L >= 4 && (a.N + 1) * tsz + kStaticLds <= lds_max;
}

template <int R, bool FP64, int KEYING, int V, int PD>
static hipError_t launch_lane_v(hipStream_t st, int block, const Launch &cfg, const McsArgs &a)
{
    const size_t tsz = FP64 ? 8 : 4;
    const uint32_t lds_w = (uint32_t)(((a.N + 1) * tsz + 15) & ~(size_t)15);
    const size_t lds_h = (size_t)(a.N + 1) * 4;
    const bool hist_lds = lds_w + lds_h + kStaticLds <= cfg.lds_max;
    const size_t bytes = lds_w + (hist_lds ? lds_h : 0);
    const bool joint = a.joint != nullptr;
    void (*k)(McsArgs, uint32_t);
    if (hist_lds)
        k = joint ? k_mcs_lane<R, FP64, KEYING, true, 1, V, PD> : k_mcs_lane<R, FP64, KEYING, true, 0, V, PD>;
    else
        k = joint ? k_mcs_lane<R, FP64, KEYING, false, 1, V, PD>
                  : k_mcs_lane<R, FP64, KEYING, false, 0, V, PD>;
    hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)bytes);
    if (e != hipSuccess) return e;
    const uint64_t per = (uint64_t)block * V;
    hipLaunchKernelGGL(k, dim3((unsigned)((a.W + per - 1) / per)), dim3(block), bytes, st, a,
                       lds_w);
    return hipGetLastError();
}

template <int R, bool FP64, int KEYING>
static hipError_t launch_lane_r(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    const LaneShape sh = lane_shape(a.L, a.W, cfg.cus, cfg.block);
    return sh.walkers == 4 ? launch_lane_v<R, FP64, KEYING, 4, 4>(st, sh.lanes, cfg, a)
                           : launch_lane_v<R, FP64, KEYING, 1, 1>(st, sh.lanes, cfg, a);
}

hipError_t launch_mcs_lane(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    if (cfg.rounds == 10) {
        if (cfg.fp64)
            return cfg.keying ? launch_lane_r<10, true, 1>(st, cfg, a)
                              : launch_lane_r<10, true, 0>(st, cfg, a);
        return cfg.keying ? launch_lane_r<10, false, 1>(st, cfg, a)
                          : launch_lane_r<10, false, 0>(st, cfg, a);
    }
    if (cfg.fp64)
        return cfg.keying ? launch_lane_r<7, true, 1>(st, cfg, a)
                          : launch_lane_r<7, true, 0>(st, cfg, a);
    return cfg.keying ? launch_lane_r<7, false, 1>(st, cfg, a)
                      : launch_lane_r<7, false, 0>(st, cfg, a);
}

// ---------------------------------------------------------------------------
// batched engine, lane tiles: a persistent grid takes tiles of blockDim
// walkers of one instance from a shared counter, largest lattices first.
// ---------------------------------------------------------------------------
// VECS: every instance's tiles hold I->lane_vec = 2 or 4 walkers per lane (all
// L > 8, all walker counts multiples of 4); otherwise one.
template <bool FP64, bool VECS>
__global__ __launch_bounds__(VECS ? 256 : 1024, VECS ? 2 : 4) void k_batch_lane(BatchArgs b)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ uint32_t s_tile;
    __shared__ lane_t<FP64> fde_tab[17];
    static_assert(sizeof(s_tile) + sizeof(fde_tab) + 16 <= kStaticLds, "static LDS");
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
        const uint32_t lw = I->lane_lds_w;
        if constexpr (VECS) {
            if (I->lane_vec == 4) {
                if (I->lane_hist)
                    lane_run<7, FP64, 0, true, 0, 4, 4>(a, lw, tile.wbase, lds, fde_tab);
                else
                    lane_run<7, FP64, 0, false, 0, 4, 4>(a, lw, tile.wbase, lds, fde_tab);
            } else {
                if (I->lane_hist)
                    lane_run<7, FP64, 0, true, 0, 2, 4>(a, lw, tile.wbase, lds, fde_tab);
                else
                    lane_run<7, FP64, 0, false, 0, 2, 4>(a, lw, tile.wbase, lds, fde_tab);
            }
        } else {
            if (I->lane_hist)
                lane_run<7, FP64, 0, true, 0, 1, 1>(a, lw, tile.wbase, lds, fde_tab);
            else
                lane_run<7, FP64, 0, false, 0, 1, 1>(a, lw, tile.wbase, lds, fde_tab);
        }
    }
}

static void (*batch_lane_kernel(int fp64, int vecs))(BatchArgs)
{
    if (vecs) return fp64 ? k_batch_lane<true, true> : k_batch_lane<false, true>;
    return fp64 ? k_batch_lane<true, false> : k_batch_lane<false, false>;
}

hipError_t launch_batch_lane(hipStream_t st, int fp64, int vecs, const BatchArgs &b, uint32_t grid,
                             uint32_t block, size_t lds_bytes)
{
    hipLaunchKernelGGL(batch_lane_kernel(fp64, vecs), dim3(grid), dim3(block), lds_bytes, st, b);
    return hipGetLastError();
}

hipError_t batch_static_lds(int fp64, int team, int vecs, size_t *bytes)
{
    hipFuncAttributes at;
    const hipError_t e = hipFuncGetAttributes(
        &at, team ? batch_team_function(fp64) : (const void *)batch_lane_kernel(fp64, vecs));
    if (e == hipSuccess) *bytes = at.sharedSizeBytes;
    return e;
}

hipError_t prepare_batch_lane(int fp64, int vecs, size_t lds_bytes)
{
    return hipFuncSetAttribute((const void *)batch_lane_kernel(fp64, vecs),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
}

}  // namespace muca
