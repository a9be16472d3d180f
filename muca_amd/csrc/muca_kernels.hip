// muca_kernels.hip -- HIP kernels of libmuca for gfx950 (MI355X).
//
// Update-kernel design: every walker is a strict serial Metropolis chain
// (fixed site order, acceptance depends on the running D = sum s^2), so the
// parallelism is across walkers: one lane per walker, walkers interleaved
// site-major in HBM so that each site access of a wavefront is one
// contiguous 64-byte segment.  The D histogram is privatised per workgroup
// in LDS (uint32) and flushed to HBM with 64-bit atomics.  Nothing in the
// update is a dense contraction, so there is no MFMA here.
#include "kernels.h"
#include "moments.h"

#include "acclog.h"
#include "philox.h"

namespace muca {

#define MUCA_CTR3 0xBADC0DEDu

// ---------------------------------------------------------------------------
// initial lattice (muca_delta_multigpu.cu:340-351; produce2_multigpu.cu:126-138)
// A thread draws one Philox block (four sites) for each of V walkers and
// stores a dword per site (V = 4, where W and the lattice are 4-aligned) or a
// byte.  Bound by the stores and the Philox products alike: L = 72, 524 288
// walkers 1.49 ms against 2.36 ms with one walker per thread and byte stores;
// L = 256, 16 384 walkers 0.77 against 1.04 ms.
// u = m 2^-24 (m = 1 | r >> 8) is compared as an integer: u < 1/3 iff
// m <= 5592405, u < 2/3 iff m <= 11184810, u < p iff m < ceil(p 2^24), all
// exact because p 2^24 is.
// ---------------------------------------------------------------------------
// strat_W > 0 selects the stratified start (no counterpart in the reference):
// walker wid of strat_W gets a nonzero spin with probability
// p = (wid + 1/2) / strat_W, sign - for u < p/2 and + for p/2 <= u < p, from
// the same Philox stream, so that the walkers start spread over D = 0..N.
template <int R, int V>
__global__ __launch_bounds__(256) void k_init_lattice(int8_t *lat, uint64_t W, uint32_t N,
                                                      int keying, uint32_t mm, uint32_t gpu,
                                                      uint32_t seed, uint32_t w_offset,
                                                      uint32_t strat_W)
{
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t nblk = (N + 3) / 4, groups = W / V;
    if (t >= groups * nblk) return;
    const uint32_t blk = (uint32_t)(t / groups);
    const uint64_t w = (t - blk * groups) * V;
    uint32_t out[4] = {};   // site 4 blk + j, walker w + v in byte v
#pragma unroll
    for (int v = 0; v < V; v++) {
        const uint32_t wid = w_offset + (uint32_t)w + v;
        philox4 r;
        if (keying == 0)
            r = philox4x32<R>(gpu * 2u + blk + 1u, seed, 0xBADCAB1Eu, 0xBADC0DEDu,
                              10u * wid + mm * 2u, 0xdecafbadu);
        else
            r = philox4x32<R>(gpu * 1000u, seed, blk + 1u, 0xBADCAFE3u, wid * 10u, 0xdecafbadu);
        uint32_t below_m = 0, below_p = 0;
        if (strat_W) {
            const double p = ((double)wid + 0.5) / (double)strat_W;
            below_m = (uint32_t)ceil(0.5 * p * 0x1p24);
            below_p = (uint32_t)ceil(p * 0x1p24);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t m = 1u | (r.v[j] >> 8);
            const int32_t sv = strat_W ? (m < below_p ? (m < below_m ? -1 : 1) : 0)
                                       : (int32_t)(m <= 5592405u) + (int32_t)(m <= 11184810u) - 1;
            out[j] |= ((uint32_t)sv & 0xffu) << (8 * v);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t site = 4u * blk + (uint32_t)j;
        if (site < N) {
            int8_t *q = lat + (uint64_t)site * W + w;
            if (V == 4)
                *(uint32_t *)q = out[j];
            else
                *q = (int8_t)out[j];
        }
    }
}

template <int R>
static void launch_init_r(hipStream_t st, int8_t *lat, uint64_t W, uint32_t N, int keying,
                          uint32_t mm, uint32_t gpu, uint32_t seed, uint32_t w_offset,
                          uint32_t strat_W)
{
    const bool vec = W % 4 == 0 && ((uintptr_t)lat & 3) == 0;
    const uint64_t total = (vec ? W / 4 : W) * ((N + 3) / 4);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (vec)
        hipLaunchKernelGGL((k_init_lattice<R, 4>), grid, dim3(256), 0, st, lat, W, N, keying, mm,
                           gpu, seed, w_offset, strat_W);
    else
        hipLaunchKernelGGL((k_init_lattice<R, 1>), grid, dim3(256), 0, st, lat, W, N, keying, mm,
                           gpu, seed, w_offset, strat_W);
}

hipError_t launch_init_lattice(hipStream_t st, int8_t *lat, uint64_t W, uint32_t N,
                               int keying, int rounds, uint32_t mm, uint32_t gpu,
                               uint32_t seed, uint32_t w_offset, uint32_t strat_W)
{
    if (rounds == 10)
        launch_init_r<10>(st, lat, W, N, keying, mm, gpu, seed, w_offset, strat_W);
    else
        launch_init_r<7>(st, lat, W, N, keying, mm, gpu, seed, w_offset, strat_W);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// per-walker E_J, D, M (muca_delta_multigpu.cu:69-83,548-571; produce2_multigpu.cu:66-89)
// ---------------------------------------------------------------------------
// The lattice is read once: the kernel is bound by HBM.  A lane holds four
// walkers in the bytes of a dword (one walker where W or the lattice is not
// 4-aligned), 32 lanes read a whole 128-byte line, and each of a workgroup's
// 32 parts walks down strips of kStrip columns with the row above in
// registers, so that a site is loaded once (and once more as the right
// neighbour of the strip before: 9/8 of the lattice).  A bond is counted once,
// as right and lower neighbour; spins are 0x00, 0x01, 0xFF, so a product of
// two is nonzero iff bit 0 of their AND is set and then negative iff bit 1 of
// their XOR is.  Counts are kept in bytes and widened every kFlush rows.
// L = 72, 524 288 walkers: 0.62 ms (4.4 TB/s of lattice) against 24.5 ms for
// sixteen lanes per walker that gathered bytes through the neighbour table;
// L = 256, 16 384 walkers: 0.37 ms against 10.1 ms; 4096 walkers at L = 72:
// 33 against 269 us.
constexpr int kStateParts = 32, kStateLanes = 32, kStrip = 8, kFlush = 8;

template <bool VEC>
__device__ __forceinline__ void state_tile(uint32_t tile, const int8_t *lat, uint64_t W, uint32_t L,
                                           int32_t *E, int32_t *D, int32_t *M)
{
    constexpr int V = VEC ? 4 : 1;                 // walkers per lane
    constexpr uint32_t kOne = 0x01010101u;
    __shared__ int32_t part[3][kStateParts / 2][kStateLanes * V];
    const uint32_t lane = threadIdx.x % kStateLanes, p = threadIdx.x / kStateLanes;
    const uint64_t w = ((uint64_t)tile * kStateLanes + lane) * V;
    int32_t sum[3][V] = {};                        // bonds, D, M
    if (w < W) {
        const uint8_t *base = (const uint8_t *)lat + w;
        auto at = [&](uint32_t y, uint32_t x) -> uint32_t {
            const uint8_t *q = base + (uint64_t)(y * L + x) * W;
            return VEC ? *(const uint32_t *)q : (uint32_t)*q;
        };
        const uint32_t strips = (L + kStrip - 1) / kStrip;
        const uint32_t segs = strips < kStateParts ? kStateParts / strips : 1;
        for (uint32_t it = p; it < strips * segs; it += kStateParts) {
            const uint32_t strip = it % strips, seg = it / strips;
            const uint32_t x0 = strip * kStrip, n = min((uint32_t)kStrip, L - x0);
            const uint32_t y0 = (uint32_t)((uint64_t)L * seg / segs);
            const uint32_t y1 = (uint32_t)((uint64_t)L * (seg + 1) / segs);
            if (y0 == y1) continue;
            const uint32_t xn = x0 + n == L ? 0 : x0 + n;   // the column right of the strip
            // columns past a narrow last strip repeat its last one on load
            // and count nothing
            uint32_t cur[kStrip], right = at(y0, xn);
#pragma unroll
            for (int c = 0; c < kStrip; c++) cur[c] = at(y0, x0 + min((uint32_t)c, n - 1));
            uint32_t nz = 0, ng = 0, ds = 0, ms = 0, rows = 0;
            for (uint32_t y = y0; y < y1; y++) {
                const uint32_t yn = y + 1 == L ? 0 : y + 1;
                uint32_t nxt[kStrip];
#pragma unroll
                for (int c = 0; c < kStrip; c++) nxt[c] = at(yn, x0 + min((uint32_t)c, n - 1));
                const uint32_t rn = at(yn, xn);
#pragma unroll
                for (int c = 0; c < kStrip; c++) {
                    const uint32_t s = (uint32_t)c < n ? cur[c] : 0u;
                    const uint32_t r = (uint32_t)c + 1 < n ? cur[(c + 1) % kStrip] : right;
                    const uint32_t br = s & r & kOne, bu = s & nxt[c] & kOne;
                    nz += br + bu;
                    ng += (((s ^ r) >> 1) & br) + (((s ^ nxt[c]) >> 1) & bu);
                    ds += s & kOne;
                    ms += (s >> 1) & kOne;
                    cur[c] = nxt[c];
                }
                right = rn;
                if (++rows == kFlush || y + 1 == y1) {
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        auto byte = [&](uint32_t q) { return (int32_t)((q >> (8 * v)) & 0xffu); };
                        sum[0][v] += byte(nz) - 2 * byte(ng);
                        sum[1][v] += byte(ds);
                        sum[2][v] += byte(ds) - 2 * byte(ms);
                    }
                    nz = ng = ds = ms = rows = 0;
                }
            }
        }
    }
    // two parts per wavefront, then the workgroup's sixteen wavefronts
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int32_t t = sum[k][v] + __shfl_xor(sum[k][v], kStateLanes);
            if (p % 2 == 0) part[k][p / 2][lane * V + v] = t;
        }
    __syncthreads();
    const uint32_t i = threadIdx.x;
    const uint64_t wi = (uint64_t)tile * kStateLanes * V + i;
    if (i < kStateLanes * V && wi < W) {
        int32_t t[3] = {};
#pragma unroll
        for (int k = 0; k < 3; k++)
            for (int q = 0; q < kStateParts / 2; q++) t[k] += part[k][q][i];
        E[wi] = -t[0];
        D[wi] = t[1];
        if (M) M[wi] = t[2];
    }
}

template <bool VEC>
__global__ __launch_bounds__(kStateParts *kStateLanes) void k_state(const int8_t *lat, uint64_t W,
                                                                    uint32_t L, int32_t *E,
                                                                    int32_t *D, int32_t *M)
{
    state_tile<VEC>(blockIdx.x, lat, W, L, E, D, M);
}

// All instances of a batch, blockIdx.y the instance: one problem of 4096
// walkers has 32 workgroups for 256 compute units (96 problems, L = 32 .. 128:
// 0.56 ms against 3.4 one after the other).
__global__ __launch_bounds__(kStateParts *kStateLanes) void k_state_batch(const BatchInst *inst,
                                                                          const int8_t *lat,
                                                                          int32_t *E, int32_t *D,
                                                                          int32_t *M)
{
    const BatchInst &I = inst[blockIdx.y];
    const int8_t *l = lat + I.lat_off;
    const uint64_t W = I.W, st = I.st_off;
    const bool vec = W % 4 == 0 && ((uintptr_t)l & 3) == 0;
    if ((uint64_t)blockIdx.x * kStateLanes * (vec ? 4 : 1) >= W) return;   // the whole workgroup
    if (vec)
        state_tile<true>(blockIdx.x, l, W, I.L, E + st, D + st, M + st);
    else
        state_tile<false>(blockIdx.x, l, W, I.L, E + st, D + st, M + st);
}

hipError_t launch_state_batch(hipStream_t st, const BatchInst *inst, uint32_t n, uint32_t tiles,
                              const int8_t *lat, int32_t *E, int32_t *D, int32_t *M)
{
    for (uint32_t i = 0; i < n; i += 32768)   // the grid's second dimension is 16 bits
        hipLaunchKernelGGL(k_state_batch, dim3(tiles, n - i < 32768 ? n - i : 32768),
                           dim3(kStateParts * kStateLanes), 0, st, inst + i, lat, E, D, M);
    return hipGetLastError();
}

uint32_t state_tiles(uint64_t W, const int8_t *lat)
{
    const uint64_t per = kStateLanes * (W % 4 == 0 && ((uintptr_t)lat & 3) == 0 ? 4 : 1);
    return (uint32_t)((W + per - 1) / per);
}

// A few kilobytes between pinned host memory and the device as part of the
// stream's work: a blocking copy of its own costs more than the data does (257
// bins: a run that returns the histogram 42 -> 32 us, setting ln W 30 -> 15 us).
__global__ __launch_bounds__(256) void k_copy(uint32_t *dst, const uint32_t *src, uint32_t words)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) dst[i] = src[i];
}

hipError_t launch_copy(hipStream_t st, void *dst, const void *src, uint64_t bytes)
{
    if (bytes > 65536) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, st);
    const uint32_t words = (uint32_t)(bytes / 4);
    hipLaunchKernelGGL(k_copy, dim3((words + 255) / 256), dim3(256), 0, st, (uint32_t *)dst,
                       (const uint32_t *)src, words);
    return hipGetLastError();
}

hipError_t launch_state(hipStream_t st, const int8_t *lat, uint64_t W, uint32_t L, int32_t *E,
                        int32_t *D, int32_t *M)
{
    const bool vec = W % 4 == 0 && ((uintptr_t)lat & 3) == 0;
    const dim3 grid(state_tiles(W, lat)), block(kStateParts * kStateLanes);
    if (vec)
        hipLaunchKernelGGL(k_state<true>, grid, block, 0, st, lat, W, L, E, D, M);
    else
        hipLaunchKernelGGL(k_state<false>, grid, block, 0, st, lat, W, L, E, D, M);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_differ(const int32_t *a, const int32_t *b, uint64_t n,
                                                uint32_t *flag)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n && a[i] != b[i]) *flag = 1u;
}

hipError_t launch_differ(hipStream_t st, const int32_t *a, const int32_t *b, uint64_t n,
                         uint32_t *flag)
{
    hipLaunchKernelGGL(k_differ, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, b, n, flag);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The update kernel, reference site order from tables (any L).
// Per walker (muca_delta_multigpu.cu:735-829; produce2_multigpu.cu:401-496):
//   keys  weight : k1 = {2w, 0xdecafbad}, k3 = {2w+50000, 0x11cafead}
//         produce: k1 = {w, 0xdecafbad},  k3 = {w+40000, 0xdecafead}
//   ctr = {++c0, seed, iter, 0xBADC0DED} once per four attempts, c0 shared
//   by the therm and production phases, attempt index restarting at 0.
//   step  = +1 if r3 < 2^31 (u01fixedpt<float>(r3) < 0.5) else -1, new in {-1,0,1}
//   dE    = -(new - old) * (sum of the four neighbours)   [equals the
//           reference's ((old==0) + old*(new-old)) * (-tmp) * sum for every
//           old, new in {-1,0,1}, tmp being its temporary write]
//   diff  = (T)(-dE*beta) + lnW[D+dDel] - lnW[D]   (T = float | double)
//   accept iff diff >= 0 or acclog(r1) < diff
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T lnw_at(const McsArgs &a, int32_t i);
template <>
__device__ __forceinline__ float lnw_at<float>(const McsArgs &a, int32_t i)
{
    return a.lnw32[i];
}
template <>
__device__ __forceinline__ double lnw_at<double>(const McsArgs &a, int32_t i)
{
    return a.lnw64[i];
}

// n entries of D histogram bin d: LDS (uint32, a workgroup adds at most
// block * nup < 2^32 to a bin) or HBM
template <bool LDSHIST>
__device__ __forceinline__ void hist_add(const McsArgs &a, uint32_t *lds_hist, int32_t d,
                                         uint64_t n)
{
    if (n == 0) return;
    if (LDSHIST)
        atomicAdd(&lds_hist[d], (uint32_t)n);
    else
        atomicAdd((unsigned long long *)&a.hist[d], (unsigned long long)n);
}

// OBS: 0 = D histogram only; 1 = joint H(D,M) per walker block
// (produce2_multigpu.cu:489); 2 = exact per-D moments per walker block
template <int R, bool FP64, int KEYING, bool LDSHIST, int OBS>
__global__ __launch_bounds__(256) void k_mcs_generic(McsArgs a)
{
    typedef typename std::conditional<FP64, double, float>::type T;
    extern __shared__ uint32_t lds_hist[];
    const uint32_t nbins = a.N + 1;
    if (LDSHIST) {
        for (uint32_t b = threadIdx.x; b < nbins; b += blockDim.x) lds_hist[b] = 0;
        __syncthreads();
    }
    const uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w < a.W) {
        const uint32_t wid = a.w_offset + (uint32_t)w;
        const uint32_t k1a = KEYING == 0 ? 2u * wid : wid;
        const uint32_t k1b = 0xdecafbadu;
        const uint32_t k3a = KEYING == 0 ? 2u * wid + 50000u : wid + 40000u;
        const uint32_t k3b = KEYING == 0 ? 0x11cafeadu : 0xdecafeadu;
        int8_t *s = a.lat + w;
        // walker counts are 32-bit (muca_params.walkers): site * W is one
        // 32 x 32 -> 64-bit multiply-add
        const uint32_t W = (uint32_t)a.W;
        int32_t e = a.E[w], d = a.D[w], m = a.M[w];
        uint64_t *jbase = nullptr;
        if (OBS == 1) jbase = a.joint + (w / a.block_walkers) * a.joint_stride;
        // per-D moment arrays of this walker's block, mstride words apart
        const uint64_t mstride = (uint64_t)a.N + 1;
        uint64_t *mbase = nullptr;
        if (OBS == 2) mbase = a.moms + (w / a.block_walkers) * (uint64_t)kMomWords * mstride;
        // the current D's moment sums and the previous D's: a walker that
        // steps back to the D it came from flushes nothing
        MomRun run{}, prev{};
        run.d = -1;
        prev.d = -1;
        // Histogram entries are counted in registers while the bin stays the
        // same (D, or (D, M) for the joint histogram, changes only on some
        // accepted moves) and added with one atomic when it changes: the
        // integer sums are the same, the atomics far fewer.
        // The bin in use and the one before it are both kept, so a walker
        // stepping back and forth between two bins adds nothing until it
        // reaches a third.
        uint64_t hrun = 0, hprun = 0, jrun = 0, jprun = 0;
        int32_t hbin = 0, hpbin = 0;
        int64_t jbin = 0, jpbin = 0;
        // Attempt t+1's site, neighbours and spins are loaded before attempt t
        // computes, so their memory latency overlaps attempt t's ln W gathers,
        // store and histogram atomic.  That is exact when attempt t's site is
        // neither attempt t+1's site nor one of its neighbours: for even L >= 4
        // consecutive sites of the order 0, 2, .., N-2, 1, 3, .., N-1 differ by
        // 2 (or are N-2 -> 1 and N-1 -> 0), never by 0, +-1, +-L, 1-L, L-1 or
        // N-L modulo N.  Other L load after the store.
        const bool ahead = (a.L % 2 == 0) && a.L >= 4;
        uint32_t c0 = 0;
        for (int phase = 0; phase < 2; phase++) {
            const uint64_t n = phase ? a.nup : a.therm;
            if (n == 0) continue;
            uint32_t pos = 0;
            // spins of the attempt about to run: site, and sum of neighbours
            uint32_t idx = a.order[0];
            int32_t old_s = s[(uint64_t)idx * W];
            int32_t nsum;
            {
                const uint32_t *nv = a.naver + 4u * idx;
                nsum = s[(uint64_t)nv[0] * W] + s[(uint64_t)nv[1] * W] + s[(uint64_t)nv[2] * W] +
                       s[(uint64_t)nv[3] * W];
            }
            philox4 r1{}, r3{};
            for (uint64_t i = 0; i < n; i++) {
                if ((i & 3) == 0) {
                    ++c0;
                    r1 = philox4x32<R>(c0, a.seed, a.iter, MUCA_CTR3, k1a, k1b);
                    r3 = philox4x32<R>(c0, a.seed, a.iter, MUCA_CTR3, k3a, k3b);
                }
                const uint32_t j = (uint32_t)(i & 3);
                const uint32_t u1 = j == 0 ? r1.v[0] : j == 1 ? r1.v[1] : j == 2 ? r1.v[2] : r1.v[3];
                const uint32_t u3 = j == 0 ? r3.v[0] : j == 1 ? r3.v[1] : j == 2 ? r3.v[2] : r3.v[3];
                const bool more = i + 1 < n;
                const uint32_t npos = (pos + 1 == a.N) ? 0 : pos + 1;
                uint32_t nidx = 0;
                int32_t nold = 0, nnsum = 0;
                if (ahead && more) {
                    nidx = a.order[npos];
                    const uint32_t *nv = a.naver + 4u * nidx;
                    nold = s[(uint64_t)nidx * W];
                    nnsum = s[(uint64_t)nv[0] * W] + s[(uint64_t)nv[1] * W] +
                            s[(uint64_t)nv[2] * W] + s[(uint64_t)nv[3] * W];
                }
                int32_t new_s = old_s + (u3 < 0x80000000u ? 1 : -1);
                new_s = new_s == 2 ? -1 : (new_s == -2 ? 1 : new_s);
                const int32_t dE = -(new_s - old_s) * nsum;
                const int32_t dDel = new_s * new_s - old_s * old_s;
                // D stays in [0, N] for a consistent (lattice, D) pair; the
                // clamp keeps every table access in bounds for any input
                const int32_t dn = min(max(d + dDel, 0), (int32_t)a.N);
                T diff = (T)(-(double)dE * a.beta);
                diff = diff + lnw_at<T>(a, dn);
                diff = diff - lnw_at<T>(a, d);
                // log(u) < diff (diff >= 0 included: log(u) < 0), screened with
                // the hardware log: exact unless diff lies within the proven
                // error band of la, where the correctly rounded log decides
                const float la = acclog_fast_u01(u1);
                const float band = acclog_fast_band(la);
                bool acc = (T)(la + band) < diff;
                const bool amb = !acc && !((T)(la - band) >= diff);
                if (__builtin_amdgcn_ballot_w64(amb)) {
                    if (amb) acc = (T)acclog_u01(u1) < diff;
                }
                if (acc) {
                    s[(uint64_t)idx * W] = (int8_t)new_s;
                    e += dE;
                    d = dn;
                    m += new_s - old_s;
                }
                if (phase) {
                    // with per-D moments the D histogram is the blocks' S0,
                    // summed after the launch (k_hist_from_moments)
                    if (OBS != 2) {
                        if (d != hbin) {
                            if (d == hpbin && hprun) {
                                const uint64_t tr = hrun;
                                hrun = hprun;
                                hprun = tr;
                                hpbin = hbin;
                            } else {
                                hist_add<LDSHIST>(a, lds_hist, hpbin, hprun);
                                hprun = hrun;
                                hpbin = hbin;
                                hrun = 0;
                            }
                            hbin = d;
                        }
                        hrun++;
                    }
                    if (OBS == 1) {
                        const int64_t mm = min(max((int64_t)m, -(int64_t)d), (int64_t)d);
                        const int64_t jb = (mm + (int64_t)d * d + 2 * (int64_t)d) / 2;
                        if (jb != jbin) {
                            if (jb == jpbin && jprun) {
                                const uint64_t tr = jrun;
                                jrun = jprun;
                                jprun = tr;
                                jpbin = jbin;
                            } else {
                                if (jprun) atomicAdd((unsigned long long *)&jbase[jpbin], jprun);
                                jprun = jrun;
                                jpbin = jbin;
                                jrun = 0;
                            }
                            jbin = jb;
                        }
                        jrun++;
                    }
                    if (OBS == 2) {
                        if (d != run.d) {
                            if (d == prev.d) {
                                const MomRun t = run;
                                run = prev;
                                prev = t;
                            } else {
                                mom_flush(prev, mbase, mstride);
                                prev = run;
                                run = MomRun{};
                                run.d = d;
                            }
                        }
                        mom_add(run, min(max(m, -d), d));
                    }
                }
                if (more) {
                    if (!ahead) {
                        nidx = a.order[npos];
                        const uint32_t *nv = a.naver + 4u * nidx;
                        nold = s[(uint64_t)nidx * W];
                        nnsum = s[(uint64_t)nv[0] * W] + s[(uint64_t)nv[1] * W] +
                                s[(uint64_t)nv[2] * W] + s[(uint64_t)nv[3] * W];
                    }
                    idx = nidx;
                    old_s = nold;
                    nsum = nnsum;
                }
                pos = npos;
            }
        }
        hist_add<LDSHIST>(a, lds_hist, hbin, hrun);
        hist_add<LDSHIST>(a, lds_hist, hpbin, hprun);
        if (OBS == 1 && jrun) atomicAdd((unsigned long long *)&jbase[jbin], jrun);
        if (OBS == 1 && jprun) atomicAdd((unsigned long long *)&jbase[jpbin], jprun);
        if (OBS == 2) {
            mom_flush(run, mbase, mstride);
            mom_flush(prev, mbase, mstride);
        }
        a.E[w] = e;
        a.D[w] = d;
        a.M[w] = m;
    }
    if (LDSHIST) {
        __syncthreads();
        for (uint32_t b = threadIdx.x; b < nbins; b += blockDim.x) {
            const uint32_t c = lds_hist[b];
            if (c) atomicAdd((unsigned long long *)&a.hist[b], (unsigned long long)c);
        }
    }
}

template <int R, bool FP64, int KEYING, bool LDSHIST, int OBS>
static void launch_generic_v(hipStream_t st, dim3 grid, int block, size_t lds, const McsArgs &a)
{
    auto k = k_mcs_generic<R, FP64, KEYING, LDSHIST, OBS>;
    if (LDSHIST)
        hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds);
    hipLaunchKernelGGL(k, grid, dim3(block), LDSHIST ? lds : 0, st, a);
}

template <int R, bool FP64, int KEYING, bool LDSHIST>
static void launch_generic_h(hipStream_t st, dim3 grid, int block, size_t lds, const McsArgs &a)
{
    // the produce path computes in FP64, so only FP64 builds the moments variant
    if (a.joint)
        launch_generic_v<R, FP64, KEYING, LDSHIST, 1>(st, grid, block, lds, a);
    else if (FP64 && a.moms)
        launch_generic_v<R, FP64, KEYING, LDSHIST, FP64 ? 2 : 0>(st, grid, block, lds, a);
    else
        launch_generic_v<R, FP64, KEYING, LDSHIST, 0>(st, grid, block, lds, a);
}

// D histogram of a launch that kept per-D moments: hist[D] = sum over blocks
// of S0[D] (every production attempt adds 1 to S0 of its walker's block)
__global__ __launch_bounds__(256) void k_hist_from_moments(const uint64_t *moms, uint32_t N,
                                                           uint32_t blocks, uint64_t *hist)
{
    const uint64_t nb = (uint64_t)N + 1;
    const uint64_t D = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (D >= nb) return;
    uint64_t h = 0;
    for (uint32_t b = 0; b < blocks; b++) h += moms[(uint64_t)b * kMomWords * nb + D];
    hist[D] = h;
}

template <int R, bool FP64, int KEYING>
static hipError_t launch_generic_r(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    const int block = (cfg.block > 0 && cfg.block <= 256) ? cfg.block : 256;   // launch bounds
    const dim3 grid((unsigned)((a.W + block - 1) / block));
    const size_t lds = (size_t)(a.N + 1) * sizeof(uint32_t);
    // uint32 LDS bins cannot overflow: a workgroup adds at most block * nup
    const bool lds_ok = lds <= cfg.lds_max && (uint64_t)block * a.nup < (1ull << 32);
    if (lds_ok)
        launch_generic_h<R, FP64, KEYING, true>(st, grid, block, lds, a);
    else
        launch_generic_h<R, FP64, KEYING, false>(st, grid, block, lds, a);
    if (FP64 && a.moms && !a.joint && a.nup > 0)
        return launch_hist_from_moments(st, a.moms, a.N, a.joint_blocks, a.hist);
    return hipGetLastError();
}

hipError_t launch_hist_from_moments(hipStream_t st, const uint64_t *moms, uint32_t N,
                                    uint32_t blocks, uint64_t *hist)
{
    const uint64_t nb = (uint64_t)N + 1;
    hipLaunchKernelGGL(k_hist_from_moments, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, st,
                       moms, N, blocks, hist);
    return hipGetLastError();
}

template <bool FP64, int KEYING>
static hipError_t launch_generic_k(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    return cfg.rounds == 10 ? launch_generic_r<10, FP64, KEYING>(st, cfg, a)
                            : launch_generic_r<7, FP64, KEYING>(st, cfg, a);
}

static hipError_t launch_mcs_generic(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    if (cfg.fp64)
        return cfg.keying == 0 ? launch_generic_k<true, 0>(st, cfg, a)
                               : launch_generic_k<true, 1>(st, cfg, a);
    return cfg.keying == 0 ? launch_generic_k<false, 0>(st, cfg, a)
                           : launch_generic_k<false, 1>(st, cfg, a);
}

hipError_t launch_mcs(hipStream_t st, const Launch &cfg, const McsArgs &a)
{
    if (a.W == 0 || (a.therm == 0 && a.nup == 0)) return hipSuccess;
    // per-D moments: the generic kernel, or (FP64) the team kernel
    const bool moments = a.moms != nullptr && a.joint == nullptr;
    if (cfg.kernel == 2 && (!moments || cfg.fp64)) {
        TeamLayout lay{};
        if (team_layout(a, cfg.fp64, cfg.lds_max, cfg.cus, lay)) return launch_mcs_team(st, cfg, a, lay);
    }
    if (cfg.kernel == 3 && !moments && lane_eligible(a, cfg.fp64, cfg.lds_max))
        return launch_mcs_lane(st, cfg, a);
    // a context of the team kernel whose launch does not fit it (odd L, a
    // thermalisation of production with moments: its histogram takes the lattices'
    // LDS) has no block of its own
    Launch g = cfg;
    if (cfg.kernel == 2 && cfg.block == 256 && cfg.cus) g.block = generic_block(a.W, cfg.cus);
    return launch_mcs_generic(st, g, a);
}

// ---------------------------------------------------------------------------
// acceptance log evaluated on the device (self-check)
// ---------------------------------------------------------------------------
__global__ void k_acclog(uint32_t k0, uint32_t n, float *out)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) out[t] = acclog_u01((k0 + t) << 9);
}

hipError_t launch_acclog(hipStream_t st, uint32_t k0, uint32_t n, float *out)
{
    hipLaunchKernelGGL(k_acclog, dim3((n + 255) / 256), dim3(256), 0, st, k0, n, out);
    return hipGetLastError();
}

__global__ void k_acclog_fast(uint32_t k0, uint32_t n, float *out)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) out[t] = acclog_fast_u01((k0 + t) << 9);
}

hipError_t launch_acclog_fast(hipStream_t st, uint32_t k0, uint32_t n, float *out)
{
    hipLaunchKernelGGL(k_acclog_fast, dim3((n + 255) / 256), dim3(256), 0, st, k0, n, out);
    return hipGetLastError();
}

__global__ void k_acclog_screen(uint32_t k0, uint32_t n, float *out)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float thi = acclog_screen((k0 + t) << 9);
    out[t] = thi;
    out[(uint64_t)n + t] = acclog_screen_lim(thi);
}

hipError_t launch_acclog_screen(hipStream_t st, uint32_t k0, uint32_t n, float *out)
{
    hipLaunchKernelGGL(k_acclog_screen, dim3((n + 255) / 256), dim3(256), 0, st, k0, n, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// produce path: exact per-D moments (S0, S1, limb words of S2 and S4) -> FP64
// in the layout of k_joint_moments' output
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_moments_fp64(const uint64_t *moms, uint32_t N,
                                                      uint32_t blocks, double *mom,
                                                      uint32_t *range_flag)
{
    const uint64_t nb = (uint64_t)N + 1;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nb * blocks) return;
    const uint64_t b = t / nb, D = t - b * nb;
    const uint64_t *s = moms + b * kMomWords * nb + D;
    double *o = mom + b * 4 * nb + D;
    const double two32 = 4294967296.0, two64 = 18446744073709551616.0;
    if (s[0] >> 32) atomicOr(range_flag, 1u);   // limb words may have wrapped
    o[0] = (double)s[0];
    o[nb] = (double)s[nb];
    o[2 * nb] = (double)s[4 * nb] * two64 + ((double)s[3 * nb] * two32 + (double)s[2 * nb]);
    o[3 * nb] = (double)s[7 * nb] * two64 + ((double)s[6 * nb] * two32 + (double)s[5 * nb]);
}

hipError_t launch_moments_fp64(hipStream_t st, const uint64_t *moms, uint32_t N,
                               uint32_t blocks, double *mom, uint32_t *range_flag)
{
    const uint64_t n = ((uint64_t)N + 1) * blocks;
    hipLaunchKernelGGL(k_moments_fp64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       moms, N, blocks, mom, range_flag);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// produce path: joint H(D,M) -> per-D moments, one wavefront per (block, D);
// lanes stride over m so the reads of a shell are contiguous.
// mom layout: [block][4][N+1] with S0 = sum H, S1 = sum |m| H, S2 = sum m^2 H,
// S4 = sum m^4 H (FP64).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_joint_moments(const uint64_t *joint, uint32_t N,
                                                       uint64_t stride, uint32_t blocks,
                                                       double *mom)
{
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / 64u;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t nb = N + 1;
    if (wave >= nb * blocks) return;
    const uint32_t b = wave / (uint32_t)nb;
    const uint64_t D = wave % nb;
    const uint64_t *h = joint + b * stride + (D * D + D) / 2;   // m = -D at offset 0
    double a0 = 0, a1 = 0, a2 = 0, a4 = 0;
    for (uint64_t j = lane; j <= D; j += 64) {
        const double c = (double)h[j];
        const double am = fabs((double)(2 * (int64_t)j - (int64_t)D));
        const double m2 = am * am;
        a0 += c;
        a1 += am * c;
        a2 += m2 * c;
        a4 += m2 * m2 * c;
    }
    for (int off = 32; off > 0; off >>= 1) {
        a0 += __shfl_down(a0, off, 64);
        a1 += __shfl_down(a1, off, 64);
        a2 += __shfl_down(a2, off, 64);
        a4 += __shfl_down(a4, off, 64);
    }
    if (lane == 0) {
        double *o = mom + (uint64_t)b * 4 * nb;
        o[D] = a0;
        o[nb + D] = a1;
        o[2 * nb + D] = a2;
        o[3 * nb + D] = a4;
    }
}

hipError_t launch_joint_moments(hipStream_t st, const uint64_t *joint, uint32_t N,
                                uint64_t stride, uint32_t blocks, double *mom)
{
    const uint64_t waves = (uint64_t)(N + 1) * blocks;
    hipLaunchKernelGGL(k_joint_moments, dim3((unsigned)((waves * 64 + 255) / 256)), dim3(256), 0,
                       st, joint, N, stride, blocks, mom);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// reweighting (produce2_multigpu.cu:295-297,391-400,498-518), one workgroup
// per (delta, block): shift = max_D(-lnW_D - beta*delta*D), then
// Z = sum_D exp(-beta*delta*D - lnW_D - shift) S0_D, A_k likewise with S_k.
// Three planes of ndelta*blocks values: out[k*plane + id*blocks + b] with
// k = 0, 1, 2 for <|M|>, chi, Binder cumulant.
// ---------------------------------------------------------------------------
__device__ static double block_reduce_sum(double v, double *sh)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int wv = threadIdx.x / 64, ln = threadIdx.x & 63;
    __syncthreads();
    if (ln == 0) sh[wv] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x / 64); i++) t += sh[i];
    return t;
}

__device__ static double block_reduce_max(double v, double *sh)
{
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    const int wv = threadIdx.x / 64, ln = threadIdx.x & 63;
    __syncthreads();
    if (ln == 0) sh[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = sh[0];
        for (int i = 1; i < (int)(blockDim.x / 64); i++) t = fmax(t, sh[i]);
        sh[8] = t;
    }
    __syncthreads();
    return sh[8];
}

__global__ __launch_bounds__(256) void k_reweight(const double *mom, const double *lnw,
                                                  uint32_t N, uint32_t blocks, double beta,
                                                  const double *deltas, double *out)
{
    __shared__ double sh[16];
    const uint32_t id = blockIdx.x / blocks, b = blockIdx.x % blocks;
    const double bd = beta * deltas[id];
    const uint64_t nb = N + 1;
    // The shift cancels in every ratio; the reference takes it over all bins
    // (produce2_multigpu.cu:391-400), which underflows every visited bin to 0
    // (and the ratios to 0/0) when the maximum sits at an unvisited D.  The
    // maximum over the block's visited bins gives the same ratios wherever
    // the reference's are finite, and finite ratios wherever a bin is visited;
    // unvisited bins are left out of the sums (their terms are 0 x exp(...)).
    const double *S = mom + (uint64_t)b * 4 * nb;
    double mx = -INFINITY;
    for (uint32_t i = threadIdx.x; i <= N; i += blockDim.x)
        if (S[i] > 0) mx = fmax(mx, -lnw[i] - bd * (double)i);
    mx = block_reduce_max(mx, sh);
    double z = 0, a1 = 0, a2 = 0, a4 = 0;
    for (uint32_t i = threadIdx.x; i <= N; i += blockDim.x) {
        if (!(S[i] > 0)) continue;   // unvisited: contributes nothing (and may overflow)
        const double bz = exp(-bd * (double)i - lnw[i] - mx);
        z += bz * S[i];
        a1 += bz * S[nb + i];
        a2 += bz * S[2 * nb + i];
        a4 += bz * S[3 * nb + i];
    }
    z = block_reduce_sum(z, sh);
    a1 = block_reduce_sum(a1, sh);
    a2 = block_reduce_sum(a2, sh);
    a4 = block_reduce_sum(a4, sh);
    if (threadIdx.x == 0) {
        const double m1 = a1 / z, m2 = a2 / z, m4 = a4 / z;
        const uint64_t plane = (uint64_t)gridDim.x;
        double *o = out + (uint64_t)id * blocks + b;
        o[0] = m1;
        o[plane] = (m2 - m1 * m1) * beta / (double)N;
        o[2 * plane] = 1.0 - m4 / (3.0 * m2 * m2);
    }
}

__global__ void k_fill_u32(uint32_t *p, uint32_t n, uint32_t v)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

hipError_t launch_fill_u32(hipStream_t st, uint32_t *p, uint32_t n, uint32_t v)
{
    hipLaunchKernelGGL(k_fill_u32, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
    return hipGetLastError();
}

hipError_t launch_reweight(hipStream_t st, const double *mom, const double *lnw, uint32_t N,
                           uint32_t blocks, double beta, const double *deltas,
                           uint32_t ndelta, double *out)
{
    hipLaunchKernelGGL(k_reweight, dim3(ndelta * blocks), dim3(256), 0, st, mom, lnw, N, blocks,
                       beta, deltas, out);
    return hipGetLastError();
}

}  // namespace muca
