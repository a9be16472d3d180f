// muca_api.cpp -- the C ABI of libmuca (include/muca.h): contexts, device
// buffers, launches and the O(N) host-side pieces of the weight iteration.
#include "../../include/muca.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "acclog.h"
#include "ctx.h"
#include "kernels.h"

// the thread's last error message (muca_last_error)
thread_local std::string g_muca_err;

namespace {

// neighbour and order tables exactly as muca_delta_multigpu.cu:157-175
void make_tables(uint32_t L, std::vector<uint32_t> &naver, std::vector<uint32_t> &order)
{
    const uint32_t N = L * L;
    naver.assign(4ull * N, 0);
    order.assign(N, 0);
    for (uint32_t i = 0; i < N; i++) {
        int right = (int)i + 1, left = (int)i - 1, up = (int)(i + L), down = (int)i - (int)L;
        if (right % (int)L == 0) right -= (int)L;
        if (i % L == 0) left += (int)L;
        if (up > (int)N - 1) up -= (int)N;
        if (down < 0) down += (int)N;
        naver[4ull * i + 0] = (uint32_t)right;
        naver[4ull * i + 1] = (uint32_t)left;
        naver[4ull * i + 2] = (uint32_t)up;
        naver[4ull * i + 3] = (uint32_t)down;
        const uint32_t half = N / 2;
        const uint32_t blk = half ? (i / half) % 2 : 0;
        order[i] = ((0 == blk) * (2 * i)) % N + ((1 == blk) * (2 * i + 1)) % N;
    }
}

void free_ctx(muca_ctx *c)
{
    if (!c) return;
    if (c->p.device >= 0) hipSetDevice(c->p.device);
    void *bufs[] = {c->lat, c->E, c->D, c->M, c->lnw64, c->naver,
                    c->hist, c->joint, c->moms, c->mom, c->deltas, c->rw_out,
                    c->rw_flag};
    for (void *b : bufs)
        if (b) hipFree(b);
    if (c->pin) hipHostFree(c->pin);
    if (c->ev0) hipEventDestroy(c->ev0);
    if (c->ev1) hipEventDestroy(c->ev1);
    if (c->st) hipStreamDestroy(c->st);
    delete c;
}

template <typename T>
int dev_alloc(T **p, uint64_t count, const char *what)
{
    hipError_t e = hipMalloc((void **)p, count * sizeof(T) ? count * sizeof(T) : 1);
    if (e != hipSuccess) {
        *p = nullptr;
        return fail(MUCA_E_NOMEM, std::string("hipMalloc(") + what + ", " +
                                      std::to_string(count * sizeof(T)) +
                                      " bytes): " + hipGetErrorString(e));
    }
    return MUCA_OK;
}

// The team kernel's layout for W walkers, with `moments` that of a launch that
// accumulates per-D moments (production launches of such a context)
bool probe_team(uint32_t L, uint64_t W, int fp64, bool moments, size_t lds, uint32_t cus,
                muca::TeamLayout &lay)
{
    uint64_t mark = 0;   // never read: a non-null pointer asks for moments
    muca::McsArgs a{};
    a.N = L * L;
    a.L = L;
    a.W = W;
    a.nup = 1;
    a.moms = moments ? &mark : nullptr;
    return muca::team_layout(a, fp64, lds, cus, lay);
}

// What the choice of a kernel depends on.  obs: 0 the D histogram, 1 the joint
// histogram, 2 per-D moments (of launches with nup > 0)
struct Shape {
    uint32_t L;
    uint64_t W;
    int fp64, obs;
    size_t lds;
    uint64_t cus;
};

Shape shape_of(const muca_ctx &c)
{
    const int obs = c.p.joint_blocks == 0 ? 0 : c.p.observables == MUCA_OBS_MOMENTS ? 2
                                            : c.cfg.fp64 ? 1 : 0;
    return {c.p.L, c.W, c.cfg.fp64, obs, c.cfg.lds_max, c.cus ? c.cus : 256u};
}

// Kernel choice (attempts/ns on MI355X).  The team kernel keeps every SIMD
// busy when walkers are few (L = 72: 82 at 4096 walkers; 76 at 16 384
// against 37 for one lane per walker); the lane kernel wins once there
// are enough wavefronts to hide its memory latency.  They meet near 128
// walkers per compute unit (L = 64, 32 768 walkers: 80 against 73; 65 536:
// 80 against 149; L = 128 the same).  Where several workgroups of teams
// share a compute unit's LDS and half-rows fill a round the teams lead
// to twice that (L = 32, 65 536 walkers: 185 against 142; 131 072: 198
// against 243).  At odd L the alternative is the generic kernel; times of
// the teams over its at 24 576, 32 768, 49 152 and 65 536 walkers: L = 9 0.82,
// 1.11, 1.45, 1.86; L = 11 0.67, 0.93, 1.18, 1.49 (few of a team's lanes
// have work); L = 17 0.46, 0.62, 0.80, 1.01; two workgroups per compute
// unit, L = 33 0.22, 0.32, 0.36, 0.47 and L = 51 0.30, 0.44, 0.53, 0.72; one,
// L = 57 0.47, 0.72, 0.88, 1.21 and L = 63 0.45, 0.67, 0.83, 1.14.  With the
// joint histogram, at 8192, 16 384, 24 576 and 32 768: L = 9 0.77, 1.42, 1.90,
// 2.30; L = 11 0.64, 1.18, 1.53, 1.93; L = 13 0.37, 0.72, 0.95, 1.18; L = 17
// 0.28, 0.47, 0.58, 0.94.  With per-D moments the alternative is the generic
// kernel, whose atomics collide: at even L and below L = 64 teams lead at any
// number (L = 9, 98 304 walkers: half its time; L = 72, 65 536: 85 against 25;
// L = 128: 97 against 45; L = 48, 262 144: 67 against 43), at larger odd L to
// 256 per compute unit (L = 65, 65 536: 0.66 of its time).  muca_autotune
// replaces this rule by measurement.
// A thermalisation of production keeps no observable and is chosen for as without
// (even L, 262 144 walkers, team over generic kernel: L = 8 4.45, L = 24 1.09, L = 64
// 1.65 times its time; the lane kernel is faster still).  Where it is part of a
// production launch and far longer than the rest, it decides (team over generic,
// therm = N, nup = N / 16: L = 8 1.3, L = 10 1.2, both from 65 536 walkers; L = 56 to
// 64, 262 144 walkers 1.03 to 1.56; nup = N / 3: L = 8 1.1, others below 1).
//   The team kernel moves whole lattices to LDS and back and sets up tables whatever
// a launch's length, so short launches go to the others.  The attempts from which it
// leads, as a share of N: 4096 walkers L = 10 0.08, L = 24 0.012, L = 72 0.008; 16 384
// walkers 0.16, 0.036, 0.062; 32 768 walkers L = 24 0.10, L = 48 0.13, L = 72 0.33, L =
// 128 0.26; 65 536 walkers L = 33 0.11, L = 45 0.16; that is about 8 + N w^2 / 65536
// with w <= 128 walkers per compute unit.  With moments (16 384 / 65 536 walkers): L =
// 24 0.013 / 0.035, L = 48 0.014 / 0.058, L = 72 0.000 / 0.007.  Where ln W and the
// lattices stay in HBM nothing is set up (L = 160, 16 384 walkers: from one attempt).
int choose_kernel(const Shape &q, uint64_t therm, uint64_t nup)
{
    const uint32_t L = q.L;
    const uint64_t N = (uint64_t)L * L, n = therm + nup, w = q.W / q.cus;
    const bool odd = L % 2 != 0, moments = q.obs == 2 && nup > 0, joint = q.obs == 1 && nup > 0;
    muca::TeamLayout lay{};
    const bool team_ok = probe_team(L, q.W, q.fp64, moments, q.lds, (uint32_t)q.cus, lay);
    muca::McsArgs a{};
    a.N = (uint32_t)N;
    a.L = L;
    const int other = !moments && muca::lane_eligible(a, q.fp64, q.lds) ? MUCA_KERNEL_LANE
                                                                        : MUCA_KERNEL_GENERIC;
    if (!team_ok) return other;
    uint64_t per_cu = 128;   // walkers per compute unit up to which teams lead
    if (moments)
        per_cu = !odd || L < 64 ? UINT64_MAX / q.cus : 256;
    else if (joint)
        per_cu = !odd || L >= 17 ? 128 : L >= 13 ? 96 : 32;
    else if (odd)
        per_cu = L < 11 ? 96 : L < 32 ? 128 : lay.bytes * 2 <= q.lds ? 256 : 192;
    else if (L >= 32 && lay.bytes * 3 <= q.lds)
        per_cu = 256;
    if (q.W > per_cu * q.cus) return other;
    if (moments) {
        if (w > 128 && (L <= 10 ? 2 * nup < therm : L >= 56 && w > 512 && 8 * nup < therm))
            return other;
        const uint64_t v = w < 64 ? w : 64;
        if (L < 132 && n < 4 + N * v / (L < 64 ? 1536 : 8192)) return other;
    } else if (!lay.lnw_global) {
        const uint64_t v = w < 128 ? w : 128;
        if (n < 8 + N * v * v / 65536) return other;
    }
    return MUCA_KERNEL_TEAM;
}

// Lanes per workgroup where none are asked for.  Lane kernel, four walkers per lane
// (lane_walkers): 256, or 512 where its LDS (ln W and the histogram) admits one
// workgroup per compute unit (524 288 walkers, L = 72: 570 attempts/ns either way).
// One walker per lane: with room for several workgroups 512 once they fill the device
// (L = 72, 262 144 walkers: 335 attempts/ns against 195 with 256); with room for one
// the walkers of a compute unit in one workgroup (L = 128, 131 072 walkers: 186 with
// 512 lanes against 103 with 256; 262 144: 324 with 1024).
int default_block(int kernel, const Shape &q)
{
    if (kernel == MUCA_KERNEL_GENERIC) return muca::generic_block(q.W, q.cus);
    if (kernel != MUCA_KERNEL_LANE) return 256;
    const size_t lds = (size_t)(q.L * q.L + 1) * ((q.fp64 ? 8 : 4) + 4);
    const bool one = lds * 2 > q.lds;
    if (muca::lane_walkers(q.L, q.W, (uint32_t)q.cus) == 4) return one ? 512 : 256;
    if (one) return q.W > 512 * q.cus ? 1024 : q.W > 256 * q.cus ? 512 : 256;
    return q.W >= 1024 * q.cus ? 512 : 256;
}

// c->d_state looked up if it is not known
int consistent(muca_ctx *c)
{
    if (c->d_state == 0) {
        const uint64_t W = c->W;
        struct Scratch {
            int32_t *p = nullptr;   // E, D, flag
            ~Scratch()
            {
                if (p) hipFree(p);
            }
        } t;
        uint32_t differ = 1;
        if (hipMalloc((void **)&t.p, (2 * W + 1) * 4) == hipSuccess) {
            uint32_t *flag = (uint32_t *)(t.p + 2 * W);
            HIP_TRY(hipMemsetAsync(flag, 0, 4, c->st));
            HIP_TRY(muca::launch_state(c->st, c->lat, W, c->p.L, t.p, t.p + W, nullptr));
            HIP_TRY(muca::launch_differ(c->st, t.p + W, c->D, W, flag));
            HIP_TRY(hipMemcpyAsync(&differ, flag, 4, hipMemcpyDeviceToHost, c->st));
            HIP_TRY(hipStreamSynchronize(c->st));
        } else {
            t.p = nullptr;
            (void)hipGetLastError();
        }
        c->d_state = differ ? -1 : 1;
    }
    return MUCA_OK;
}

// The configuration of a launch: the context's kernel (chosen for this launch where
// none was asked for or tuned) if the walkers' D is their lattices' (looked up once
// after either was set from outside), else the generic kernel, whose accesses stay
// in bounds for any D.
int launch_config(muca_ctx *c, uint64_t therm, uint64_t nup, muca::Launch &cfg)
{
    cfg = c->cfg;
    if (c->p.kernel == MUCA_KERNEL_AUTO && !c->tuned) {
        cfg.kernel = choose_kernel(shape_of(*c), therm, nup);
        if (c->p.block == 0) cfg.block = default_block(cfg.kernel, shape_of(*c));
    }
    if (cfg.kernel == MUCA_KERNEL_GENERIC) return MUCA_OK;
    if (int rc = consistent(c)) return rc;
    if (c->d_state < 0) {
        cfg.kernel = MUCA_KERNEL_GENERIC;
        if (c->p.block == 0) cfg.block = default_block(cfg.kernel, shape_of(*c));
    }
    return MUCA_OK;
}

}  // namespace

extern "C" {

const char *muca_last_error(void)
{
    return g_muca_err.c_str();
}

int muca_default_walkers(int32_t device, uint32_t *walkers)
{
    if (!walkers) return fail(MUCA_E_ARG, "walkers is NULL");
    int mt = 0, cu = 0;
    HIP_TRY(hipDeviceGetAttribute(&mt, hipDeviceAttributeMaxThreadsPerMultiProcessor, device));
    HIP_TRY(hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device));
    *walkers = (uint32_t)mt * (uint32_t)cu;
    return MUCA_OK;
}

int muca_create(const muca_params *params, muca_ctx **out)
{
    if (!params || !out) return fail(MUCA_E_ARG, "NULL argument");
    *out = nullptr;
    const muca_params &p = *params;
    if (p.L < 2 || p.L > 46340) return fail(MUCA_E_ARG, "L must be in [2, 46340]");
    if (p.rounds != 7 && p.rounds != 10) return fail(MUCA_E_ARG, "rounds must be 7 or 10");
    if (p.precision != MUCA_REF32 && p.precision != MUCA_FP64)
        return fail(MUCA_E_ARG, "precision must be MUCA_REF32 or MUCA_FP64");
    if (p.keying != MUCA_KEYING_WEIGHT && p.keying != MUCA_KEYING_PRODUCE)
        return fail(MUCA_E_ARG, "keying must be MUCA_KEYING_WEIGHT or MUCA_KEYING_PRODUCE");
    if (!(p.beta > 0) || !std::isfinite(p.beta)) return fail(MUCA_E_ARG, "beta must be > 0");
    if (p.observables != MUCA_OBS_JOINT && p.observables != MUCA_OBS_MOMENTS)
        return fail(MUCA_E_ARG, "observables must be MUCA_OBS_JOINT or MUCA_OBS_MOMENTS");
    const bool moments = p.joint_blocks > 0 && p.observables == MUCA_OBS_MOMENTS;
    if (moments && p.precision != MUCA_FP64)
        return fail(MUCA_E_ARG, "per-D moments are accumulated in MUCA_FP64 mode only");
    if (moments && p.kernel == MUCA_KERNEL_LANE)
        return fail(MUCA_E_ARG, "per-D moments are accumulated by the generic and team kernels only");
    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (p.device < 0 || p.device >= ndev)
        return fail(MUCA_E_ARG, "device " + std::to_string(p.device) + " not present (" +
                                    std::to_string(ndev) + " visible)");
    HIP_TRY(hipSetDevice(p.device));
    muca_ctx *c = new muca_ctx();
    c->p = p;
    c->N = p.L * p.L;
    uint32_t W = p.walkers;
    if (W == 0) {
        int rc = muca_default_walkers(p.device, &W);
        if (rc) {
            free_ctx(c);
            return rc;
        }
    }
    c->W = W;
    c->p.walkers = W;
    int cu = 0, lds = 0;
    hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, p.device);
    hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, p.device);
    c->cus = (uint32_t)cu;
    c->cfg.rounds = (int)p.rounds;
    c->cfg.fp64 = p.precision == MUCA_FP64;
    c->cfg.keying = p.keying;
    c->cfg.cus = c->cus;
    c->cfg.lds_max = (size_t)(lds > 0 ? lds : 65536);
    // the kernel of full-length launches; a launch that differs chooses for itself
    c->cfg.kernel = p.kernel != MUCA_KERNEL_AUTO ? p.kernel
                                                 : choose_kernel(shape_of(*c), c->N, c->N);
    if (p.block != 0 && (p.block < 64 || p.block > 1024 || p.block % 64 != 0)) {
        delete c;
        return fail(MUCA_E_ARG, "block must be 0 or a multiple of 64 in [64, 1024]");
    }
    c->cfg.block = p.block ? (int)p.block : default_block(c->cfg.kernel, shape_of(*c));
    const uint64_t N = c->N;
    int rc = MUCA_OK;
    if (!rc) rc = dev_alloc(&c->lat, N * W, "lattice");
    if (!rc) rc = dev_alloc(&c->E, W, "E");
    if (!rc) rc = dev_alloc(&c->D, W, "D");
    if (!rc) rc = dev_alloc(&c->M, W, "M");
    // ln W in both precisions, one copy per set
    if (!rc) rc = dev_alloc(&c->lnw64, (N + 1) * 3 / 2 + 1, "lnw");
    if (!rc) c->lnw32 = (float *)(c->lnw64 + N + 1);
    if (!rc) rc = dev_alloc(&c->naver, 5 * N, "site tables");   // naver, then order
    if (!rc) c->order = c->naver + 4 * N;
    if (!rc) rc = dev_alloc(&c->hist, N + 1, "hist");
    if (!rc && p.joint_blocks > 0) {
        if (p.joint_blocks > W) {
            free_ctx(c);
            return fail(MUCA_E_ARG, "joint_blocks exceeds walkers");
        }
        c->block_walkers = (W + p.joint_blocks - 1) / p.joint_blocks;
        if (p.observables == MUCA_OBS_MOMENTS) {
            rc = dev_alloc(&c->moms, (uint64_t)muca::kMomWords * (N + 1) * p.joint_blocks,
                           "per-D moments");
        } else {
            c->joint_stride = (N + 1) * (N + 2) / 2;
            rc = dev_alloc(&c->joint, c->joint_stride * p.joint_blocks, "joint histogram");
        }
    }
    if (rc) {
        free_ctx(c);
        return rc;
    }
    std::vector<uint32_t> naver, order;
    make_tables(p.L, naver, order);
    hipError_t e = hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking);
    // N + 1 values of ln W in both precisions are the least it is for
    if ((N + 1) * 12 <= kPinMax) c->pin_bytes = N * 20 + 12 < kPinMax ? N * 20 + 12 : kPinMax;
    if (c->pin_bytes && hipHostMalloc(&c->pin, c->pin_bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        c->pin = nullptr;
        c->pin_bytes = 0;
    }
    if (e == hipSuccess) e = hipEventCreate(&c->ev0);
    if (e == hipSuccess) e = hipEventCreate(&c->ev1);
    if (e == hipSuccess && 20 * N <= c->pin_bytes) {
        memcpy(c->pin, naver.data(), 16 * N);
        memcpy((char *)c->pin + 16 * N, order.data(), 4 * N);
        e = muca::launch_copy(c->st, c->naver, c->pin, 20 * N);
    } else if (e == hipSuccess) {
        e = hipMemcpyAsync(c->naver, naver.data(), 16 * N, hipMemcpyHostToDevice, c->st);
        if (e == hipSuccess)
            e = hipMemcpyAsync(c->order, order.data(), 4 * N, hipMemcpyHostToDevice, c->st);
    }
    // on the context's stream: one of the null stream would not be ordered
    // before the launches that follow
    if (e == hipSuccess) e = hipMemsetAsync(c->lat, 0, N * W, c->st);
    if (e == hipSuccess) e = hipMemsetAsync(c->E, 0, W * 4, c->st);
    if (e == hipSuccess) e = hipMemsetAsync(c->D, 0, W * 4, c->st);
    if (e == hipSuccess) e = hipMemsetAsync(c->M, 0, W * 4, c->st);
    if (e == hipSuccess && c->moms)
        e = hipMemsetAsync(c->moms, 0, (uint64_t)muca::kMomWords * (N + 1) * p.joint_blocks * 8,
                           c->st);
    if (e == hipSuccess) e = hipStreamSynchronize(c->st);
    if (e != hipSuccess) {
        free_ctx(c);
        return fail(MUCA_E_HIP, std::string("context setup: ") + hipGetErrorString(e));
    }
    *out = c;
    return MUCA_OK;
}

int muca_destroy(muca_ctx *c)
{
    free_ctx(c);
    return MUCA_OK;
}

int muca_query(const muca_ctx *c, muca_info *info)
{
    if (!c || !info) return fail(MUCA_E_ARG, "NULL argument");
    info->L = c->p.L;
    info->N = c->N;
    info->walkers = (uint32_t)c->W;
    info->nbins = c->N + 1;
    info->device = c->p.device;
    info->kernel = c->cfg.kernel;
    info->cus = c->cus;
    info->block = (uint32_t)c->cfg.block;
    info->lattice_bytes = (uint64_t)c->N * c->W;
    info->joint_bins = c->joint_stride * c->p.joint_blocks;
    info->lds_per_block = (uint32_t)c->cfg.lds_max;
    muca::TeamLayout lay{};
    info->lds_lattice = c->cfg.kernel == MUCA_KERNEL_TEAM &&
                        probe_team(c->p.L, c->W, c->cfg.fp64, c->moms != nullptr, c->cfg.lds_max,
                                   c->cus, lay) &&
                        lay.lat_lds;
    return MUCA_OK;
}

int muca_init_lattice(muca_ctx *c, uint32_t mm, uint32_t gpu_index, uint32_t seed)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(muca::launch_init_lattice(c->st, c->lat, c->W, c->N, c->p.keying, (int)c->p.rounds,
                                      mm, gpu_index, seed, 0));
    c->d_state = 0;
    HIP_TRY(hipStreamSynchronize(c->st));
    return MUCA_OK;
}

int muca_init_lattice_stratified(muca_ctx *c, uint32_t mm, uint32_t gpu_index, uint32_t seed)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(muca::launch_init_lattice(c->st, c->lat, c->W, c->N, c->p.keying, (int)c->p.rounds,
                                      mm, gpu_index, seed, 0, (uint32_t)c->W));
    c->d_state = 0;
    HIP_TRY(hipStreamSynchronize(c->st));
    return MUCA_OK;
}

int muca_set_lattice(muca_ctx *c, const int8_t *src, uint64_t bytes)
{
    if (!c || !src) return fail(MUCA_E_ARG, "NULL argument");
    if (bytes != (uint64_t)c->N * c->W) return fail(MUCA_E_ARG, "lattice size mismatch");
    for (uint64_t i = 0; i < bytes; i++)
        if (src[i] < -1 || src[i] > 1) return fail(MUCA_E_ARG, "spins must be in {-1,0,1}");
    HIP_TRY(hipSetDevice(c->p.device));
    c->d_state = 0;
    HIP_TRY(hipMemcpy(c->lat, src, bytes, hipMemcpyHostToDevice));
    return MUCA_OK;
}

int muca_get_lattice(muca_ctx *c, int8_t *dst, uint64_t bytes)
{
    if (!c || !dst) return fail(MUCA_E_ARG, "NULL argument");
    if (bytes != (uint64_t)c->N * c->W) return fail(MUCA_E_ARG, "lattice size mismatch");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(hipStreamSynchronize(c->st));
    HIP_TRY(hipMemcpy(dst, c->lat, bytes, hipMemcpyDeviceToHost));
    return MUCA_OK;
}

int muca_compute_state(muca_ctx *c)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(muca::launch_state(c->st, c->lat, c->W, c->p.L, c->E, c->D, c->M));
    HIP_TRY(hipStreamSynchronize(c->st));
    c->d_state = 1;
    return MUCA_OK;
}

int muca_get_state(muca_ctx *c, int32_t *E, int32_t *D, int32_t *M)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(hipStreamSynchronize(c->st));
    if (E) HIP_TRY(hipMemcpy(E, c->E, c->W * 4, hipMemcpyDeviceToHost));
    if (D) HIP_TRY(hipMemcpy(D, c->D, c->W * 4, hipMemcpyDeviceToHost));
    if (M) HIP_TRY(hipMemcpy(M, c->M, c->W * 4, hipMemcpyDeviceToHost));
    return MUCA_OK;
}

int muca_set_state(muca_ctx *c, const int32_t *E, const int32_t *D, const int32_t *M)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    if (D)
        for (uint64_t w = 0; w < c->W; w++)
            if (D[w] < 0 || (uint32_t)D[w] > c->N) return fail(MUCA_E_ARG, "D out of [0, N]");
    HIP_TRY(hipSetDevice(c->p.device));
    if (D) c->d_state = 0;
    if (E) HIP_TRY(hipMemcpy(c->E, E, c->W * 4, hipMemcpyHostToDevice));
    if (D) HIP_TRY(hipMemcpy(c->D, D, c->W * 4, hipMemcpyHostToDevice));
    if (M) HIP_TRY(hipMemcpy(c->M, M, c->W * 4, hipMemcpyHostToDevice));
    return MUCA_OK;
}

int muca_set_log_weight(muca_ctx *c, const double *lnw, uint32_t nbins)
{
    if (!c || !lnw) return fail(MUCA_E_ARG, "NULL argument");
    if (nbins != c->N + 1) return fail(MUCA_E_ARG, "nbins must be N+1");
    for (uint32_t i = 0; i < nbins; i++)
        if (!std::isfinite(lnw[i])) return fail(MUCA_E_ARG, "ln W must be finite");
    std::vector<double> pageable(c->pin ? 0 : (nbins * 12ull + 7) / 8);
    double *w64 = c->pin ? (double *)c->pin : pageable.data();
    float *w32 = (float *)(w64 + nbins);
    memcpy(w64, lnw, nbins * sizeof(double));
    for (uint32_t i = 0; i < nbins; i++) w32[i] = (float)lnw[i];
    HIP_TRY(hipSetDevice(c->p.device));
    if (c->pin)
        HIP_TRY(muca::launch_copy(c->st, c->lnw64, w64, nbins * 12ull));
    else
        HIP_TRY(hipMemcpyAsync(c->lnw64, w64, nbins * 12ull, hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    c->have_weights = true;
    return MUCA_OK;
}

int muca_run(muca_ctx *c, uint32_t iter, uint32_t seed, uint64_t therm, uint64_t nup,
             uint64_t *hist_out, float *kernel_ms)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    if (!c->have_weights) return fail(MUCA_E_STATE, "muca_set_log_weight was not called");
    HIP_TRY(hipSetDevice(c->p.device));
    const uint64_t N = c->N;
    HIP_TRY(hipMemsetAsync(c->hist, 0, (N + 1) * sizeof(uint64_t), c->st));
    const bool joint = c->joint && c->p.precision == MUCA_FP64 && nup > 0;
    if (joint)
        HIP_TRY(hipMemsetAsync(c->joint, 0, c->joint_stride * c->p.joint_blocks * 8, c->st));
    const bool moments = c->moms && nup > 0;
    if (moments && (nup >> 32))
        return fail(MUCA_E_ARG, "per-D moments take nupdates < 2^32 per launch");
    if (moments)
        HIP_TRY(hipMemsetAsync(c->moms, 0,
                               (uint64_t)muca::kMomWords * (N + 1) * c->p.joint_blocks * 8, c->st));
    muca::McsArgs a{};
    a.lat = c->lat;
    a.E = c->E;
    a.D = c->D;
    a.M = c->M;
    a.lnw32 = c->lnw32;
    a.lnw64 = c->lnw64;
    a.order = c->order;
    a.naver = c->naver;
    a.hist = c->hist;
    a.joint = joint ? c->joint : nullptr;
    a.moms = moments ? c->moms : nullptr;
    a.W = c->W;
    a.N = c->N;
    a.L = c->p.L;
    a.w_offset = 0;
    a.iter = iter;
    a.seed = seed;
    a.therm = therm;
    a.nup = nup;
    a.beta = c->p.beta;
    a.joint_stride = c->joint_stride;
    a.block_walkers = c->block_walkers ? c->block_walkers : c->W;
    a.joint_blocks = c->p.joint_blocks;
    a.hist_preload = c->hist_preload;
    muca::Launch cfg;
    if (int rc = launch_config(c, therm, nup, cfg)) return rc;
    HIP_TRY(hipEventRecord(c->ev0, c->st));
    HIP_TRY(muca::launch_mcs(c->st, cfg, a));
    HIP_TRY(hipEventRecord(c->ev1, c->st));
    if (hist_out && c->pin)
        HIP_TRY(muca::launch_copy(c->st, c->pin, c->hist, (N + 1) * sizeof(uint64_t)));
    else if (hist_out)
        HIP_TRY(hipMemcpyAsync(hist_out, c->hist, (N + 1) * sizeof(uint64_t), hipMemcpyDeviceToHost,
                               c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    if (kernel_ms) HIP_TRY(hipEventElapsedTime(kernel_ms, c->ev0, c->ev1));
    if (hist_out && c->pin) memcpy(hist_out, c->pin, (N + 1) * sizeof(uint64_t));
    return MUCA_OK;
}

int muca_set_test_hist_preload(muca_ctx *c, uint32_t preload)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    c->hist_preload = preload;
    return MUCA_OK;
}

int muca_test_lane_shape(uint32_t L, uint64_t walkers, uint32_t cus, uint32_t block,
                         uint32_t *lanes, uint32_t *per_lane)
{
    if (!lanes || !per_lane) return fail(MUCA_E_ARG, "NULL argument");
    const muca::LaneShape s = muca::lane_shape(L, walkers, cus, (int)block);
    *lanes = (uint32_t)s.lanes;
    *per_lane = (uint32_t)s.walkers;
    return MUCA_OK;
}

int muca_test_choose_kernel(uint32_t L, uint64_t walkers, int32_t precision, int32_t observables,
                            uint64_t therm, uint64_t nup, uint32_t lds, uint32_t cus,
                            int32_t *kernel, uint32_t *block)
{
    if (!kernel || !block) return fail(MUCA_E_ARG, "NULL argument");
    const Shape q{L, walkers, precision == MUCA_FP64, observables, lds, cus};
    *kernel = choose_kernel(q, therm, nup);
    *block = (uint32_t)default_block(*kernel, q);
    return MUCA_OK;
}

int muca_test_team_layout(uint32_t L, uint64_t walkers, int32_t precision, int32_t moments,
                          uint32_t lds, uint32_t cus, uint32_t *out)
{
    if (!out) return fail(MUCA_E_ARG, "NULL argument");
    muca::TeamLayout lay{};
    out[0] = probe_team(L, walkers, precision == MUCA_FP64, moments != 0, lds, cus, lay);
    out[1] = lay.lat_lds;
    out[2] = lay.lds_hist;
    out[3] = lay.lnw_global;
    out[4] = lay.rounds;
    out[5] = lay.order;
    out[6] = lay.row;
    out[7] = (uint32_t)lay.bytes;
    return MUCA_OK;
}

int muca_autotune(muca_ctx *c, uint64_t attempts, int32_t *kernel, uint32_t *block, float *ms)
{
    if (!c) return fail(MUCA_E_ARG, "NULL context");
    if (!c->have_weights) return fail(MUCA_E_STATE, "muca_set_log_weight was not called");
    if (attempts == 0) return fail(MUCA_E_ARG, "attempts must be > 0");
    HIP_TRY(hipSetDevice(c->p.device));
    const uint64_t N = c->N, W = c->W;
    int rc = consistent(c);
    if (rc) return rc;
    int8_t *lat0 = nullptr;
    int32_t *st0 = nullptr;
    rc = dev_alloc(&lat0, N * W, "autotune lattice copy");
    if (rc) return rc;
    // walkers whose D is not their lattice's are tuned with their lattice's state
    // (the lane and team kernels run no others); their own follows the copies
    const bool own = c->d_state > 0;
    rc = dev_alloc(&st0, (own ? 3 : 6) * W, "autotune state copy");
    if (rc) {
        hipFree(lat0);
        return rc;
    }
    int32_t *const state[3] = {c->E, c->D, c->M};
    auto keep_state = [&](bool save) -> hipError_t {
        hipError_t e = hipSuccess;
        for (int k = 0; k < 3 && e == hipSuccess; k++)
            e = hipMemcpyAsync(save ? st0 + (3 + k) * W : state[k], save ? state[k] : st0 + (3 + k) * W,
                               W * 4, hipMemcpyDeviceToDevice, c->st);
        return e;
    };
    auto save_restore = [&](bool save) -> hipError_t {
        hipError_t e;
        if (save) {
            e = hipMemcpyAsync(lat0, c->lat, N * W, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess) e = hipMemcpyAsync(st0, c->E, W * 4, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess)
                e = hipMemcpyAsync(st0 + W, c->D, W * 4, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess)
                e = hipMemcpyAsync(st0 + 2 * W, c->M, W * 4, hipMemcpyDeviceToDevice, c->st);
        } else {
            e = hipMemcpyAsync(c->lat, lat0, N * W, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess) e = hipMemcpyAsync(c->E, st0, W * 4, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess)
                e = hipMemcpyAsync(c->D, st0 + W, W * 4, hipMemcpyDeviceToDevice, c->st);
            if (e == hipSuccess)
                e = hipMemcpyAsync(c->M, st0 + 2 * W, W * 4, hipMemcpyDeviceToDevice, c->st);
        }
        return e;
    };
    muca::McsArgs a{};
    a.lat = c->lat;
    a.E = c->E;
    a.D = c->D;
    a.M = c->M;
    a.lnw32 = c->lnw32;
    a.lnw64 = c->lnw64;
    a.order = c->order;
    a.naver = c->naver;
    a.hist = c->hist;
    a.W = W;
    a.N = c->N;
    a.L = c->p.L;
    a.iter = 0xFFFFFFFFu;
    a.seed = 0;
    a.therm = attempts - attempts / 2;
    a.nup = attempts / 2;
    a.beta = c->p.beta;
    a.block_walkers = W;
    struct Cand {
        int kernel, block;
    };
    std::vector<Cand> cands;
    muca::TeamLayout lay{};
    const bool moments = c->moms != nullptr;   // accumulated by the generic and team kernels
    if (moments) {
        // timed as production runs: with the per-D moments
        if (a.nup >> 32) {
            hipFree(lat0);
            hipFree(st0);
            return fail(MUCA_E_ARG, "per-D moments take nupdates < 2^32 per launch");
        }
        a.moms = c->moms;
        a.joint_blocks = c->p.joint_blocks;
        a.block_walkers = c->block_walkers ? c->block_walkers : c->W;
    }
    if (muca::team_layout(a, c->cfg.fp64, c->cfg.lds_max, c->cus, lay))
        cands.push_back({MUCA_KERNEL_TEAM, 256});
    if (!moments && muca::lane_eligible(a, c->cfg.fp64, c->cfg.lds_max))
        for (int b : {256, 512, 1024}) cands.push_back({MUCA_KERNEL_LANE, b});
    for (int b : {64, 128, 256}) cands.push_back({MUCA_KERNEL_GENERIC, b});
    hipError_t e = own ? hipSuccess : keep_state(true);
    if (e == hipSuccess && !own)
        e = muca::launch_state(c->st, c->lat, W, c->p.L, c->E, c->D, c->M);
    if (e == hipSuccess) e = save_restore(true);
    float best = 0;
    Cand pick = {c->cfg.kernel, c->cfg.block};
    for (const Cand &cd : cands) {
        muca::Launch cfg = c->cfg;
        cfg.kernel = cd.kernel;
        cfg.block = cd.block;
        float t = 0;
        for (int rep = 0; rep < 2 && e == hipSuccess; rep++) {
            e = save_restore(false);
            if (e == hipSuccess) e = hipMemsetAsync(c->hist, 0, (N + 1) * 8, c->st);
            if (e == hipSuccess && moments)
                e = hipMemsetAsync(c->moms, 0,
                                   (uint64_t)muca::kMomWords * (N + 1) * c->p.joint_blocks * 8,
                                   c->st);
            if (e == hipSuccess) e = hipEventRecord(c->ev0, c->st);
            if (e == hipSuccess) e = muca::launch_mcs(c->st, cfg, a);
            if (e == hipSuccess) e = hipEventRecord(c->ev1, c->st);
            if (e == hipSuccess) e = hipEventSynchronize(c->ev1);
            if (e == hipSuccess) e = hipEventElapsedTime(&t, c->ev0, c->ev1);
        }
        if (e != hipSuccess) break;
        if (best == 0 || t < best) {
            best = t;
            pick = cd;
        }
    }
    if (e == hipSuccess) e = save_restore(false);
    if (e == hipSuccess && !own) e = keep_state(false);
    if (e == hipSuccess) e = hipStreamSynchronize(c->st);
    hipFree(lat0);
    hipFree(st0);
    if (e != hipSuccess) return fail(MUCA_E_HIP, std::string("autotune: ") + hipGetErrorString(e));
    c->tuned = true;
    c->cfg.kernel = pick.kernel;
    c->cfg.block = pick.block;
    if (kernel) *kernel = pick.kernel;
    if (block) *block = (uint32_t)pick.block;
    if (ms) *ms = best;
    return MUCA_OK;
}

int muca_get_hist(muca_ctx *c, uint64_t *hist, uint32_t nbins, float *copy_ms)
{
    if (!c || !hist) return fail(MUCA_E_ARG, "NULL argument");
    if (nbins != c->N + 1) return fail(MUCA_E_ARG, "nbins must be N+1");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(hipEventRecord(c->ev0, c->st));
    HIP_TRY(hipMemcpyAsync(hist, c->hist, (uint64_t)nbins * 8, hipMemcpyDeviceToHost, c->st));
    HIP_TRY(hipEventRecord(c->ev1, c->st));
    HIP_TRY(hipEventSynchronize(c->ev1));
    if (copy_ms) HIP_TRY(hipEventElapsedTime(copy_ms, c->ev0, c->ev1));
    return MUCA_OK;
}

int muca_get_joint(muca_ctx *c, uint32_t block, uint64_t *dst, uint64_t nbins)
{
    if (!c || !dst) return fail(MUCA_E_ARG, "NULL argument");
    if (!c->joint) return fail(MUCA_E_STATE, "context has no joint histogram");
    if (block >= c->p.joint_blocks) return fail(MUCA_E_ARG, "block out of range");
    if (nbins != c->joint_stride) return fail(MUCA_E_ARG, "nbins must be (N+1)(N+2)/2");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(hipStreamSynchronize(c->st));
    HIP_TRY(hipMemcpy(dst, c->joint + (uint64_t)block * c->joint_stride, nbins * 8,
                      hipMemcpyDeviceToHost));
    return MUCA_OK;
}

int muca_get_moments(muca_ctx *c, uint32_t block, uint64_t *dst, uint64_t nwords)
{
    if (!c || !dst) return fail(MUCA_E_ARG, "NULL argument");
    if (!c->moms) return fail(MUCA_E_STATE, "context has no per-D moments");
    if (block >= c->p.joint_blocks) return fail(MUCA_E_ARG, "block out of range");
    const uint64_t nb = (uint64_t)c->N + 1, n = (uint64_t)muca::kMomWords * nb;
    if (nwords != 6 * nb) return fail(MUCA_E_ARG, "nwords must be 6 (N+1)");
    HIP_TRY(hipSetDevice(c->p.device));
    HIP_TRY(hipStreamSynchronize(c->st));
    std::vector<uint64_t> w(n);
    HIP_TRY(hipMemcpy(w.data(), c->moms + (uint64_t)block * n, n * 8, hipMemcpyDeviceToHost));
    // limb words w0 + w1 2^32 + w2 2^64 -> (low, high) words of a 128-bit integer
    for (uint64_t d = 0; d < nb; d++) {
        if (w[d] >> 32) return fail(MUCA_E_RANGE, "a D bin holds 2^32 or more entries");
        dst[d] = w[d];
        dst[nb + d] = w[nb + d];
        for (int k = 0; k < 2; k++) {
            const uint64_t *l = &w[(2 + 3 * k) * nb + d];
            const unsigned __int128 v = (unsigned __int128)l[0] +
                                        ((unsigned __int128)l[nb] << 32) +
                                        ((unsigned __int128)l[2 * nb] << 64);
            dst[(2 + 2 * k) * nb + d] = (uint64_t)v;
            dst[(3 + 2 * k) * nb + d] = (uint64_t)(v >> 64);
        }
    }
    return MUCA_OK;
}

int muca_reweight(muca_ctx *c, const double *deltas, uint32_t ndelta, double *absM,
                  double *chi, double *binder)
{
    if (!c || !deltas || ndelta == 0) return fail(MUCA_E_ARG, "bad arguments");
    if (!c->joint && !c->moms)
        return fail(MUCA_E_STATE, "context has no joint histogram or per-D moments");
    if (!c->have_weights) return fail(MUCA_E_STATE, "muca_set_log_weight was not called");
    HIP_TRY(hipSetDevice(c->p.device));
    const uint32_t B = c->p.joint_blocks;
    const uint64_t nb = c->N + 1;
    if (!c->mom) {
        int rc = dev_alloc(&c->mom, (uint64_t)B * 4 * nb, "moments");
        if (rc) return rc;
    }
    if (!c->rw_flag) {
        int rc = dev_alloc(&c->rw_flag, 1, "range flag");
        if (rc) return rc;
    }
    if (ndelta > c->rw_cap) {
        if (c->deltas) hipFree(c->deltas);
        if (c->rw_out) hipFree(c->rw_out);
        c->deltas = nullptr;
        c->rw_out = nullptr;
        c->rw_cap = 0;
        int rc = dev_alloc(&c->deltas, ndelta, "deltas");
        if (!rc) rc = dev_alloc(&c->rw_out, (uint64_t)ndelta * B * 3, "reweight output");
        if (rc) return rc;
        c->rw_cap = ndelta;
    }
    HIP_TRY(hipMemcpyAsync(c->deltas, deltas, ndelta * 8, hipMemcpyHostToDevice, c->st));
    if (c->joint)
        HIP_TRY(muca::launch_joint_moments(c->st, c->joint, c->N, c->joint_stride, B, c->mom));
    else {
        HIP_TRY(hipMemsetAsync(c->rw_flag, 0, 4, c->st));
        HIP_TRY(muca::launch_moments_fp64(c->st, c->moms, c->N, B, c->mom, c->rw_flag));
    }
    HIP_TRY(muca::launch_reweight(c->st, c->mom, c->lnw64, c->N, B, c->p.beta, c->deltas,
                                  ndelta, c->rw_out));
    std::vector<double> o((size_t)ndelta * B * 3);
    uint32_t range = 0;
    HIP_TRY(hipMemcpyAsync(o.data(), c->rw_out, o.size() * 8, hipMemcpyDeviceToHost, c->st));
    if (!c->joint)
        HIP_TRY(hipMemcpyAsync(&range, c->rw_flag, 4, hipMemcpyDeviceToHost, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    if (range) return fail(MUCA_E_RANGE, "a D bin holds 2^32 or more entries");
    const size_t plane = (size_t)ndelta * B;
    for (size_t i = 0; i < plane; i++) {
        if (absM) absM[i] = o[i];
        if (chi) chi[i] = o[plane + i];
        if (binder) binder[i] = o[2 * plane + i];
    }
    return MUCA_OK;
}

// ---- host-side pieces of the weight iteration ------------------------------

int muca_hist_range(const uint64_t *hist, uint32_t N, int32_t *start, int32_t *end)
{
    if (!hist || !start || !end) return fail(MUCA_E_ARG, "NULL argument");
    int32_t s = (int32_t)N + 1, e = 0;
    for (uint32_t i = 0; i <= N; i++)
        if (hist[i] > 1) {
            s = (int32_t)i;
            break;
        }
    for (uint32_t i = N + 1; i-- > 0;)
        if (hist[i] > 1) {
            e = (int32_t)i;
            break;
        }
    if (s > e) s = e = 0;
    *start = s;
    *end = e;
    return MUCA_OK;
}

double muca_kull_leibler(const uint64_t *hist, uint32_t N)
{
    double bins = 0, events = 0, kld = 0;
    for (uint32_t i = 0; i <= N; i++)
        if (hist[i] > 0) {
            events = events + (double)hist[i];
            bins = bins + 1.0;
        }
    for (uint32_t i = 0; i <= N; i++)
        if (hist[i] > 0) {
            const double P = (double)hist[i] / events;
            const double Q = 1.0 / bins;
            kld = kld + P * std::log(P / Q);
        }
    return kld;
}

int muca_update_trivial(const uint64_t *hist, uint32_t N, double *lnw)
{
    if (!hist || !lnw) return fail(MUCA_E_ARG, "NULL argument");
    for (uint32_t i = 0; i <= N; i++)
        if (hist[i] > 1) lnw[i] = lnw[i] - std::log((double)hist[i]);
    return MUCA_OK;
}

int muca_update_recursive(const uint64_t *hist, uint32_t N, int32_t start, int32_t end,
                          double *p_acc, double *lnw)
{
    if (!hist || !lnw || !p_acc) return fail(MUCA_E_ARG, "NULL argument");
    if (start < 0 || end > (int32_t)N || start > end) return fail(MUCA_E_ARG, "bad range");
    std::vector<double> bf(lnw, lnw + N + 1);
    for (int32_t i = start; i < end; i++) {
        const uint64_t a = hist[i], b = hist[i + 1];
        if ((a != 0) & (b != 0)) {
            const double p = (double)(a * b) / (double)(a + b);
            const double k = p / (p + p_acc[i]);
            const double dS = -bf[i] + bf[i + 1] + k * std::log((double)a / (double)b);
            lnw[i + 1] = lnw[i] + dS;
            p_acc[i] = p_acc[i] + p;
        }
    }
    return MUCA_OK;
}

int muca_normalise(uint32_t N, double *lnw)
{
    if (!lnw) return fail(MUCA_E_ARG, "NULL argument");
    const double t = lnw[0];
    for (uint32_t i = 0; i <= N; i++) lnw[i] = lnw[i] - t;
    return MUCA_OK;
}

int muca_jackknife(const double *x, uint32_t J, double *avg_out, double *err_out)
{
    if (!x || !avg_out || !err_out || J == 0) return fail(MUCA_E_ARG, "bad arguments");
    double avg = 0;
    for (uint32_t i = 0; i < J; i++) avg += x[i];
    std::vector<double> mi(J);
    for (uint32_t i = 0; i < J; i++) mi[i] = (avg - x[i]) / (double)(J - 1);
    avg = avg / (double)J;
    double dev = 0;
    for (uint32_t i = 0; i < J; i++) dev += (avg - mi[i]) * (avg - mi[i]);
    dev = (J - 1) * dev / (double)J;
    *avg_out = avg;
    *err_out = std::sqrt(dev);
    return MUCA_OK;
}

// ---- self-checks -----------------------------------------------------------

float muca_acclog_host(uint32_t r)
{
    return acclog_u01(r);
}

int muca_acclog_host_range(uint32_t k0, uint32_t n, float *out)
{
    if (!out) return fail(MUCA_E_ARG, "NULL argument");
    for (uint32_t t = 0; t < n; t++) out[t] = acclog_u01((k0 + t) << 9);
    return MUCA_OK;
}

int muca_acclog_device(int32_t device, uint32_t k0, uint32_t n, float *out)
{
    if (!out || n == 0) return fail(MUCA_E_ARG, "bad arguments");
    HIP_TRY(hipSetDevice(device));
    float *d = nullptr;
    int rc = dev_alloc(&d, n, "acclog");
    if (rc) return rc;
    hipError_t e = muca::launch_acclog(nullptr, k0, n, d);
    if (e == hipSuccess) e = hipMemcpy(out, d, (size_t)n * 4, hipMemcpyDeviceToHost);
    hipFree(d);
    if (e != hipSuccess) return fail(MUCA_E_HIP, std::string("acclog: ") + hipGetErrorString(e));
    return MUCA_OK;
}

int muca_acclog_fast_device(int32_t device, uint32_t k0, uint32_t n, float *out)
{
    if (!out || n == 0) return fail(MUCA_E_ARG, "bad arguments");
    HIP_TRY(hipSetDevice(device));
    float *d = nullptr;
    int rc = dev_alloc(&d, n, "acclog_fast");
    if (rc) return rc;
    hipError_t e = muca::launch_acclog_fast(nullptr, k0, n, d);
    if (e == hipSuccess) e = hipMemcpy(out, d, (size_t)n * 4, hipMemcpyDeviceToHost);
    hipFree(d);
    if (e != hipSuccess)
        return fail(MUCA_E_HIP, std::string("acclog_fast: ") + hipGetErrorString(e));
    return MUCA_OK;
}

int muca_acclog_screen_device(int32_t device, uint32_t k0, uint32_t n, float *thi, float *lim)
{
    if (!thi || !lim || n == 0) return fail(MUCA_E_ARG, "bad arguments");
    HIP_TRY(hipSetDevice(device));
    float *d = nullptr;
    int rc = dev_alloc(&d, 2ull * n, "acclog_screen");
    if (rc) return rc;
    hipError_t e = muca::launch_acclog_screen(nullptr, k0, n, d);
    if (e == hipSuccess) e = hipMemcpy(thi, d, (size_t)n * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(lim, d + n, (size_t)n * 4, hipMemcpyDeviceToHost);
    hipFree(d);
    if (e != hipSuccess)
        return fail(MUCA_E_HIP, std::string("acclog_screen: ") + hipGetErrorString(e));
    return MUCA_OK;
}

}  // extern "C"
