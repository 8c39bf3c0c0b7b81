// capi.hip -- the C ABI of include/gempic_hip.h.
//
// Owns the device memory of each handle (SoA particles with a sort double
// buffer, the field/current grid slots, the constant tables, reduction
// scratch), drives the kernels of pass1d.hip on the handle's stream, and
// maps kernel error flags onto the reference's exceptions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/gempic_hip.h"
#include "host_setup.hpp"
#include "lib_internal.hpp"
#include "transfer.hpp"

using namespace gl;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string &msg)
{
    g_last_error = msg;
    return code;
}

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(GEMPIC_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

int check_device()
{
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1) {
        const char *hv = getenv("HIP_VISIBLE_DEVICES");
        const char *rv = getenv("ROCR_VISIBLE_DEVICES");
        return fail(GEMPIC_ERR_DEVICE,
                    std::string("no usable AMD GPU: the particle-field path runs only on the GPU "
                                "(hipGetDeviceCount: ") +
                        hipGetErrorName(e) + ", count " + std::to_string(n) +
                        ", HIP_VISIBLE_DEVICES=" + (hv ? hv : "unset") +
                        ", ROCR_VISIBLE_DEVICES=" + (rv ? rv : "unset") + ")");
    }
    return GEMPIC_OK;
}

int device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        return 256;
    return cus;
}

}  // namespace

int gl::abi_fail(int code, const char *msg) { return fail(code, msg); }
int gl::abi_check_device() { return check_device(); }
int gl::abi_device_cus() { return device_cus(); }
hipError_t gl::to_host(void *dst, const void *src, size_t bytes, hipStream_t after, int device)
{
    return TransferPool::get().to_host(dst, src, bytes, after, device);
}
void gl::transfer_acquire() { TransferPool::get().acquire(); }
void gl::transfer_release() { TransferPool::get().release(); }

namespace {

bool pair_supported(int p0, int p1)
{
    return (p0 == 1 && (p1 == 0 || p1 == 1)) || (p0 == 2 && (p1 == 1 || p1 == 2)) ||
           (p0 == 3 && (p1 == 2 || p1 == 3));
}

struct Launch {
    int blocks;
    int64_t chunk;
    int iters;
    int ngroups;
};

// Workgroups of a 1D particle pass: 4 particles per thread, fewer (down to
// one) while that makes under 512 workgroups, two per CU. A workgroup's start
// and drain cost about 8 us against 0.5 us per particle of a lane, so a small
// count wants the chip filled first. us per step at (least particles per
// thread, workgroups below which it does not apply) = (8, 0), (8, 256),
// (4, 256), (4, 512):
//   fused 1D2V     16,384: 35.7, 19.2, 19.3, 19.2   300,001: 34.4, 31.5, 31.7, 31.1
//               1,048,576: 41.3, 41.7, 33.2, 33.4
//   1D1V (hot)    100,000: 46.1, 24.2, 24.3, 22.0   400,000: 40.8, 38.2, 33.2, 33.2
//   24 instances of 65,536 to 524,288 particles in one ensemble, whose
//   workgroups fill the chip together: 164, 175, 176, 181
// An ensemble's instances keep their stand-alone partition (equal results);
// its pass takes several such blocks per workgroup (k_pass1d_batch), and a
// block's start and drain were cut since: these 24 instances 159 now. Instances of
// 131,072 to 262,144 particles still pay for it (24 of 262,144: 162, with (8, 0) and
// the drain as it was 155); gempic_ensemble_autotune finds them a partition.
constexpr int kPerThread = 4;
constexpr int kFewBlocks = 512;

Launch plan(int64_t n, int max_blocks)
{
    Launch L;
    int64_t want = (n + (int64_t)kBlock * kPerThread - 1) / ((int64_t)kBlock * kPerThread);
    want = std::max(want, std::min<int64_t>(kFewBlocks, (n + kBlock - 1) / kBlock));
    if (want < 1) want = 1;
    int64_t blocks = std::min<int64_t>(want, max_blocks);
    int64_t per = (n + blocks - 1) / blocks;
    L.chunk = ((per + kBlock - 1) / kBlock) * kBlock;
    if (L.chunk < kBlock) L.chunk = kBlock;
    L.iters = (int)(L.chunk / kBlock);
    L.blocks = (int)((n + L.chunk - 1) / L.chunk);
    if (L.blocks < 1) L.blocks = 1;
    L.ngroups = (L.blocks + kGroup - 1) / kGroup;
    return L;
}

#ifndef GEMPIC_GEN_SKEW
#define GEMPIC_GEN_SKEW 0.25
#endif
#ifndef GEMPIC_ADJ_GEN_SKEW
#define GEMPIC_ADJ_GEN_SKEW 0.15
#endif
constexpr double kGenSkew = GEMPIC_GEN_SKEW;         // forward and Boris passes
constexpr double kAdjGenSkew = GEMPIC_ADJ_GEN_SKEW;  // reverse-mode passes

// The particle pass's partition in generations. A launch of G * cus
// workgroups (2 <= G <= kMaxGen) fills every CU G deep, workgroup b on CU
// b mod cus beside b +- cus, ..., and a SIMD issues from its oldest wave
// first: with equal chunks the last generation ends well after the first,
// and each CU runs the end of the pass with few waves. Chunks that shrink
// linearly from the first generation to the last (weights 1 + skew (G - 1 -
// 2g) / (G - 1), in whole waves of 64 particles) let the generations end
// together. The partition depends only on n, the launch and the CU count,
// so every deposit's summation order stays a fixed function of the particle
// order.
void set_generations(PassArgs &a, const Launch &L, int cus, double skew = kGenSkew)
{
    a.gen_blocks = 0;
    if (skew <= 0.0 || cus < 1 || L.blocks % cus != 0) return;
    const int G = L.blocks / cus;
    if (G < 2 || G > kMaxGen) return;
    // waves of 64 particles per column of G workgroups (one per generation)
    const int64_t T = (a.n + (int64_t)64 * cus - 1) / ((int64_t)64 * cus);
    if (T < 8 * G) return;
    double wt[kMaxGen], wsum = 0.0;
    for (int g = 0; g < G; ++g) {
        wt[g] = 1.0 + skew * (double)(G - 1 - 2 * g) / (double)(G - 1);
        wsum += wt[g];
    }
    int64_t acc = 0, waves[kMaxGen];
    for (int g = 0; g + 1 < G; ++g) {
        waves[g] = std::max<int64_t>(1, std::llround((double)T * wt[g] / wsum));
        acc += waves[g];
    }
    if (T - acc < 1) return;
    waves[G - 1] = T - acc;
    a.gen_base[0] = 0;
    for (int g = 0; g < G; ++g) {
        a.gen_chunk[g] = waves[g] * 64;
        if (g + 1 < G) a.gen_base[g + 1] = a.gen_base[g] + a.gen_chunk[g] * cus;
    }
    a.gen_blocks = cus;
}

}  // namespace

// ---------------------------------------------------------------------------
// splitting handle
// ---------------------------------------------------------------------------
struct gempic_splitting {
    int device = 0;
    hipStream_t stream = nullptr;
    int dim_v = 2, n_weights = 1, ld = 4;
    int64_t n = 0, nx = 0;
    double xmin = 0, xmax = 0, Lx = 0, dx = 0;
    int mdeg = 3, deg0 = 3, deg1 = 2, sm0 = 0, sm1 = 0;
    double scaling0 = 1, scaling1 = 1, charge = 1, mass = 1, cw = 0, qm = 1;
    double qx1[3] = {0, 0, 0}, qw1[3] = {0, 0, 0};
    gh::Maxwell1DTables tabs;

    double *d_x = nullptr, *d_v1 = nullptr, *d_v2 = nullptr, *d_w = nullptr;
    int64_t *d_id = nullptr;
    double *d_x2 = nullptr, *d_v12 = nullptr, *d_v22 = nullptr, *d_w2 = nullptr;
    int64_t *d_id2 = nullptr;
    double *d_grid = nullptr, *d_tabs = nullptr;
    double *d_part = nullptr, *d_gpart = nullptr;
    unsigned *d_cnt = nullptr;
    int *d_err = nullptr;
    double *d_diag = nullptr;
    int *d_sort_counts = nullptr, *d_sort_gsum = nullptr;
    SortGeometry sortg{};
    double *d_stage = nullptr;

    int max_blocks = 1024;            // capacity of the reduction scratch
    int dep_blocks = 0;               // workgroups of every deposit-bearing pass (0: not set)
    int boris_blocks = 0;             // workgroups of the Boris passes
    int override_blocks = 0;          // gempic_set_launch
    int cus = 256;
    int kernels_per_step = 1;         // fused Strang step in 1 or 2 particle kernels
    int arith = GEMPIC_ARITH_REFERENCE;  // arithmetic of the 1d2v passes of strang_splitting and the operators
    int64_t sort_interval = 20;
    int64_t steps_since_sort = 0;
    bool particles_set = false;

    // reverse mode (gempic_strang_splitting_adjoint): field records, particle
    // checkpoints, the recompute buffer of one checkpoint interval, the
    // particle cotangents (x, v1, v2) and the adjoint grid slots
    double *d_hist = nullptr, *d_ckpt = nullptr, *d_seg = nullptr, *d_lam = nullptr;
    double *d_agrid = nullptr;
    double *d_wsnap = nullptr;        // weights of every sort epoch
    int *d_perm = nullptr;            // each epoch's sort: perm[new index] = old index
    int64_t epoch_cap = 0;            // sort epochs d_wsnap and d_perm hold
    int64_t *d_ids = nullptr;         // the particle order (id) the call started from
    size_t hist_cap = 0, ckpt_cap = 0, seg_cap = 0, ids_cap = 0, wsnap_cap = 0, perm_cap = 0;
    int *cur_perm = nullptr;          // SortArgs::perm of the next sort
    double *cur_hist = nullptr;       // PassArgs::hist of the next launches
    double *cur_cx = nullptr;         // PassArgs::cx/cv1/cv2 (x, v1, v2 at n-strides)
    const int64_t *adj_id0 = nullptr; // particle order of the reverse-mode result
    int adj_blocks = 0;
    bool adj_ready = false;

    // profiling
    bool profile = false;
    int profile_every = 1;            // sample every n-th launch of each kernel id
    static constexpr int kProfIds = 13;
    int64_t prof_seen[kProfIds] = {};
    struct Pend { int id; hipEvent_t a, b; };
    std::vector<Pend> pending;
    std::vector<hipEvent_t> pool;
    double prof_ms[kProfIds] = {};
    int64_t prof_cnt[kProfIds] = {};
};

struct gempic_maxwell1d {
    hipStream_t stream = nullptr;
    int64_t nx = 0;
    double xmin = 0, xmax = 0, dx = 0;
    int degree = 3;
    gh::Maxwell1DTables tabs;
    double *d_grid = nullptr, *d_tabs = nullptr, *d_scalar = nullptr;
};

namespace {

hipEvent_t take_event(gempic_splitting *h)
{
    if (!h->pool.empty()) {
        hipEvent_t e = h->pool.back();
        h->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

struct ProfScope {
    gempic_splitting *h;
    int id;
    hipEvent_t a = nullptr, b = nullptr;
    ProfScope(gempic_splitting *hh, int kid) : h(hh), id(kid)
    {
        if (h->profile && h->prof_seen[id]++ % h->profile_every == 0) {
            a = take_event(h);
            b = take_event(h);
            if (a) (void)hipEventRecord(a, h->stream);
        }
    }
    ~ProfScope()
    {
        if (a && b) {
            (void)hipEventRecord(b, h->stream);
            h->pending.push_back({id, a, b});
        } else {
            if (a) h->pool.push_back(a);
            if (b) h->pool.push_back(b);
        }
    }
};

void resolve_profile(gempic_splitting *h)
{
    if (h->pending.empty()) return;
    (void)hipStreamSynchronize(h->stream);
    for (auto &p : h->pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
            h->prof_ms[p.id] += ms;
            h->prof_cnt[p.id] += 1;
        }
        h->pool.push_back(p.a);
        h->pool.push_back(p.b);
    }
    h->pending.clear();
}

PassArgs pass_args(gempic_splitting *h)
{
    PassArgs a;
    std::memset(&a, 0, sizeof(a));
    a.n = h->n;
    a.nx = (int)h->nx;
    a.xmin = h->xmin;
    a.dx = h->dx;
    a.Lx = h->Lx;
    a.scaling0 = h->scaling0;
    a.scaling1 = h->scaling1;
    for (int k = 0; k < 3; ++k) { a.qx[k] = h->qx1[k]; a.qw[k] = h->qw1[k]; }
    a.charge = h->charge;
    a.mass = h->mass;
    a.cw = h->cw;
    a.qm = h->qm;
    a.x = h->d_x; a.v1 = h->d_v1; a.v2 = h->d_v2; a.w = h->d_w;
    a.grid = h->d_grid;
    a.tabs = h->d_tabs;
    a.part = h->d_part;
    a.gpart = h->d_gpart;
    a.cnt = h->d_cnt;
    a.err = h->d_err;
    a.diag = h->d_diag;
    a.hist = h->cur_hist;
    if (h->cur_cx) {
        a.cx = h->cur_cx;
        a.cv1 = h->cur_cx + h->n;
        a.cv2 = h->cur_cx + 2 * h->n;
    }
    return a;
}

bool mode_deposits(int mode)
{
    return (mode & (M_HP2A | M_HP1 | M_HP2B | M_RHO | M_DIAG | M_WITH_J2A)) != 0;
}

// Deposit-bearing passes all use one workgroup count, so the deposits of the
// fused and the sub-step paths are summed in the same order: CUs times the
// fewest workgroups per CU among those kernels (one full round, no tail).
void set_dep_blocks(gempic_splitting *h)
{
    std::vector<int> modes;
    if (h->dim_v == 2)
        modes = {M_HP2A, M_HP1, M_HE | M_HP2A | M_HP1 | M_HP2B,
                 M_HE_PREV | M_HE | M_HP2A | M_HP1 | M_HP2B, M_HE_PREV | M_HE | M_HP2A | M_NOEPI,
                 M_HP1 | M_HP2B | M_WITH_J2A, M_RHO, M_DIAG};
    else
        modes = {M_V1 | M_HP1, M_V1 | M_HE | M_HP1, M_V1 | M_HE_PREV | M_HE | M_HP1, M_RHO};
    int bpc = 64;
    for (int m : modes)
        bpc = std::min(bpc, pass_blocks_per_cu(h->deg0, h->deg1, m, pass_shmem_bytes((int)h->nx, m)));
    h->dep_blocks = std::max(1, std::min(h->max_blocks, h->cus * bpc));
}

int run_pass(gempic_splitting *h, int mode, double dt_he, double dt_hp2, double dt_hp1, int more,
             int prof_id)
{
    PassArgs a = pass_args(h);
    int target;
    if (h->override_blocks) target = h->override_blocks;
    else if (mode_deposits(mode)) target = h->dep_blocks;
    else target = std::min(h->max_blocks,
                           h->cus * pass_blocks_per_cu(h->deg0, h->deg1, mode,
                                                       pass_shmem_bytes((int)h->nx, mode)));
    Launch L = plan(h->n, target);
    a.chunk = L.chunk;
    a.iters = L.iters;
    a.ngroups = L.ngroups;
    a.rgroups = epi_groups(L.blocks);
    set_generations(a, L, h->cus);
    a.dt_he = dt_he;
    a.dt_hp2 = dt_hp2;
    a.dt_hp1 = dt_hp1;
    a.dtqm_he = dt_he * h->qm;
    a.dtqm_hp2 = dt_hp2 * h->qm;
    a.more = more;
    {
        ProfScope ps(h, prof_id);
        hipError_t e = launch_pass(h->deg0, h->deg1, mode, a, L.blocks,
                                   pass_shmem_bytes((int)h->nx, mode), h->stream);
        if (e != hipSuccess)
            return fail(GEMPIC_ERR_DEVICE, std::string("particle pass launch: ") + hipGetErrorString(e));
    }
    return GEMPIC_OK;
}

int run_grid(gempic_splitting *h, const GridProg &g)
{
    ProfScope ps(h, 5);
    hipError_t e = launch_grid(g, (int)h->nx, h->dx, h->d_grid, h->d_tabs, nullptr, h->stream);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("field program launch: ") + hipGetErrorString(e));
    return GEMPIC_OK;
}

GridProg prog1(int op, double dt, int a, int b, int out)
{
    GridProg g;
    std::memset(&g, 0, sizeof(g));
    g.nops = 1;
    g.op[0] = op; g.dt[0] = dt; g.slot_a[0] = a; g.slot_b[0] = b; g.slot_out[0] = out;
    return g;
}

void prog_add(GridProg &g, int op, double dt, int a, int b, int out)
{
    int k = g.nops++;
    g.op[k] = op; g.dt[k] = dt; g.slot_a[k] = a; g.slot_b[k] = b; g.slot_out[k] = out;
}

int run_sort(gempic_splitting *h)
{
    ProfScope ps(h, 6);
    SortArgs s;
    s.n = h->n;
    s.nx = (int)h->nx;
    s.sub = h->sortg.sub;
    s.nbins = h->sortg.nbins;
    s.ntiles = h->sortg.ntiles;
    s.tiles_per_group = h->sortg.tiles_per_group;
    s.ngroups = h->sortg.ngroups;
    s.xmin = h->xmin;
    s.dx = h->dx;
    s.x = h->d_x; s.v1 = h->d_v1; s.v2 = h->d_v2; s.w = h->d_w; s.id = h->d_id;
    s.x2 = h->d_x2; s.v12 = h->d_v12; s.v22 = h->d_v22; s.w2 = h->d_w2; s.id2 = h->d_id2;
    s.counts = h->d_sort_counts;
    s.gsum = h->d_sort_gsum;
    s.perm = h->cur_perm;
    hipError_t e = launch_sort(s, h->dim_v == 2, h->stream);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("sort launch: ") + hipGetErrorString(e));
    std::swap(h->d_x, h->d_x2);
    std::swap(h->d_v1, h->d_v12);
    std::swap(h->d_v2, h->d_v22);
    std::swap(h->d_w, h->d_w2);
    std::swap(h->d_id, h->d_id2);
    h->steps_since_sort = 0;
    return GEMPIC_OK;
}

int finish(gempic_splitting *h)
{
    HIP_TRY(hipStreamSynchronize(h->stream));
    int err = 0;
    HIP_TRY(hipMemcpy(&err, h->d_err, sizeof(int), hipMemcpyDeviceToHost));
    if (err) {
        HIP_TRY(hipMemset(h->d_err, 0, sizeof(int)));
        if (err & E_INEXACT)
            return fail(GEMPIC_ERR_INEXACT,
                        "InexactError: trunc(Int64, x): a particle position is not finite or lies "
                        "beyond 1e9 cells of the domain");
        if (err & E_FAR)
            return fail(GEMPIC_ERR_INEXACT,
                        "a particle crossed more than 65536 cells in one Hp1 push");
        return fail(GEMPIC_ERR_ARGUMENT, "BoundsError: a particle lies outside the pp matrix");
    }
    return GEMPIC_OK;
}

#define CHECK_H(h)                                                                    \
    do {                                                                              \
        if (!(h)) return fail(GEMPIC_ERR_ARGUMENT, "null handle");                    \
        if (hipSetDevice((h)->device) != hipSuccess)                                  \
            return fail(GEMPIC_ERR_DEVICE, "hipSetDevice failed");                    \
    } while (0)

#define CHECK_P(h)                                                                    \
    do {                                                                              \
        if (!(h)->particles_set) return fail(GEMPIC_ERR_STATE, "particles not set");  \
    } while (0)

template <typename T>
hipError_t dalloc(T **p, size_t count)
{
    return hipMalloc((void **)p, sizeof(T) * std::max<size_t>(count, 1));
}

}  // namespace

extern "C" {

int gempic_version(void) { return 100; }

const char *gempic_last_error(void) { return g_last_error.c_str(); }

int gempic_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int gempic_device_info(int *cus, char *arch, int arch_len)
{
    int rc = check_device();
    if (rc) return rc;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
        return fail(GEMPIC_ERR_DEVICE, "hipGetDeviceProperties failed");
    if (cus) *cus = prop.multiProcessorCount;
    if (arch && arch_len > 0) {
        std::strncpy(arch, prop.gcnArchName, (size_t)arch_len - 1);
        arch[arch_len - 1] = '\0';
    }
    return GEMPIC_OK;
}

int gempic_splitting_create(int64_t nx, double xmin, double xmax, int maxwell_degree, int degree0,
                            int smoothing0, int degree1, int smoothing1, int dim_v,
                            int64_t n_particles, int n_weights, double charge, double mass,
                            double common_weight, gempic_splitting **out)
{
    if (!out) return fail(GEMPIC_ERR_ARGUMENT, "out is NULL");
    *out = nullptr;
    if (maxwell_degree < 1 || maxwell_degree > 3)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: Wrong value of degree (1,2 or 3)");
    if (smoothing0 != GEMPIC_GALERKIN && smoothing0 != GEMPIC_COLLOCATION)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: smoothing type not implemented");
    if (smoothing1 != GEMPIC_GALERKIN && smoothing1 != GEMPIC_COLLOCATION)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: smoothing type not implemented");
    if (!pair_supported(degree0, degree1))
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: smoother degrees (p, p-1) or (p, p) with p in 1..3 are supported");
    if (dim_v != 1 && dim_v != 2) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: dim_v must be 1 or 2");
    if (n_weights != 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: n_weights must be 1");
    if (nx < 2 || nx > kNxMax || (nx % 2) != 0)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: nx must be even and in [2, 256]");
    if (n_particles < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: n_particles must be positive");
    if (n_particles > (int64_t)INT32_MAX - kSortTile)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: n_particles must be below 2^31 - 1024 per handle "
                                         "(32-bit sort offsets)");
    if (!(xmax > xmin)) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: xmax must exceed xmin");
    int rc = check_device();
    if (rc) return rc;

    gempic_splitting *h = new gempic_splitting();
    transfer_acquire();
    (void)hipGetDevice(&h->device);
    h->dim_v = dim_v;
    h->n_weights = n_weights;
    h->ld = 1 + dim_v + n_weights;
    h->n = n_particles;
    h->nx = nx;
    h->xmin = xmin;
    h->xmax = xmax;
    // Maxwell1DFEM: Lx = xmax - xmin, delta_x = Lx / n_dofs (maxwell_1d_fem.jl:50-53);
    // ParticleMeshCoupling1D: delta_x = (xmax - xmin) / n_grid, the same value.
    h->Lx = xmax - xmin;
    h->dx = h->Lx / (double)nx;
    h->mdeg = maxwell_degree;
    h->deg0 = degree0;
    h->deg1 = degree1;
    h->sm0 = smoothing0;
    h->sm1 = smoothing1;
    h->scaling0 = smoothing0 == GEMPIC_COLLOCATION ? 1.0 / h->dx : 1.0;
    h->scaling1 = smoothing1 == GEMPIC_COLLOCATION ? 1.0 / h->dx : 1.0;
    h->charge = charge;
    h->mass = mass;
    h->cw = common_weight == 0.0 ? 1.0 / (double)n_particles : common_weight;
    h->qm = charge / mass;
    gh::gauss_legendre((degree1 + 2) / 2, h->qx1, h->qw1);
    if (!gh::maxwell1d_tables(nx, maxwell_degree, h->tabs)) {
        transfer_release();
        delete h;
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: invalid Maxwell1DFEM size");
    }
    h->cus = device_cus();
    h->max_blocks = h->cus * 8;
    const int max_groups = std::max((h->max_blocks + kGroup - 1) / kGroup, kEpiGroupsMax);
    const size_t n = (size_t)n_particles;
    h->sortg = sort_geometry((int64_t)n, (int)nx);
    hipError_t e = hipSuccess;
    auto ok = [&](hipError_t r) { if (r != hipSuccess && e == hipSuccess) e = r; };
    ok(hipStreamCreate(&h->stream));
    ok(dalloc(&h->d_x, n)); ok(dalloc(&h->d_v1, n)); ok(dalloc(&h->d_w, n)); ok(dalloc(&h->d_id, n));
    ok(dalloc(&h->d_x2, n)); ok(dalloc(&h->d_v12, n)); ok(dalloc(&h->d_w2, n)); ok(dalloc(&h->d_id2, n));
    if (dim_v == 2) { ok(dalloc(&h->d_v2, n)); ok(dalloc(&h->d_v22, n)); }
    ok(dalloc(&h->d_grid, (size_t)NSLOT * nx));
    ok(dalloc(&h->d_tabs, (size_t)NTAB * nx));
    ok(dalloc(&h->d_part, (size_t)h->max_blocks * NDEP * nx + 64));
    ok(dalloc(&h->d_gpart, (size_t)max_groups * NDEP * nx + 64));
    ok(dalloc(&h->d_cnt, (size_t)max_groups + 2));
    ok(dalloc(&h->d_err, 1));
    ok(dalloc(&h->d_diag, 16));
    ok(dalloc(&h->d_sort_counts, (size_t)h->sortg.ntiles * h->sortg.nbins));
    ok(dalloc(&h->d_sort_gsum, (size_t)h->sortg.ngroups * h->sortg.nbins));
    if (e == hipSuccess) {
        ok(hipMemset(h->d_grid, 0, sizeof(double) * NSLOT * nx));
        ok(hipMemset(h->d_cnt, 0, sizeof(unsigned) * (max_groups + 2)));
        ok(hipMemset(h->d_err, 0, sizeof(int)));
        ok(hipMemset(h->d_diag, 0, sizeof(double) * 16));
        std::vector<double> T((size_t)NTAB * nx, 0.0);
        auto put = [&](int slot, const std::vector<double> &v) {
            std::copy(v.begin(), v.end(), T.begin() + (size_t)slot * nx);
        };
        put(T_COS, h->tabs.cos_tab); put(T_SIN, h->tabs.sin_tab);
        put(T_INVM0, h->tabs.inv_mass0); put(T_INVM1, h->tabs.inv_mass1);
        put(T_AMP, h->tabs.eig_weak_ampere); put(T_POIS, h->tabs.eig_weak_poisson);
        put(T_M0, h->tabs.eig_mass0); put(T_M1, h->tabs.eig_mass1);
        put(T_CM0, h->tabs.circ_m0); put(T_CM1, h->tabs.circ_m1); put(T_CAMP, h->tabs.circ_amp);
        put(T_CMASS1, h->tabs.circ_mass1); put(T_CPOIS, h->tabs.circ_pois);
        ok(hipMemcpy(h->d_tabs, T.data(), sizeof(double) * T.size(), hipMemcpyHostToDevice));
    }
    if (e != hipSuccess) {
        gempic_splitting_destroy(h);
        return fail(GEMPIC_ERR_DEVICE, std::string("device allocation: ") + hipGetErrorString(e));
    }
    set_dep_blocks(h);
    h->boris_blocks = std::max(1, std::min(h->max_blocks,
                                           h->cus * boris_blocks_per_cu(h->deg0, h->deg1,
                                                                        boris_shmem_bytes((int)h->nx))));
    *out = h;
    return GEMPIC_OK;
}

int gempic_splitting_destroy(gempic_splitting *h)
{
    if (!h) return GEMPIC_OK;
    (void)hipSetDevice(h->device);
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    void *bufs[] = {h->d_x, h->d_v1, h->d_v2, h->d_w, h->d_id, h->d_x2, h->d_v12, h->d_v22,
                    h->d_w2, h->d_id2, h->d_grid, h->d_tabs, h->d_part, h->d_gpart, h->d_cnt,
                    h->d_err, h->d_diag, h->d_sort_counts, h->d_sort_gsum, h->d_stage,
                    h->d_hist, h->d_ckpt, h->d_seg, h->d_lam, h->d_agrid, h->d_ids, h->d_wsnap,
                    h->d_perm};
    for (void *p : bufs)
        if (p) (void)hipFree(p);
    for (auto &p : h->pending) { (void)hipEventDestroy(p.a); (void)hipEventDestroy(p.b); }
    for (auto e : h->pool) (void)hipEventDestroy(e);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    transfer_release();
    delete h;
    return GEMPIC_OK;
}

static int ensure_stage(gempic_splitting *h)
{
    if (!h->d_stage) HIP_TRY(dalloc(&h->d_stage, (size_t)h->n * h->ld));
    return GEMPIC_OK;
}

int gempic_set_particles(gempic_splitting *h, const double *aos, int64_t ld, int64_t n)
{
    CHECK_H(h);
    if (!aos) return fail(GEMPIC_ERR_ARGUMENT, "particle array is NULL");
    if (ld != h->ld) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: leading dimension must be D+V+n_weights");
    if (n != h->n) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: particle count differs from the handle's");
    int rc = ensure_stage(h);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(h->d_stage, aos, sizeof(double) * (size_t)n * ld, hipMemcpyHostToDevice, h->stream));
    HIP_TRY(launch_aos_to_soa(h->d_stage, ld, n, h->dim_v, h->d_x, h->d_v1, h->d_v2, h->d_w, h->d_id, h->stream));
    h->particles_set = true;
    rc = run_sort(h);
    if (rc) return rc;
    return finish(h);
}

namespace {

int sample_args(int dim_v, int64_t n, double alpha, double k, double sigma, double dimx)
{
    if (dim_v != 1 && dim_v != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "MethodError: sample! is defined for ParticleGroup{1,1} and {1,2}");
    if (n < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: n_particles must be >= 1");
    if (!(k > 0.0) || !(alpha >= 0.0 && alpha < 1.0) || !(sigma >= 0.0) || !(dimx > 0.0))
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: need k > 0, 0 <= alpha < 1, sigma >= 0, dimx > 0");
    if (dim_v == 2) {
        // @assert mesh.dimx ≈ 2π / k (particle_sampling.jl:297)
        const double L = 6.283185307179586 / k;
        if (!(std::fabs(dimx - L) <= 1.4901161193847656e-8 * std::max(std::fabs(dimx), std::fabs(L))))
            return fail(GEMPIC_ERR_ASSERTION, "AssertionError: mesh.dimx ≈ 2π / k");
    }
    return GEMPIC_OK;
}

}  // namespace

int gempic_sample_landau(int dim_v, int64_t n, double alpha, double k, double sigma, double dimx,
                         double *aos, int64_t ld)
{
    int rc = sample_args(dim_v, n, alpha, k, sigma, dimx);
    if (rc) return rc;
    if (!aos) return fail(GEMPIC_ERR_ARGUMENT, "particle array is NULL");
    if (ld < 2 + dim_v) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: ld must be >= 2 + V");
    rc = check_device();
    if (rc) return rc;
    hipStream_t s = nullptr;
    double *dx_ = nullptr, *dv1 = nullptr, *dv2 = nullptr, *dw = nullptr, *dst = nullptr;
    int64_t *did = nullptr;
    int *derr = nullptr;
    hipError_t e = hipStreamCreate(&s);
    auto ok = [&](hipError_t r) { if (r != hipSuccess && e == hipSuccess) e = r; };
    ok(dalloc(&dx_, n)); ok(dalloc(&dv1, n)); ok(dalloc(&dv2, n)); ok(dalloc(&dw, n));
    ok(dalloc(&did, n)); ok(dalloc(&derr, 1)); ok(dalloc(&dst, (size_t)n * ld));
    int herr = 0;
    if (e == hipSuccess) {
        ok(hipMemsetAsync(derr, 0, sizeof(int), s));
        ok(hipMemsetAsync(dst, 0, sizeof(double) * (size_t)n * ld, s));
        ok(launch_sample_landau(n, dim_v, alpha, k, sigma, dimx, dx_, dv1, dv2, dw, did, derr, s));
        ok(launch_soa_to_aos(dst, ld, n, dim_v, dx_, dv1, dv2, dw, did, s));
        ok(hipMemcpyAsync(aos, dst, sizeof(double) * (size_t)n * ld, hipMemcpyDeviceToHost, s));
        ok(hipMemcpyAsync(&herr, derr, sizeof(int), hipMemcpyDeviceToHost, s));
        ok(hipStreamSynchronize(s));
    }
    void *bufs[] = {dx_, dv1, dv2, dw, did, derr, dst};
    for (void *p : bufs)
        if (p) (void)hipFree(p);
    if (s) (void)hipStreamDestroy(s);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("sample!: ") + hipGetErrorString(e));
    if (herr) return fail(GEMPIC_ERR_ARGUMENT, "newton did not converge in 200 iterations");
    return GEMPIC_OK;
}

int gempic_sample_landau_particles(gempic_splitting *h, double alpha, double k, double sigma)
{
    CHECK_H(h);
    int rc = sample_args(h->dim_v, h->n, alpha, k, sigma, h->Lx);
    if (rc) return rc;
    if (h->n_weights != 1) return fail(GEMPIC_ERR_ARGUMENT, "sample! sets one weight per particle");
    HIP_TRY(launch_sample_landau(h->n, h->dim_v, alpha, k, sigma, h->Lx, h->d_x, h->d_v1, h->d_v2,
                                 h->d_w, h->d_id, h->d_err, h->stream));
    h->particles_set = true;
    rc = run_sort(h);
    if (rc) return rc;
    rc = finish(h);
    if (rc == GEMPIC_ERR_INEXACT) return fail(GEMPIC_ERR_ARGUMENT, "newton did not converge in 200 iterations");
    return rc;
}

int gempic_get_particles(gempic_splitting *h, double *aos, int64_t ld, int64_t n)
{
    CHECK_H(h);
    CHECK_P(h);
    if (!aos) return fail(GEMPIC_ERR_ARGUMENT, "particle array is NULL");
    if (ld != h->ld) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: leading dimension must be D+V+n_weights");
    if (n != h->n) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: particle count differs from the handle's");
    int rc = ensure_stage(h);
    if (rc) return rc;
    HIP_TRY(launch_soa_to_aos(h->d_stage, ld, n, h->dim_v, h->d_x, h->d_v1, h->d_v2, h->d_w, h->d_id, h->stream));
    HIP_TRY(to_host(aos, h->d_stage, sizeof(double) * (size_t)n * ld, h->stream, h->device));
    return finish(h);
}

int gempic_set_fields(gempic_splitting *h, const double *e1, const double *e2, const double *b)
{
    CHECK_H(h);
    const size_t nb = sizeof(double) * h->nx;
    if (e1) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E1 * h->nx, e1, nb, hipMemcpyHostToDevice, h->stream));
    if (e2) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E2 * h->nx, e2, nb, hipMemcpyHostToDevice, h->stream));
    if (b) HIP_TRY(hipMemcpyAsync(h->d_grid + S_B * h->nx, b, nb, hipMemcpyHostToDevice, h->stream));
    return finish(h);
}

// `count` neighbouring grid slots from `slot` on, in one copy, then to the
// caller's arrays (any of them may be NULL)
static int get_slots(gempic_splitting *h, int slot, int count, double *const *out)
{
    double tmp[3 * kNxMax];
    HIP_TRY(hipMemcpyAsync(tmp, h->d_grid + slot * h->nx, sizeof(double) * count * h->nx, hipMemcpyDeviceToHost,
                           h->stream));
    const int rc = finish(h);
    if (rc == GEMPIC_ERR_DEVICE) return rc;
    for (int k = 0; k < count; ++k)
        if (out[k]) std::memcpy(out[k], tmp + k * h->nx, sizeof(double) * h->nx);
    return rc;
}

int gempic_get_fields(gempic_splitting *h, double *e1, double *e2, double *b)
{
    CHECK_H(h);
    static_assert(S_E2 == S_E1 + 1 && S_B == S_E1 + 2, "neighbouring slots");
    double *const out[3] = {e1, e2, b};
    return get_slots(h, S_E1, 3, out);
}

int gempic_get_j(gempic_splitting *h, double *j1, double *j2)
{
    CHECK_H(h);
    static_assert(S_J2 == S_J1 + 1, "neighbouring slots");
    double *const out[2] = {j1, j2};
    return get_slots(h, S_J1, 2, out);
}

// the mode bit of the handle's arithmetic for its 1d2v particle passes
static int fm(const gempic_splitting *h) { return h->arith == GEMPIC_ARITH_FUSED ? M_FAST : 0; }

int gempic_operator_hb(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    int rc;
    if (h->dim_v == 2) {
        rc = run_grid(h, prog1(G_HB, dt, S_B, S_B, S_E2));
    } else {
        CHECK_P(h);
        rc = run_pass(h, M_V1 | M_HE, dt, 0.0, 0.0, 0, 7);
    }
    if (rc) return rc;
    return finish(h);
}

int gempic_operator_he(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    if (h->dim_v != 2) return fail(GEMPIC_ERR_ARGUMENT, "MethodError: operatorHE is defined for 1d2v only");
    int rc = run_pass(h, fm(h) | M_HE, dt, 0.0, 0.0, 0, 2);
    if (rc) return rc;
    return finish(h);
}

int gempic_operator_hp2(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    if (h->dim_v != 2) return fail(GEMPIC_ERR_ARGUMENT, "MethodError: operatorHp2 is defined for 1d2v only");
    int rc = run_pass(h, fm(h) | M_HP2A, 0.0, dt, 0.0, 0, 3);
    if (rc) return rc;
    return finish(h);
}

int gempic_operator_hp1(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    int mode = h->dim_v == 2 ? (fm(h) | M_HP1) : (M_V1 | M_HP1);
    int rc = run_pass(h, mode, 0.0, 0.0, dt, 0, 4);
    if (rc) return rc;
    return finish(h);
}

static int maybe_sort(gempic_splitting *h)
{
    if (h->sort_interval > 0 && h->steps_since_sort >= h->sort_interval) return run_sort(h);
    return GEMPIC_OK;
}

int gempic_strang_splitting(gempic_splitting *h, double dt, int64_t n_steps, int flags)
{
    CHECK_H(h);
    CHECK_P(h);
    if (n_steps < 0) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: number_steps must be >= 0");
    if (n_steps == 0) return finish(h);
    const double hdt = 0.5 * dt;
    int rc = GEMPIC_OK;
    const bool substep = (flags & GEMPIC_STRANG_SUBSTEP) != 0;
    if (h->dim_v == 2) {
        if (substep) {
            for (int64_t s = 0; s < n_steps && !rc; ++s) {
                rc = maybe_sort(h);
                if (!rc) rc = run_grid(h, prog1(G_HB, hdt, S_B, S_B, S_E2));
                if (!rc) rc = run_pass(h, fm(h) | M_HE, hdt, 0, 0, 0, 2);
                if (!rc) rc = run_pass(h, fm(h) | M_HP2A, 0, hdt, 0, 0, 3);
                if (!rc) rc = run_pass(h, fm(h) | M_HP1, 0, 0, 1.0 * dt, 0, 4);
                if (!rc) rc = run_pass(h, fm(h) | M_HP2A, 0, hdt, 0, 0, 3);
                if (!rc) rc = run_pass(h, fm(h) | M_HE, hdt, 0, 0, 0, 2);
                if (!rc) rc = run_grid(h, prog1(G_HB, hdt, S_B, S_B, S_E2));
                h->steps_since_sort++;
            }
        } else {
            // HB(dt/2) and HE's B update of the first step touch only fields
            GridProg g = prog1(G_HB, hdt, S_B, S_B, S_E2);
            prog_add(g, G_HE_B, hdt, S_E2, S_E2, S_B);
            rc = run_grid(h, g);
            for (int64_t s = 0; s < n_steps && !rc; ++s) {
                rc = maybe_sort(h);
                const int prev = s == 0 ? 0 : M_HE_PREV;
                const int more = s + 1 < n_steps;
                if (h->kernels_per_step == 1) {
                    const int mode = fm(h) | prev | M_HE | M_HP2A | M_HP1 | M_HP2B;
                    if (!rc) rc = run_pass(h, mode, hdt, hdt, 1.0 * dt, more, 0);
                } else {
                    // HE pair + first Hp2, then Hp1 + second Hp2 with the field solves;
                    // Hp1 reads only B, which the first Hp2's solve leaves unchanged
                    if (!rc) rc = run_pass(h, prev | M_HE | M_HP2A | M_NOEPI, hdt, hdt, 0, 0, 8);
                    if (!rc) rc = run_pass(h, M_HP1 | M_HP2B | M_WITH_J2A, hdt, hdt, 1.0 * dt, more, 0);
                }
                h->steps_since_sort++;
            }
            if (!rc) rc = run_pass(h, fm(h) | M_HE_PREV, hdt, 0, 0, 0, 1);
        }
    } else {
        if (substep) {
            for (int64_t s = 0; s < n_steps && !rc; ++s) {
                rc = maybe_sort(h);
                if (!rc) rc = run_pass(h, M_V1 | M_HE, hdt, 0, 0, 0, 7);
                if (!rc) rc = run_pass(h, M_V1 | M_HP1, 0, 0, dt, 0, 4);
                if (!rc) rc = run_pass(h, M_V1 | M_HE, hdt, 0, 0, 0, 7);
                h->steps_since_sort++;
            }
        } else {
            for (int64_t s = 0; s < n_steps && !rc; ++s) {
                rc = maybe_sort(h);
                const int mode = M_V1 | (s == 0 ? 0 : M_HE_PREV) | M_HE | M_HP1;
                if (!rc) rc = run_pass(h, mode, hdt, 0, dt, s + 1 < n_steps, 0);
                h->steps_since_sort++;
            }
            if (!rc) rc = run_pass(h, M_V1 | M_HE_PREV, hdt, 0, 0, 0, 1);
        }
    }
    if (rc) return rc;
    if (flags & GEMPIC_ASYNC) return GEMPIC_OK;
    return finish(h);
}

// ---------------------------------------------------------------------------
// Reverse mode of strang_splitting! (1d2v): the forward run records the
// fields of every step and checkpoints the particles every K steps; the
// reverse sweep re-runs each interval of K steps forward from its checkpoint
// (k_adj1d R_FWD, no deposits) and then steps back through it with the
// reverse passes and their field parts.
// ---------------------------------------------------------------------------
namespace {

int grow(double **p, size_t *cap, size_t need)
{
    if (*cap >= need && *p) return GEMPIC_OK;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    HIP_TRY(dalloc(p, need));
    *cap = need;
    return GEMPIC_OK;
}

AdjArgs adj_args(gempic_splitting *h, double dt, const Launch &L)
{
    AdjArgs A;
    std::memset(&A, 0, sizeof(A));
    A.p = pass_args(h);
    A.p.hist = nullptr;
    A.p.chunk = L.chunk;
    A.p.iters = L.iters;
    A.p.ngroups = L.ngroups;
    set_generations(A.p, L, h->cus, kAdjGenSkew);
    const double hdt = 0.5 * dt;
    A.p.dt_he = hdt;
    A.p.dt_hp2 = hdt;
    A.p.dt_hp1 = 1.0 * dt;
    A.p.dtqm_he = hdt * h->qm;
    A.p.dtqm_hp2 = hdt * h->qm;
    A.agrid = h->d_agrid;
    A.lx = h->d_lam;
    A.lv1 = h->d_lam + h->n;
    A.lv2 = h->d_lam + 2 * h->n;
    return A;
}

int adj_launch(gempic_splitting *h, int rm, const AdjArgs &A, int blocks)
{
    ProfScope ps(h, (rm & R_REV) ? 10 : (rm & R_FWD) ? 11 : 7);
    hipError_t e = launch_adj(h->deg0, h->deg1, rm, A, blocks, h->stream);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("reverse pass launch: ") + hipGetErrorString(e));
    return GEMPIC_OK;
}

int adj_epi(gempic_splitting *h, int kind, const AdjArgs &A, int blocks)
{
    ProfScope ps(h, 12);
    hipError_t e = launch_adj_epi(kind, A, blocks, h->stream);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("reverse field part launch: ") + hipGetErrorString(e));
    return GEMPIC_OK;
}

// Sort epochs a reverse-mode call of T steps with checkpoints every K can
// start: the first at step 1, then one per sort. Sorts run only where an
// interval starts after the first (intervals 1 .. nck-1), the first of them
// as early as interval 1 (the handle may enter the call with a sort due), the
// others at least ceil(sort_interval / K) intervals apart; none when the
// handle never sorts.
int64_t adj_epoch_bound(const gempic_splitting *h, int64_t T, int64_t K)
{
    const int64_t nck = (T + K - 1) / K;
    if (h->sort_interval <= 0 || nck < 2) return 1;
    const int64_t gap = (h->sort_interval + K - 1) / K;
    return std::min<int64_t>(nck, 2 + (nck - 2) / gap);
}

// the epoch about to start at a due sort must fit the reserved epochs
int adj_epoch_check(const gempic_splitting *h, int64_t ne)
{
    const bool due = h->sort_interval > 0 && h->steps_since_sort >= h->sort_interval;
    if (due && ne >= h->epoch_cap)
        return fail(GEMPIC_ERR_ASSERTION, "AssertionError: more sort epochs than reserved in the reverse mode");
    return GEMPIC_OK;
}

int adj_workspace(gempic_splitting *h, int64_t T, int64_t K)
{
    const size_t n = (size_t)h->n, nx = (size_t)h->nx;
    const size_t nck = (size_t)((T + K - 1) / K);
    const size_t nep = (size_t)adj_epoch_bound(h, T, K);
    int rc = grow(&h->d_hist, &h->hist_cap, (size_t)(T + 2) * NHIST * nx);
    if (!rc) rc = grow(&h->d_ckpt, &h->ckpt_cap, nck * 3 * n);
    if (!rc) rc = grow(&h->d_wsnap, &h->wsnap_cap, nep * n);
    if (!rc && h->ids_cap < n) {
        HIP_TRY(dalloc(&h->d_ids, n));
        h->ids_cap = n;
    }
    if (!rc && h->perm_cap < nep * n) {
        if (h->d_perm) (void)hipFree(h->d_perm);
        h->d_perm = nullptr;
        h->perm_cap = 0;
        HIP_TRY(dalloc(&h->d_perm, nep * n));
        h->perm_cap = nep * n;
    }
    if (!rc) h->epoch_cap = (int64_t)nep;
    if (!rc && K > 1) rc = grow(&h->d_seg, &h->seg_cap, (size_t)(K - 1) * 3 * n);
    if (!rc && !h->d_lam) HIP_TRY(dalloc(&h->d_lam, 3 * n));
    if (!rc && !h->d_agrid) HIP_TRY(dalloc(&h->d_agrid, (size_t)NASLOT * nx));
    if (!rc && !h->adj_blocks)
        h->adj_blocks = std::max(1, std::min(h->max_blocks,
                                             h->cus * adj_blocks_per_cu(h->deg0, h->deg1, R_REV)));
    return rc;
}

}  // namespace

int gempic_strang_splitting_adjoint(gempic_splitting *h, double dt, int64_t n_steps,
                                    int64_t checkpoint_every, double loss_weight,
                                    const double *ct_particles, int64_t ld, const double *ct_e1,
                                    const double *ct_e2, const double *ct_b, int flags)
{
    CHECK_H(h);
    CHECK_P(h);
    if (h->dim_v != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: the reverse mode covers the 1d2v Strang splitting");
    if (n_steps < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: number_steps must be >= 1");
    if (checkpoint_every < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: checkpoint_every must be >= 1");
    if (h->nx > kAdjNxMax || h->nx < 4)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: the reverse mode needs 4 <= nx <= 128");
    if (ct_particles && ld != h->ld)
        return fail(GEMPIC_ERR_ASSERTION, "AssertionError: leading dimension must be D+V+n_weights");
    const int64_t T = n_steps, K = std::min<int64_t>(checkpoint_every, n_steps);
    struct RecordOff {      // no record pointers survive the call, on any path
        gempic_splitting *h;
        ~RecordOff() { h->cur_hist = nullptr; h->cur_cx = nullptr; h->cur_perm = nullptr; }
    } record_off{h};
    int rc = adj_workspace(h, T, K);
    if (!rc) rc = ensure_stage(h);
    if (rc) return rc;
    h->adj_ready = false;
    const size_t n = (size_t)h->n, nx = (size_t)h->nx;
    const size_t nb = sizeof(double) * n;
    const double hdt = 0.5 * dt;
    double *hist = h->d_hist;
    auto rec = [&](int64_t s) { return hist + (size_t)s * NHIST * nx; };

    // ---- forward, recorded ----
    // B before the first step (the prologue's HB reads it)
    HIP_TRY(hipMemcpyAsync(rec(0) + H_BEND * nx, h->d_grid + S_B * nx, sizeof(double) * nx,
                           hipMemcpyDeviceToDevice, h->stream));
    GridProg g = prog1(G_HB, hdt, S_B, S_B, S_E2);
    prog_add(g, G_HE_B, hdt, S_E2, S_E2, S_B);
    rc = run_grid(h, g);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(rec(1), h->d_grid, sizeof(double) * 4 * nx, hipMemcpyDeviceToDevice, h->stream));
    // Particles are re-sorted only where a checkpoint interval starts (when
    // the sort interval has passed), so each interval runs in one particle
    // order. Each sort starts an epoch whose weights and order (id) are
    // kept, to run the interval's reverse passes and to carry the particle
    // cotangents across the sort on the way back. The fused pass that ends an
    // interval stores its state into the next checkpoint itself (a copy is
    // made only after a sort); with one step per interval nothing is re-run on
    // the way back.
    const int64_t nck = (T + K - 1) / K;
    std::vector<int64_t> epoch_of((size_t)nck, 0);
    int64_t ne = 0;
    for (int64_t s = 1; s <= T && !rc; ++s) {
        if ((s - 1) % K == 0) {
            const size_t j = (size_t)((s - 1) / K);
            bool sorted = false;
            if (s > 1) {
                rc = adj_epoch_check(h, ne);
                if (rc) break;
                h->cur_perm = h->d_perm + (size_t)ne * n;     // this epoch's, if a sort runs
                rc = maybe_sort(h);
                h->cur_perm = nullptr;
                if (rc) break;
                sorted = h->steps_since_sort == 0;
            } else {
                HIP_TRY(hipMemcpyAsync(h->d_ids, h->d_id, sizeof(int64_t) * n, hipMemcpyDeviceToDevice,
                                       h->stream));
            }
            if (s == 1 || sorted) {
                HIP_TRY(hipMemcpyAsync(h->d_wsnap + (size_t)ne * n, h->d_w, nb, hipMemcpyDeviceToDevice,
                                       h->stream));
                ++ne;
            }
            epoch_of[j] = ne - 1;
            if (s == 1 || sorted) {
                double *ck = h->d_ckpt + j * 3 * n;
                HIP_TRY(hipMemcpyAsync(ck, h->d_x, nb, hipMemcpyDeviceToDevice, h->stream));
                HIP_TRY(hipMemcpyAsync(ck + n, h->d_v1, nb, hipMemcpyDeviceToDevice, h->stream));
                HIP_TRY(hipMemcpyAsync(ck + 2 * n, h->d_v2, nb, hipMemcpyDeviceToDevice, h->stream));
            }
        }
        h->cur_hist = rec(s);
        // the pass that ends an interval stores its state as the next checkpoint
        h->cur_cx = (s % K == 0 && s < T) ? h->d_ckpt + (size_t)(s / K) * 3 * n : nullptr;
        const int mode = (s > 1 ? M_HE_PREV : 0) | M_HE | M_HP2A | M_HP1 | M_HP2B;
        rc = run_pass(h, mode, hdt, hdt, 1.0 * dt, s < T, 0);
        h->steps_since_sort++;
    }
    h->cur_cx = nullptr;
    h->cur_hist = nullptr;
    if (!rc) rc = run_pass(h, M_HE_PREV, hdt, 0, 0, 0, 1);
    if (rc) return rc;

    // ---- reverse ----
    const Launch L = plan(h->n, h->adj_blocks);
    AdjArgs A = adj_args(h, dt, L);
    A.wloss = loss_weight;
    HIP_TRY(hipMemsetAsync(h->d_agrid, 0, sizeof(double) * NASLOT * nx, h->stream));
    const size_t fb = sizeof(double) * nx;
    if (ct_e1) HIP_TRY(hipMemcpyAsync(h->d_agrid + A_E1 * nx, ct_e1, fb, hipMemcpyHostToDevice, h->stream));
    if (ct_e2) HIP_TRY(hipMemcpyAsync(h->d_agrid + A_E2 * nx, ct_e2, fb, hipMemcpyHostToDevice, h->stream));
    if (ct_b) HIP_TRY(hipMemcpyAsync(h->d_agrid + A_B * nx, ct_b, fb, hipMemcpyHostToDevice, h->stream));
    if (ct_particles) {
        HIP_TRY(hipMemcpyAsync(h->d_stage, ct_particles, sizeof(double) * n * h->ld,
                               hipMemcpyHostToDevice, h->stream));
        HIP_TRY(launch_adj_rows_in(h->d_stage, h->ld, h->n, h->d_id, A.lx, A.lv1, A.lv2, h->stream));
    } else {
        HIP_TRY(hipMemsetAsync(h->d_lam, 0, 3 * nb, h->stream));
    }
    // the trailing HE, then the field part of the last step
    A.x = h->d_x;
    A.fields = rec(T + 1);
    rc = adj_launch(h, R_HEONLY, A, L.blocks);
    A.bend = rec(T) + H_BEND * nx;
    if (!rc) rc = adj_epi(h, AE_TAIL, A, L.blocks);
    for (int64_t j = nck - 1; j >= 0 && !rc; --j) {
        const int64_t s_lo = j * K + 1, s_hi = std::min((j + 1) * K, T);
        // state before step s: the checkpoint for s = s_lo, else the recompute buffer
        auto state = [&](int64_t s, double **x, double **v1, double **v2) {
            double *b = s == s_lo ? h->d_ckpt + (size_t)j * 3 * n : h->d_seg + (size_t)(s - s_lo - 1) * 3 * n;
            *x = b;
            *v1 = b + n;
            *v2 = b + 2 * n;
        };
        A.p.w = h->d_wsnap + (size_t)epoch_of[(size_t)j] * n;   // the interval's particle order
        for (int64_t s = s_lo; s < s_hi && !rc; ++s) {
            double *x, *v1, *v2;
            state(s, &x, &v1, &v2);
            A.x = x; A.v1 = v1; A.v2 = v2;
            state(s + 1, &A.xo, &A.v1o, &A.v2o);
            A.fields = rec(s);
            rc = adj_launch(h, R_FWD | (s > 1 ? R_PREV : 0), A, L.blocks);
        }
        for (int64_t s = s_hi; s >= s_lo && !rc; --s) {
            double *x, *v1, *v2;
            state(s, &x, &v1, &v2);
            A.x = x; A.v1 = v1; A.v2 = v2;
            A.fields = rec(s);
            rc = adj_launch(h, R_REV | (s > 1 ? R_PREV : 0), A, L.blocks);
            if (rc) break;
            if (s > 1) {
                A.bend = rec(s - 1) + H_BEND * nx;
                rc = adj_epi(h, AE_STEP, A, L.blocks);
            } else {
                A.bend = rec(0) + H_BEND * nx;
                rc = adj_epi(h, AE_HEAD, A, L.blocks);
            }
        }
        // into the particle order of the previous interval when a sort ran between them
        if (!rc && j > 0 && epoch_of[(size_t)j] != epoch_of[(size_t)j - 1]) {
            double *other = A.lx == h->d_lam ? h->d_stage : h->d_lam;
            hipError_t e = launch_adj_unsort(h->d_perm + (size_t)epoch_of[(size_t)j] * n, h->n, A.lx,
                                             other, h->stream);
            if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("unsort launch: ") + hipGetErrorString(e));
            A.lx = other;
            A.lv1 = other + n;
            A.lv2 = other + 2 * n;
        }
    }
    if (rc) return rc;
    if (A.lx != h->d_lam)
        HIP_TRY(hipMemcpyAsync(h->d_lam, A.lx, 3 * nb, hipMemcpyDeviceToDevice, h->stream));
    h->adj_id0 = h->d_ids;
    h->adj_ready = true;
    if (flags & GEMPIC_ASYNC) return GEMPIC_OK;
    return finish(h);
}

int gempic_get_adjoint(gempic_splitting *h, double *loss, double *g_particles, int64_t ld, int64_t n,
                       double *g_e1, double *g_e2, double *g_b)
{
    CHECK_H(h);
    if (!h->adj_ready) return fail(GEMPIC_ERR_STATE, "no reverse-mode result: call gempic_strang_splitting_adjoint first");
    const size_t nx = (size_t)h->nx, fb = sizeof(double) * nx;
    if (g_particles) {
        if (ld != h->ld) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: leading dimension must be D+V+n_weights");
        if (n != h->n) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: particle count differs from the handle's");
        int rc = ensure_stage(h);
        if (rc) return rc;
        // the cotangents are in the particle order the call started from
        HIP_TRY(launch_adj_rows_out(h->d_stage, ld, n, h->adj_id0, h->d_lam, h->d_lam + n,
                                    h->d_lam + 2 * n, h->stream));
        HIP_TRY(to_host(g_particles, h->d_stage, sizeof(double) * (size_t)n * ld, h->stream, h->device));
    }
    if (g_e1) HIP_TRY(hipMemcpyAsync(g_e1, h->d_agrid + A_E1 * nx, fb, hipMemcpyDeviceToHost, h->stream));
    if (g_e2) HIP_TRY(hipMemcpyAsync(g_e2, h->d_agrid + A_E2 * nx, fb, hipMemcpyDeviceToHost, h->stream));
    if (g_b) HIP_TRY(hipMemcpyAsync(g_b, h->d_agrid + A_B * nx, fb, hipMemcpyDeviceToHost, h->stream));
    if (loss) HIP_TRY(hipMemcpyAsync(loss, h->d_agrid + A_LOSS * nx, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    return finish(h);
}

int gempic_get_adjoint_domain(gempic_splitting *h, double *g_length, double *g_weight_sum)
{
    CHECK_H(h);
    if (!h->adj_ready) return fail(GEMPIC_ERR_STATE, "no reverse-mode result: call gempic_strang_splitting_adjoint first");
    double sc[4] = {0, 0, 0, 0};
    HIP_TRY(hipMemcpyAsync(sc, h->d_agrid + A_LOSS * h->nx, sizeof(sc), hipMemcpyDeviceToHost, h->stream));
    int rc = finish(h);
    if (rc) return rc;
    // dx = Lx / nx: d/d Lx = (1/nx) d/d dx, plus the mod's periods
    if (g_length) *g_length = sc[AS_DX] / (double)h->nx + sc[AS_MOD];
    if (g_weight_sum) *g_weight_sum = sc[AS_W];
    return GEMPIC_OK;
}

int gempic_solve_poisson_adjoint(gempic_splitting *h, const double *ct_e, double *g_x)
{
    CHECK_H(h);
    CHECK_P(h);
    if (!ct_e || !g_x) return fail(GEMPIC_ERR_ARGUMENT, "ct_e and g_x must not be NULL");
    if (h->nx > kAdjNxMax) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: the reverse mode needs nx <= 128");
    int rc = adj_workspace(h, 1, 1);
    if (!rc) rc = ensure_stage(h);
    if (rc) return rc;
    h->adj_ready = false;
    const size_t nx = (size_t)h->nx, n = (size_t)h->n;
    const Launch L = plan(h->n, h->adj_blocks);
    AdjArgs A = adj_args(h, 0.0, L);
    A.x = h->d_x;
    HIP_TRY(hipMemcpyAsync(h->d_agrid + A_NU * nx, ct_e, sizeof(double) * nx, hipMemcpyHostToDevice, h->stream));
    rc = adj_epi(h, AE_POIS, A, 0);
    if (!rc) rc = adj_launch(h, R_POIS, A, L.blocks);
    if (rc) return rc;
    // one row out, through the caller's order: rows 0..2 of a 3-row staging array
    HIP_TRY(launch_adj_rows_out(h->d_stage, 3, h->n, h->d_id, A.lx, A.lx, A.lx, h->stream));
    std::vector<double> tmp(3 * n);
    HIP_TRY(hipMemcpyAsync(tmp.data(), h->d_stage, sizeof(double) * 3 * n, hipMemcpyDeviceToHost, h->stream));
    rc = finish(h);
    if (rc) return rc;
    for (size_t i = 0; i < n; ++i) g_x[i] = tmp[3 * i];
    return GEMPIC_OK;
}

// ---------------------------------------------------------------------------
// HamiltonianSplittingBoris (hamiltonian_splitting_boris.jl) on the handle's
// state: e_dofs, b_dofs and j_dofs are the handle's fields, e_dofs_mid and
// b_dofs_mid its S_E1M, S_E2M, S_BM slots (zero at creation, :50-60).
// ---------------------------------------------------------------------------
namespace {

int run_boris(gempic_splitting *h, int ops, double dt_e, double dt_b, double dt_x, int kind,
              int more, int prof_id)
{
    PassArgs a = pass_args(h);
    const int target = h->override_blocks ? h->override_blocks : h->boris_blocks;
    Launch L = plan(h->n, target);
    a.chunk = L.chunk;
    a.iters = L.iters;
    a.ngroups = L.ngroups;
    set_generations(a, L, h->cus);
    a.dtqm_he = dt_e * h->qm;              // dt * qm .* [E1, E2]
    a.dtqm_hp2 = h->qm * 0.5 * dt_b;       // qm * 0.5 * dt
    a.dt_hp1 = dt_x;
    a.more = more;
    a.rgroups = epi_groups(L.blocks);
    {
        ProfScope ps(h, prof_id);
        hipError_t e = launch_boris(h->deg0, h->deg1, ops, kind, a, L.blocks, boris_shmem_bytes((int)h->nx),
                                    h->stream);
        if (e != hipSuccess)
            return fail(GEMPIC_ERR_DEVICE, std::string("Boris pass launch: ") + hipGetErrorString(e));
    }
    return GEMPIC_OK;
}

int boris_check(gempic_splitting *h)
{
    if (h->dim_v != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "MethodError: HamiltonianSplittingBoris needs ParticleGroup{1,2}");
    return GEMPIC_OK;
}

}  // namespace

int gempic_boris_push_v_epart(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = boris_check(h);
    if (!rc) rc = run_boris(h, BO_EPART, dt, 0.0, 0.0, BE_J, 0, 2);
    if (rc) return rc;
    return finish(h);
}

int gempic_boris_push_v_bpart(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = boris_check(h);
    if (!rc) rc = run_boris(h, BO_BPART, 0.0, dt, 0.0, BE_J, 0, 3);
    if (rc) return rc;
    return finish(h);
}

int gempic_boris_push_x_accumulate_j(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = boris_check(h);
    if (!rc) rc = run_boris(h, BO_PUSHX, 0.0, 0.0, dt, BE_J, 0, 4);
    if (rc) return rc;
    return finish(h);
}

int gempic_boris_staggering(gempic_splitting *h, double dt)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = boris_check(h);
    if (!rc) rc = run_boris(h, BO_PUSHX, 0.0, 0.0, dt * 0.5, BE_STAGGER, 0, 4);
    if (rc) return rc;
    return finish(h);
}

int gempic_boris_strang_splitting(gempic_splitting *h, double dt, int64_t n_steps, int flags)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = boris_check(h);
    if (rc) return rc;
    if (n_steps < 0) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: number_steps must be >= 0");
    if (n_steps == 0) return finish(h);
    // the first step's B_mid = (B + b_from_e(B, dt, E2_mid)) / 2 (:138-144);
    // the later steps' run at the end of the previous step's field part
    GridProg g = prog1(G_COPY, 0.0, S_B, S_B, S_BM);
    prog_add(g, G_HE_B, dt, S_E2M, S_E2M, S_B);
    prog_add(g, G_AVG, 0.0, S_B, S_B, S_BM);
    rc = run_grid(h, g);
    const int all = BO_EPART | BO_BPART | BO_EPART2 | BO_PUSHX;
    for (int64_t s = 0; s < n_steps && !rc; ++s) {
        rc = maybe_sort(h);
        if (!rc) rc = run_boris(h, all, 0.5 * dt, dt, dt, BE_STEP, s + 1 < n_steps, 0);
        h->steps_since_sort++;
    }
    if (rc) return rc;
    if (flags & GEMPIC_ASYNC) return GEMPIC_OK;
    return finish(h);
}

int gempic_boris_set_mid(gempic_splitting *h, const double *e1_mid, const double *e2_mid,
                         const double *b_mid)
{
    CHECK_H(h);
    const size_t nb = sizeof(double) * h->nx;
    if (e1_mid) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E1M * h->nx, e1_mid, nb, hipMemcpyHostToDevice, h->stream));
    if (e2_mid) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E2M * h->nx, e2_mid, nb, hipMemcpyHostToDevice, h->stream));
    if (b_mid) HIP_TRY(hipMemcpyAsync(h->d_grid + S_BM * h->nx, b_mid, nb, hipMemcpyHostToDevice, h->stream));
    return finish(h);
}

int gempic_boris_get_mid(gempic_splitting *h, double *e1_mid, double *e2_mid, double *b_mid)
{
    CHECK_H(h);
    const size_t nb = sizeof(double) * h->nx;
    if (e1_mid) HIP_TRY(hipMemcpyAsync(e1_mid, h->d_grid + S_E1M * h->nx, nb, hipMemcpyDeviceToHost, h->stream));
    if (e2_mid) HIP_TRY(hipMemcpyAsync(e2_mid, h->d_grid + S_E2M * h->nx, nb, hipMemcpyDeviceToHost, h->stream));
    if (b_mid) HIP_TRY(hipMemcpyAsync(b_mid, h->d_grid + S_BM * h->nx, nb, hipMemcpyDeviceToHost, h->stream));
    return finish(h);
}

// ---------------------------------------------------------------------------
// Ensembles: independent splittings (each with its own particles, grid,
// domain and tables) stepped together, one particle-pass launch and one
// field-part launch per Strang step for all of them. Each instance keeps the
// launch geometry of its own strang_splitting!, so its results are bit for
// bit those of a stand-alone run.
// ---------------------------------------------------------------------------
struct gempic_ensemble {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<gempic_splitting *> hs;
    int p0 = 3, p1 = 2, max_nx = 0;
    PassArgs *d_args = nullptr;        // [2][ninst]: another step follows / the last step
    int *d_bstart = nullptr, *d_estart = nullptr;
    std::vector<int> bstart, estart;
    SortArgs *d_sargs = nullptr;       // the batched sort's tables
    int *d_tstart = nullptr, *d_gstart = nullptr;
    AdjArgs *d_aargs = nullptr;        // the batched reverse mode's arguments and tables
    int *d_abstart = nullptr, *d_aestart = nullptr;
    // GEMPIC_GRAPH: the regular step (pass and field part) as a HIP graph,
    // with the launch geometry it was captured for
    hipGraphExec_t step_graph = nullptr;
    int graph_blocks = 0, graph_groups = 0, graph_mode = -1;
    size_t graph_sh_pass = 0, graph_sh_epi = 0;
};

namespace {

// per-instance arguments of the fused pass (more = 1 and more = 0) and the
// workgroup tables; uploaded again after a re-sort moves the particle arrays
int ens_upload(gempic_ensemble *e, const double *dts)
{
    const size_t ni = e->hs.size();
    std::vector<PassArgs> args(2 * ni);
    e->bstart.assign(ni + 1, 0);
    e->estart.assign(ni + 1, 0);
    for (size_t i = 0; i < ni; ++i) {
        gempic_splitting *h = e->hs[i];
        const double dt = dts[i], hdt = 0.5 * dt;
        const int target = h->override_blocks ? h->override_blocks : h->dep_blocks;
        const Launch L = plan(h->n, target);
        PassArgs a = pass_args(h);
        a.chunk = L.chunk;
        a.iters = L.iters;
        a.ngroups = L.ngroups;
        set_generations(a, L, h->cus);
        a.dt_he = hdt;
        a.dt_hp2 = hdt;
        a.dt_hp1 = 1.0 * dt;
        a.dtqm_he = hdt * h->qm;
        a.dtqm_hp2 = hdt * h->qm;
        a.more = 1;
        args[i] = a;
        a.more = 0;
        args[ni + i] = a;
        e->bstart[i + 1] = e->bstart[i] + L.blocks;
        e->estart[i + 1] = e->estart[i] + epi_groups(L.blocks);
    }
    HIP_TRY(hipMemcpy(e->d_args, args.data(), sizeof(PassArgs) * args.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(e->d_bstart, e->bstart.data(), sizeof(int) * (ni + 1), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(e->d_estart, e->estart.data(), sizeof(int) * (ni + 1), hipMemcpyHostToDevice));
    return GEMPIC_OK;
}

// SortArgs of a handle's sort (run_sort's), into its double buffer
SortArgs sort_args(gempic_splitting *h)
{
    SortArgs s;
    std::memset(&s, 0, sizeof(s));
    s.n = h->n;
    s.nx = (int)h->nx;
    s.sub = h->sortg.sub;
    s.nbins = h->sortg.nbins;
    s.ntiles = h->sortg.ntiles;
    s.tiles_per_group = h->sortg.tiles_per_group;
    s.ngroups = h->sortg.ngroups;
    s.xmin = h->xmin;
    s.dx = h->dx;
    s.x = h->d_x; s.v1 = h->d_v1; s.v2 = h->d_v2; s.w = h->d_w; s.id = h->d_id;
    s.x2 = h->d_x2; s.v12 = h->d_v12; s.v22 = h->d_v22; s.w2 = h->d_w2; s.id2 = h->d_id2;
    s.counts = h->d_sort_counts;
    s.gsum = h->d_sort_gsum;
    s.perm = h->cur_perm;
    return s;
}

void sort_swap(gempic_splitting *h)
{
    std::swap(h->d_x, h->d_x2);
    std::swap(h->d_v1, h->d_v12);
    std::swap(h->d_v2, h->d_v22);
    std::swap(h->d_w, h->d_w2);
    std::swap(h->d_id, h->d_id2);
    h->steps_since_sort = 0;
}

// the sorts that are due, in one launch per stage
int ens_sort(gempic_ensemble *e, bool *any)
{
    std::vector<SortArgs> args;
    std::vector<int> tstart(1, 0), gstart(1, 0);
    std::vector<gempic_splitting *> due;
    int max_bins = 1;
    for (auto *h : e->hs)
        if (h->sort_interval > 0 && h->steps_since_sort >= h->sort_interval) {
            SortArgs a = sort_args(h);
            args.push_back(a);
            tstart.push_back(tstart.back() + (a.ntiles + kWaves - 1) / kWaves);
            gstart.push_back(gstart.back() + a.ngroups);
            max_bins = std::max(max_bins, a.nbins);
            due.push_back(h);
        }
    *any = !due.empty();
    if (due.empty()) return GEMPIC_OK;
    const size_t nd = due.size();
    HIP_TRY(hipMemcpy(e->d_sargs, args.data(), sizeof(SortArgs) * nd, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(e->d_tstart, tstart.data(), sizeof(int) * (nd + 1), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(e->d_gstart, gstart.data(), sizeof(int) * (nd + 1), hipMemcpyHostToDevice));
    SortBatch b;
    b.args = e->d_sargs;
    b.tile_start = e->d_tstart;
    b.group_start = e->d_gstart;
    b.ninst = (int)nd;
    HIP_TRY(launch_sort_batch(b, tstart.back(), gstart.back(), max_bins, e->stream));
    for (auto *h : due) sort_swap(h);
    return GEMPIC_OK;
}

// the instances' own work (sorts, field programs) goes to the ensemble's
// stream for the duration of an ensemble call
struct EnsStreams {
    gempic_ensemble *e;
    std::vector<hipStream_t> saved;
    explicit EnsStreams(gempic_ensemble *ee) : e(ee)
    {
        for (auto *h : e->hs) {
            (void)hipStreamSynchronize(h->stream);
            saved.push_back(h->stream);
            h->stream = e->stream;
        }
    }
    ~EnsStreams()
    {
        (void)hipStreamSynchronize(e->stream);
        for (size_t i = 0; i < e->hs.size(); ++i) e->hs[i]->stream = saved[i];
    }
};

}  // namespace

int gempic_ensemble_create(int n_instances, gempic_splitting *const *handles, gempic_ensemble **out)
{
    if (!out) return fail(GEMPIC_ERR_ARGUMENT, "out is NULL");
    *out = nullptr;
    if (n_instances < 1 || !handles) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: need at least one splitting");
    gempic_splitting *h0 = handles[0];
    if (!h0) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
    for (int i = 0; i < n_instances; ++i) {
        gempic_splitting *h = handles[i];
        if (!h) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
        if (h->dim_v != 2) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: ensembles step 1d2v splittings");
        if (h->device != h0->device) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: every splitting must live on one GPU");
        if (h->deg0 != h0->deg0 || h->deg1 != h0->deg1)
            return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: every splitting must use the same smoother degrees");
        for (int j = 0; j < i; ++j)
            if (handles[j] == h) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: a splitting appears twice");
    }
    if (hipSetDevice(h0->device) != hipSuccess) return fail(GEMPIC_ERR_DEVICE, "hipSetDevice failed");
    gempic_ensemble *e = new gempic_ensemble();
    e->device = h0->device;
    e->hs.assign(handles, handles + n_instances);
    e->p0 = h0->deg0;
    e->p1 = h0->deg1;
    for (auto *h : e->hs) e->max_nx = std::max(e->max_nx, (int)h->nx);
    hipError_t r = hipStreamCreate(&e->stream);
    if (r == hipSuccess) r = dalloc(&e->d_args, 2 * (size_t)n_instances);
    if (r == hipSuccess) r = dalloc(&e->d_bstart, (size_t)n_instances + 1);
    if (r == hipSuccess) r = dalloc(&e->d_estart, (size_t)n_instances + 1);
    if (r == hipSuccess) r = dalloc(&e->d_sargs, (size_t)n_instances);
    if (r == hipSuccess) r = dalloc(&e->d_tstart, (size_t)n_instances + 1);
    if (r == hipSuccess) r = dalloc(&e->d_gstart, (size_t)n_instances + 1);
    if (r == hipSuccess) r = dalloc(&e->d_aargs, (size_t)n_instances);
    if (r == hipSuccess) r = dalloc(&e->d_abstart, (size_t)n_instances + 1);
    if (r == hipSuccess) r = dalloc(&e->d_aestart, (size_t)n_instances + 1);
    if (r != hipSuccess) {
        gempic_ensemble_destroy(e);
        return fail(GEMPIC_ERR_DEVICE, std::string("ensemble allocation: ") + hipGetErrorString(r));
    }
    *out = e;
    return GEMPIC_OK;
}

int gempic_ensemble_destroy(gempic_ensemble *e)
{
    if (!e) return GEMPIC_OK;
    (void)hipSetDevice(e->device);
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    void *bufs[] = {e->d_args, e->d_bstart, e->d_estart, e->d_sargs, e->d_tstart, e->d_gstart,
                    e->d_aargs, e->d_abstart, e->d_aestart};
    for (void *p : bufs)
        if (p) (void)hipFree(p);
    if (e->step_graph) (void)hipGraphExecDestroy(e->step_graph);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
    return GEMPIC_OK;
}

namespace {

// Workgroups of an ensemble's pass at most, twice those that are on the chip
// together: the second half evens out what the first ends at. us a step (24
// instances, 65,536 to 524,288 particles) at 4, 8, 16 a CU and one workgroup
// per block: 180, 172, 175, 183.
constexpr int kEnsPerCu = 8;
int ens_places(const gempic_ensemble *e)
{
    return e->hs[0]->cus * kEnsPerCu;
}

// the regular Strang step of an ensemble (another step follows, the previous
// one's HE pending) as a graph: captured on the ensemble's stream, then
// replayed; captured again when the launch geometry changed
int ens_step_graph(gempic_ensemble *e, const BatchArgs &b, int mode, size_t sh_pass, size_t sh_epi)
{
    const int ni = (int)e->hs.size();
    if (e->step_graph && e->graph_blocks == e->bstart[ni] && e->graph_groups == e->estart[ni] &&
        e->graph_mode == mode && e->graph_sh_pass == sh_pass && e->graph_sh_epi == sh_epi)
        return GEMPIC_OK;
    if (e->step_graph) {
        (void)hipGraphExecDestroy(e->step_graph);
        e->step_graph = nullptr;
    }
    hipGraph_t g = nullptr;
    HIP_TRY(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    const hipError_t e1 = launch_pass_batch(e->p0, e->p1, mode, b, sh_pass, e->stream);
    const hipError_t e2 = launch_epi_batch(e->p0, e->p1, mode, b, e->estart[ni], sh_epi, e->stream);
    const hipError_t e3 = hipStreamEndCapture(e->stream, &g);
    if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return fail(GEMPIC_ERR_DEVICE, "capturing the ensemble step as a HIP graph failed");
    }
    const hipError_t e4 = hipGraphInstantiate(&e->step_graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e4 != hipSuccess) {
        e->step_graph = nullptr;
        return fail(GEMPIC_ERR_DEVICE, "instantiating the ensemble step graph failed");
    }
    e->graph_blocks = e->bstart[ni];
    e->graph_groups = e->estart[ni];
    e->graph_mode = mode;
    e->graph_sh_pass = sh_pass;
    e->graph_sh_epi = sh_epi;
    return GEMPIC_OK;
}

}  // namespace

int gempic_ensemble_strang_splitting(gempic_ensemble *e, const double *dt, int64_t n_steps, int flags)
{
    if (!e) return fail(GEMPIC_ERR_ARGUMENT, "null ensemble");
    if (!dt) return fail(GEMPIC_ERR_ARGUMENT, "dt is NULL");
    if (hipSetDevice(e->device) != hipSuccess) return fail(GEMPIC_ERR_DEVICE, "hipSetDevice failed");
    if (n_steps < 0) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: number_steps must be >= 0");
    for (auto *h : e->hs)
        if (!h->particles_set) return fail(GEMPIC_ERR_STATE, "particles not set");
    if (n_steps == 0) return GEMPIC_OK;
    // the batch runs in the members' arithmetic, which they must share
    const int fast = fm(e->hs[0]);
    for (auto *h : e->hs)
        if (fm(h) != fast)
            return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: an ensemble's splittings must share one arithmetic");
    EnsStreams streams(e);
    const int ni = (int)e->hs.size();
    // HB(dt/2) and HE's B update of the first step, per instance
    for (int i = 0; i < ni; ++i) {
        const double hdt = 0.5 * dt[i];
        GridProg g = prog1(G_HB, hdt, S_B, S_B, S_E2);
        prog_add(g, G_HE_B, hdt, S_E2, S_E2, S_B);
        int rc = run_grid(e->hs[i], g);
        if (rc) return rc;
    }
    int rc = ens_upload(e, dt);
    if (rc) return rc;
    const size_t sh_pass = pass_shmem_bytes(e->max_nx, M_HE_PREV | M_HE | M_HP2A | M_HP1 | M_HP2B);
    const size_t sh_epi = epi_shmem_bytes(e->max_nx);
    for (int64_t s = 0; s < n_steps; ++s) {
        bool moved = false;
        rc = ens_sort(e, &moved);
        if (rc) return rc;
        if (moved) {
            rc = ens_upload(e, dt);
            if (rc) return rc;
        }
        const int mode = (s == 0 ? 0 : M_HE_PREV) | M_HE | M_HP2A | M_HP1 | M_HP2B | fast;
        BatchArgs b;
        b.args = e->d_args + (s + 1 < n_steps ? 0 : ni);
        b.block_start = e->d_bstart;
        b.epi_start = e->d_estart;
        b.ninst = ni;
        b.total = e->bstart[ni];
        b.places = ens_places(e);
        if ((flags & GEMPIC_GRAPH) && s > 0 && s + 1 < n_steps) {
            rc = ens_step_graph(e, b, mode, sh_pass, sh_epi);
            if (rc) return rc;
            HIP_TRY(hipGraphLaunch(e->step_graph, e->stream));
        } else {
            HIP_TRY(launch_pass_batch(e->p0, e->p1, mode, b, sh_pass, e->stream));
            HIP_TRY(launch_epi_batch(e->p0, e->p1, mode, b, e->estart[ni], sh_epi, e->stream));
        }
        for (auto *h : e->hs) h->steps_since_sort++;
    }
    // the last step's trailing HE
    BatchArgs b;
    b.args = e->d_args + ni;
    b.block_start = e->d_bstart;
    b.epi_start = e->d_estart;
    b.ninst = ni;
    b.total = e->bstart[ni];
    b.places = ens_places(e);
    HIP_TRY(launch_pass_batch(e->p0, e->p1, M_HE_PREV | fast, b,
                              pass_shmem_bytes(e->max_nx, M_HE_PREV), e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));
    for (auto *h : e->hs) {
        rc = finish(h);
        if (rc) return rc;
    }
    return GEMPIC_OK;
}


// Launch autotuning of an ensemble: for each candidate number of particles
// per workgroup, every instance's pass takes ceil(N / ppw) workgroups (at most
// its reduction scratch); n_steps batched steps are timed twice from the same
// state (restored after every trial, on the device) and the fastest
// candidate stays set on the member handles.
int gempic_ensemble_autotune(gempic_ensemble *e, const double *dt, int64_t n_steps, const int *ppw,
                             int n_candidates, int *best_ppw, double *ms_per_step)
{
    if (!e) return fail(GEMPIC_ERR_ARGUMENT, "null ensemble");
    if (!dt || !ppw) return fail(GEMPIC_ERR_ARGUMENT, "dt and the candidates must not be NULL");
    if (n_steps < 1 || n_steps > 100000)
        return fail(GEMPIC_ERR_ARGUMENT, "autotune: n_steps must be in [1, 100000]");
    if (n_candidates < 1 || n_candidates > 64)
        return fail(GEMPIC_ERR_ARGUMENT, "autotune: 1 to 64 candidates");
    for (int c = 0; c < n_candidates; ++c)
        if (ppw[c] < kBlock) return fail(GEMPIC_ERR_ARGUMENT, "autotune: a candidate is below 256 particles per workgroup");
    if (hipSetDevice(e->device) != hipSuccess) return fail(GEMPIC_ERR_DEVICE, "hipSetDevice failed");
    for (auto *h : e->hs)
        if (!h->particles_set) return fail(GEMPIC_ERR_STATE, "particles not set");
    const size_t ni = e->hs.size();
    // snapshot of every instance: particles in device order, ids, field slots, steps since sort
    std::vector<size_t> off(ni + 1, 0);
    for (size_t i = 0; i < ni; ++i) {
        const gempic_splitting *h = e->hs[i];
        off[i + 1] = off[i] + 5 * (size_t)h->n + (size_t)NSLOT * (size_t)h->nx;
    }
    double *snap = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (auto *h : e->hs) HIP_TRY(hipStreamSynchronize(h->stream));
    hipError_t err = dalloc(&snap, std::max<size_t>(off[ni], 1));
    if (err == hipSuccess) err = hipEventCreate(&ev[0]);
    if (err == hipSuccess) err = hipEventCreate(&ev[1]);
    std::vector<int64_t> since(ni);
    std::vector<int> saved_blocks(ni);
    for (size_t i = 0; i < ni; ++i) {
        since[i] = e->hs[i]->steps_since_sort;
        saved_blocks[i] = e->hs[i]->override_blocks;
    }
    auto copy_state = [&](bool save) -> hipError_t {
        hipError_t c = hipSuccess;
        for (size_t i = 0; i < ni && c == hipSuccess; ++i) {
            gempic_splitting *h = e->hs[i];
            const size_t n = (size_t)h->n;
            double *base = snap + off[i];
            double *dev[4] = {h->d_x, h->d_v1, h->d_v2, h->d_w};
            for (int k = 0; k < 4 && c == hipSuccess; ++k)
                c = hipMemcpyAsync(save ? base + k * n : dev[k], save ? dev[k] : base + k * n,
                                   sizeof(double) * n, hipMemcpyDeviceToDevice, e->stream);
            if (c == hipSuccess)
                c = hipMemcpyAsync(save ? (void *)(base + 4 * n) : (void *)h->d_id,
                                   save ? (const void *)h->d_id : (const void *)(base + 4 * n),
                                   sizeof(int64_t) * n, hipMemcpyDeviceToDevice, e->stream);
            if (c == hipSuccess)
                c = hipMemcpyAsync(save ? base + 5 * n : h->d_grid, save ? h->d_grid : base + 5 * n,
                                   sizeof(double) * (size_t)NSLOT * (size_t)h->nx,
                                   hipMemcpyDeviceToDevice, e->stream);
            h->steps_since_sort = since[i];
        }
        if (c == hipSuccess) c = hipStreamSynchronize(e->stream);
        return c;
    };
    bool saved = false;
    if (err == hipSuccess) {
        err = copy_state(true);
        saved = err == hipSuccess;
    }
    int rc = err == hipSuccess ? GEMPIC_OK
                               : fail(GEMPIC_ERR_DEVICE, std::string("ensemble autotune set-up: ") +
                                                             hipGetErrorString(err));
    double best = 0;
    int bi = -1;
    auto set_ppw = [&](int p) {
        for (auto *h : e->hs) {
            const int64_t b = (h->n + p - 1) / p;
            h->override_blocks = (int)std::max<int64_t>(1, std::min<int64_t>(b, h->max_blocks));
        }
    };
    for (int c = 0; c < n_candidates && !rc; ++c) {
        set_ppw(ppw[c]);
        float t = 0;
        for (int r = 0; r < 2 && !rc; ++r) {
            float ms = 0;
            err = hipEventRecord(ev[0], e->stream);
            if (err == hipSuccess) {
                rc = gempic_ensemble_strang_splitting(e, dt, n_steps, 0);
                if (!rc) err = hipEventRecord(ev[1], e->stream);
                if (!rc && err == hipSuccess) err = hipEventSynchronize(ev[1]);
                if (!rc && err == hipSuccess) err = hipEventElapsedTime(&ms, ev[0], ev[1]);
                if (!rc && err == hipSuccess) err = copy_state(false);
            }
            if (!rc && err != hipSuccess)
                rc = fail(GEMPIC_ERR_DEVICE, std::string("ensemble autotune: ") + hipGetErrorString(err));
            if (r == 0 || ms < t) t = ms;
        }
        if (rc) break;
        const double per = (double)t / (double)n_steps;
        if (ms_per_step) ms_per_step[c] = per;
        if (bi < 0 || per < best) {
            best = per;
            bi = c;
        }
    }
    if (rc) {
        const std::string msg = gempic_last_error();
        if (saved) (void)copy_state(false);
        for (size_t i = 0; i < ni; ++i) e->hs[i]->override_blocks = saved_blocks[i];
        g_last_error = msg;
    } else {
        set_ppw(ppw[bi]);
        if (best_ppw) *best_ppw = ppw[bi];
    }
    if (ev[0]) (void)hipEventDestroy(ev[0]);
    if (ev[1]) (void)hipEventDestroy(ev[1]);
    if (snap) (void)hipFree(snap);
    return rc;
}

// Reverse mode of an ensemble: gempic_strang_splitting_adjoint for every
// instance, with the recorded forward, the re-runs, the reverse passes and
// their field parts batched over the instances (one launch each per step;
// the field parts as two). Each instance's loss and cotangents equal those
// of its own gempic_strang_splitting_adjoint bit for bit (gempic_get_adjoint
// reads them per splitting). No cotangents of the final state: the loss is
// loss_weight[i] * sum_s 1/2 l2norm_squared(B_s).
int gempic_ensemble_strang_splitting_adjoint(gempic_ensemble *e, const double *dt, int64_t n_steps,
                                             int64_t checkpoint_every, const double *loss_weight,
                                             int flags)
{
    if (!e) return fail(GEMPIC_ERR_ARGUMENT, "null ensemble");
    if (!dt || !loss_weight) return fail(GEMPIC_ERR_ARGUMENT, "dt and loss_weight must not be NULL");
    if (hipSetDevice(e->device) != hipSuccess) return fail(GEMPIC_ERR_DEVICE, "hipSetDevice failed");
    if (n_steps < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: number_steps must be >= 1");
    if (checkpoint_every < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: checkpoint_every must be >= 1");
    for (auto *h : e->hs) {
        if (!h->particles_set) return fail(GEMPIC_ERR_STATE, "particles not set");
        if (h->nx > kAdjNxMax || h->nx < 4)
            return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: the reverse mode needs 4 <= nx <= 128");
    }
    EnsStreams streams(e);
    struct RecordOff {
        gempic_ensemble *e;
        ~RecordOff()
        {
            for (auto *h : e->hs) { h->cur_hist = nullptr; h->cur_cx = nullptr; h->cur_perm = nullptr; }
        }
    } record_off{e};
    const int ni = (int)e->hs.size();
    const int64_t T = n_steps, K = std::min<int64_t>(checkpoint_every, n_steps);
    const int64_t nck = (T + K - 1) / K;
    int rc = GEMPIC_OK;
    for (auto *h : e->hs) {
        rc = adj_workspace(h, T, K);
        if (!rc) rc = ensure_stage(h);
        if (rc) return rc;
        h->adj_ready = false;
    }
    auto rec = [](gempic_splitting *h, int64_t s) { return h->d_hist + (size_t)s * NHIST * h->nx; };
    struct Inst {
        std::vector<int64_t> epoch_of;
        int64_t ne = 0;
        double *lam = nullptr;
        Launch L{};
    };
    std::vector<Inst> st((size_t)ni);

    // ---- forward, recorded ----
    for (int i = 0; i < ni; ++i) {
        gempic_splitting *h = e->hs[i];
        const size_t nx = (size_t)h->nx;
        const double hdt = 0.5 * dt[i];
        HIP_TRY(hipMemcpyAsync(rec(h, 0) + H_BEND * nx, h->d_grid + S_B * nx, sizeof(double) * nx,
                               hipMemcpyDeviceToDevice, e->stream));
        GridProg g = prog1(G_HB, hdt, S_B, S_B, S_E2);
        prog_add(g, G_HE_B, hdt, S_E2, S_E2, S_B);
        rc = run_grid(h, g);
        if (rc) return rc;
        HIP_TRY(hipMemcpyAsync(rec(h, 1), h->d_grid, sizeof(double) * 4 * nx, hipMemcpyDeviceToDevice,
                               e->stream));
        st[i].epoch_of.assign((size_t)nck, 0);
    }
    rc = ens_upload(e, dt);          // workgroup tables (the arguments are rebuilt every step)
    if (rc) return rc;
    const size_t sh_pass = pass_shmem_bytes(e->max_nx, M_HE_PREV | M_HE | M_HP2A | M_HP1 | M_HP2B);
    const size_t sh_epi = epi_shmem_bytes(e->max_nx);
    std::vector<PassArgs> pa((size_t)ni);
    auto pass_step = [&](int64_t s, bool trailing) -> int {
        for (int i = 0; i < ni; ++i) {
            gempic_splitting *h = e->hs[i];
            const int target = h->override_blocks ? h->override_blocks : h->dep_blocks;
            const Launch L = plan(h->n, target);
            h->cur_hist = trailing ? nullptr : rec(h, s);
            h->cur_cx = (!trailing && s % K == 0 && s < T) ? h->d_ckpt + (size_t)(s / K) * 3 * h->n
                                                            : nullptr;
            PassArgs a = pass_args(h);
            const double hdt = 0.5 * dt[i];
            a.chunk = L.chunk;
            a.iters = L.iters;
            a.ngroups = L.ngroups;
            set_generations(a, L, h->cus);
            a.dt_he = hdt;
            a.dt_hp2 = hdt;
            a.dt_hp1 = 1.0 * dt[i];
            a.dtqm_he = hdt * h->qm;
            a.dtqm_hp2 = hdt * h->qm;
            a.more = (!trailing && s < T) ? 1 : 0;
            pa[(size_t)i] = a;
            h->cur_hist = nullptr;
            h->cur_cx = nullptr;
        }
        HIP_TRY(hipMemcpy(e->d_args, pa.data(), sizeof(PassArgs) * (size_t)ni, hipMemcpyHostToDevice));
        BatchArgs b;
        b.args = e->d_args;
        b.block_start = e->d_bstart;
        b.epi_start = e->d_estart;
        b.ninst = ni;
        b.total = e->bstart[ni];
        b.places = ens_places(e);
        if (trailing) {
            HIP_TRY(launch_pass_batch(e->p0, e->p1, M_HE_PREV, b,
                                      pass_shmem_bytes(e->max_nx, M_HE_PREV), e->stream));
            return GEMPIC_OK;
        }
        const int mode = (s > 1 ? M_HE_PREV : 0) | M_HE | M_HP2A | M_HP1 | M_HP2B;
        HIP_TRY(launch_pass_batch(e->p0, e->p1, mode, b, sh_pass, e->stream));
        HIP_TRY(launch_epi_batch(e->p0, e->p1, mode, b, e->estart[ni], sh_epi, e->stream));
        return GEMPIC_OK;
    };
    for (int64_t s = 1; s <= T; ++s) {
        if ((s - 1) % K == 0) {
            const size_t j = (size_t)((s - 1) / K);
            std::vector<char> sorted((size_t)ni, 0);
            if (s > 1) {
                for (int i = 0; i < ni; ++i) {
                    rc = adj_epoch_check(e->hs[i], st[i].ne);
                    if (rc) return rc;
                }
                for (int i = 0; i < ni; ++i)
                    e->hs[i]->cur_perm = e->hs[i]->d_perm + (size_t)st[i].ne * e->hs[i]->n;
                bool any = false;
                rc = ens_sort(e, &any);
                for (auto *h : e->hs) h->cur_perm = nullptr;
                if (rc) return rc;
                for (int i = 0; i < ni; ++i) sorted[i] = e->hs[i]->steps_since_sort == 0;
                if (any) {
                    rc = ens_upload(e, dt);
                    if (rc) return rc;
                }
            }
            for (int i = 0; i < ni; ++i) {
                gempic_splitting *h = e->hs[i];
                const size_t n = (size_t)h->n, nb = sizeof(double) * n;
                if (s == 1)
                    HIP_TRY(hipMemcpyAsync(h->d_ids, h->d_id, sizeof(int64_t) * n, hipMemcpyDeviceToDevice,
                                           e->stream));
                if (s == 1 || sorted[i]) {
                    HIP_TRY(hipMemcpyAsync(h->d_wsnap + (size_t)st[i].ne * n, h->d_w, nb,
                                           hipMemcpyDeviceToDevice, e->stream));
                    ++st[i].ne;
                }
                st[i].epoch_of[j] = st[i].ne - 1;
                if (s == 1 || sorted[i]) {
                    double *ck = h->d_ckpt + j * 3 * n;
                    HIP_TRY(hipMemcpyAsync(ck, h->d_x, nb, hipMemcpyDeviceToDevice, e->stream));
                    HIP_TRY(hipMemcpyAsync(ck + n, h->d_v1, nb, hipMemcpyDeviceToDevice, e->stream));
                    HIP_TRY(hipMemcpyAsync(ck + 2 * n, h->d_v2, nb, hipMemcpyDeviceToDevice, e->stream));
                }
            }
        }
        rc = pass_step(s, false);
        if (rc) return rc;
        for (auto *h : e->hs) h->steps_since_sort++;
    }
    rc = pass_step(T, true);
    if (rc) return rc;

    // ---- reverse ----
    std::vector<int> abstart((size_t)ni + 1, 0), aestart((size_t)ni + 1, 0);
    for (int i = 0; i < ni; ++i) {
        gempic_splitting *h = e->hs[i];
        st[i].L = plan(h->n, h->adj_blocks);
        st[i].lam = h->d_lam;
        abstart[i + 1] = abstart[i] + st[i].L.blocks;
        aestart[i + 1] = aestart[i] + epi_groups(st[i].L.blocks);
        HIP_TRY(hipMemsetAsync(h->d_agrid, 0, sizeof(double) * NASLOT * h->nx, e->stream));
        HIP_TRY(hipMemsetAsync(h->d_lam, 0, sizeof(double) * 3 * h->n, e->stream));
    }
    HIP_TRY(hipMemcpy(e->d_abstart, abstart.data(), sizeof(int) * (ni + 1), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(e->d_aestart, aestart.data(), sizeof(int) * (ni + 1), hipMemcpyHostToDevice));
    AdjBatch ab;
    ab.args = e->d_aargs;
    ab.block_start = e->d_abstart;
    ab.epi_start = e->d_aestart;
    ab.ninst = ni;
    ab.max_nx = e->max_nx;
    std::vector<AdjArgs> aa((size_t)ni);
    // fill one AdjArgs per instance, upload, launch the pass and (kind >= 0) its field part
    auto rev_launch = [&](int rm, int kind, const std::function<void(int, AdjArgs &)> &set) -> int {
        for (int i = 0; i < ni; ++i) {
            gempic_splitting *h = e->hs[i];
            AdjArgs A = adj_args(h, dt[i], st[i].L);
            A.wloss = loss_weight[i];
            A.lx = st[i].lam;
            A.lv1 = st[i].lam + h->n;
            A.lv2 = st[i].lam + 2 * h->n;
            set(i, A);
            aa[(size_t)i] = A;
        }
        HIP_TRY(hipMemcpy(e->d_aargs, aa.data(), sizeof(AdjArgs) * (size_t)ni, hipMemcpyHostToDevice));
        HIP_TRY(launch_adj_batch(e->p0, e->p1, rm, ab, abstart[ni], e->stream));
        if (kind >= 0) HIP_TRY(launch_adj_epi_batch(kind, ab, aestart[ni], e->stream));
        return GEMPIC_OK;
    };
    rc = rev_launch(R_HEONLY, AE_TAIL, [&](int i, AdjArgs &A) {
        gempic_splitting *h = e->hs[i];
        A.x = h->d_x;
        A.fields = rec(h, T + 1);
        A.bend = rec(h, T) + H_BEND * h->nx;
    });
    for (int64_t j = nck - 1; j >= 0 && !rc; --j) {
        const int64_t s_lo = j * K + 1, s_hi = std::min((j + 1) * K, T);
        auto state = [&](gempic_splitting *h, int64_t s) {
            const size_t n = (size_t)h->n;
            return s == s_lo ? h->d_ckpt + (size_t)j * 3 * n : h->d_seg + (size_t)(s - s_lo - 1) * 3 * n;
        };
        auto common = [&](int i, AdjArgs &A, int64_t s) {
            gempic_splitting *h = e->hs[i];
            const size_t n = (size_t)h->n;
            double *b0 = state(h, s);
            A.x = b0;
            A.v1 = b0 + n;
            A.v2 = b0 + 2 * n;
            A.fields = rec(h, s);
            A.p.w = h->d_wsnap + (size_t)st[i].epoch_of[(size_t)j] * n;
        };
        for (int64_t s = s_lo; s < s_hi && !rc; ++s)
            rc = rev_launch(R_FWD | (s > 1 ? R_PREV : 0), -1, [&](int i, AdjArgs &A) {
                common(i, A, s);
                gempic_splitting *h = e->hs[i];
                double *b1 = state(h, s + 1);
                A.xo = b1;
                A.v1o = b1 + h->n;
                A.v2o = b1 + 2 * h->n;
            });
        for (int64_t s = s_hi; s >= s_lo && !rc; --s)
            rc = rev_launch(R_REV | (s > 1 ? R_PREV : 0), s > 1 ? AE_STEP : AE_HEAD,
                            [&](int i, AdjArgs &A) {
                                common(i, A, s);
                                gempic_splitting *h = e->hs[i];
                                A.bend = rec(h, s > 1 ? s - 1 : 0) + H_BEND * h->nx;
                            });
        if (!rc && j > 0)
            for (int i = 0; i < ni; ++i) {
                if (st[i].epoch_of[(size_t)j] == st[i].epoch_of[(size_t)j - 1]) continue;
                gempic_splitting *h = e->hs[i];
                double *other = st[i].lam == h->d_lam ? h->d_stage : h->d_lam;
                HIP_TRY(launch_adj_unsort(h->d_perm + (size_t)st[i].epoch_of[(size_t)j] * h->n, h->n,
                                          st[i].lam, other, e->stream));
                st[i].lam = other;
            }
    }
    if (rc) return rc;
    for (int i = 0; i < ni; ++i) {
        gempic_splitting *h = e->hs[i];
        if (st[i].lam != h->d_lam)
            HIP_TRY(hipMemcpyAsync(h->d_lam, st[i].lam, sizeof(double) * 3 * h->n, hipMemcpyDeviceToDevice,
                                   e->stream));
        h->adj_id0 = h->d_ids;
        h->adj_ready = true;
    }
    (void)flags;
    HIP_TRY(hipStreamSynchronize(e->stream));
    for (auto *h : e->hs) {
        rc = finish(h);
        if (rc) return rc;
    }
    return GEMPIC_OK;
}

int gempic_synchronize(gempic_splitting *h)
{
    CHECK_H(h);
    return finish(h);
}

int gempic_set_sort_interval(gempic_splitting *h, int64_t interval)
{
    CHECK_H(h);
    if (interval < 0) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: interval must be >= 0");
    h->sort_interval = interval;
    return GEMPIC_OK;
}

int gempic_sort_particles(gempic_splitting *h)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = run_sort(h);
    if (rc) return rc;
    return finish(h);
}

int gempic_solve_poisson(gempic_splitting *h, double *efield, double *rho)
{
    CHECK_H(h);
    CHECK_P(h);
    int rc = run_pass(h, M_RHO, 0, 0, 0, 0, 7);
    if (rc) return rc;
    const size_t nb = sizeof(double) * h->nx;
    if (efield) HIP_TRY(hipMemcpyAsync(efield, h->d_grid + S_EPOIS * h->nx, nb, hipMemcpyDeviceToHost, h->stream));
    if (rho) HIP_TRY(hipMemcpyAsync(rho, h->d_grid + S_RHO * h->nx, nb, hipMemcpyDeviceToHost, h->stream));
    return finish(h);
}

int gempic_write_step(gempic_splitting *h, double time, int degree, const double *e1_n,
                      const double *e2_n, const double *efield_poisson, double *out11)
{
    CHECK_H(h);
    CHECK_P(h);
    if (!out11) return fail(GEMPIC_ERR_ARGUMENT, "out is NULL");
    if (h->dim_v != 2) return fail(GEMPIC_ERR_ARGUMENT, "write_step! reads v1, v2: 1d2v only");
    if (degree != h->mdeg) return fail(GEMPIC_ERR_ARGUMENT, "degree must be the Maxwell solver's s_deg_0");
    const size_t nb = sizeof(double) * h->nx;
    const int64_t nx = h->nx;
    if (e1_n) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E1N * nx, e1_n, nb, hipMemcpyHostToDevice, h->stream));
    else HIP_TRY(hipMemcpyAsync(h->d_grid + S_E1N * nx, h->d_grid + S_E1 * nx, nb, hipMemcpyDeviceToDevice, h->stream));
    if (e2_n) HIP_TRY(hipMemcpyAsync(h->d_grid + S_E2N * nx, e2_n, nb, hipMemcpyHostToDevice, h->stream));
    else HIP_TRY(hipMemcpyAsync(h->d_grid + S_E2N * nx, h->d_grid + S_E2 * nx, nb, hipMemcpyDeviceToDevice, h->stream));
    int rc;
    if (efield_poisson) {
        HIP_TRY(hipMemcpyAsync(h->d_grid + S_EPOIS * nx, efield_poisson, nb, hipMemcpyHostToDevice, h->stream));
    } else {
        rc = run_pass(h, M_RHO, 0, 0, 0, 0, 7);
        if (rc) return rc;
    }
    rc = run_pass(h, M_DIAG, 0, 0, 0, 0, 7);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(out11, h->d_diag, sizeof(double) * 11, hipMemcpyDeviceToHost, h->stream));
    rc = finish(h);
    out11[0] = time;
    return rc;
}

int gempic_profile_enable(gempic_splitting *h, int enable)
{
    CHECK_H(h);
    if (enable < 0) return fail(GEMPIC_ERR_ARGUMENT, "enable must be >= 0");
    if (!enable) resolve_profile(h);
    h->profile = enable != 0;
    h->profile_every = enable > 1 ? enable : 1;
    for (int k = 0; k < gempic_splitting::kProfIds; ++k) h->prof_seen[k] = 0;
    return GEMPIC_OK;
}

int gempic_profile_read(gempic_splitting *h, int kernel_id, double *total_ms, int64_t *count)
{
    CHECK_H(h);
    if (kernel_id < 0 || kernel_id >= gempic_splitting::kProfIds)
        return fail(GEMPIC_ERR_ARGUMENT, "kernel id in 0..12");
    resolve_profile(h);
    if (total_ms) *total_ms = h->prof_ms[kernel_id];
    if (count) *count = h->prof_cnt[kernel_id];
    return GEMPIC_OK;
}

int gempic_profile_reset(gempic_splitting *h)
{
    CHECK_H(h);
    resolve_profile(h);
    for (int k = 0; k < gempic_splitting::kProfIds; ++k) { h->prof_ms[k] = 0; h->prof_cnt[k] = 0; }
    return GEMPIC_OK;
}

int gempic_set_fusion(gempic_splitting *h, int kernels_per_step)
{
    CHECK_H(h);
    if (kernels_per_step != 1 && kernels_per_step != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "kernels_per_step must be 1 or 2");
    if (kernels_per_step == 2 && h->arith != GEMPIC_ARITH_REFERENCE)
        return fail(GEMPIC_ERR_ARGUMENT, "the two-kernel step runs in the reference's arithmetic only");
    h->kernels_per_step = kernels_per_step;
    return GEMPIC_OK;
}

int gempic_set_arithmetic(gempic_splitting *h, int arith)
{
    CHECK_H(h);
    if (arith != GEMPIC_ARITH_REFERENCE && arith != GEMPIC_ARITH_FUSED)
        return fail(GEMPIC_ERR_ARGUMENT, "arithmetic must be GEMPIC_ARITH_REFERENCE or GEMPIC_ARITH_FUSED");
    if (arith == GEMPIC_ARITH_FUSED && h->dim_v != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "fused arithmetic covers the 1d2v passes");
    if (arith == GEMPIC_ARITH_FUSED && h->kernels_per_step != 1)
        return fail(GEMPIC_ERR_ARGUMENT, "fused arithmetic needs the one-kernel fused step");
    h->arith = arith;
    return GEMPIC_OK;
}

int gempic_set_launch(gempic_splitting *h, int blocks)
{
    CHECK_H(h);
    if (blocks < 0) return fail(GEMPIC_ERR_ARGUMENT, "blocks must be >= 0");
    if (blocks > h->max_blocks)
        return fail(GEMPIC_ERR_ARGUMENT, "blocks exceeds the reduction scratch (8 per CU)");
    h->override_blocks = blocks;
    return GEMPIC_OK;
}

int gempic_autotune(gempic_splitting *h, double dt, int64_t n_steps, const int *blocks,
                    int n_blocks, const int64_t *sort_intervals, int n_intervals, int *best_blocks,
                    int64_t *best_interval, double *ms_per_step)
{
    CHECK_H(h);
    CHECK_P(h);
    if (n_steps < 1 || n_steps > 100000)
        return fail(GEMPIC_ERR_ARGUMENT, "autotune: n_steps must be in [1, 100000]");
    if (!blocks || n_blocks < 1 || n_blocks > 64 || !sort_intervals || n_intervals < 1 ||
        n_intervals > 64)
        return fail(GEMPIC_ERR_ARGUMENT, "autotune: 1 to 64 candidates of each kind");
    for (int i = 0; i < n_blocks; ++i)
        if (blocks[i] < 0 || blocks[i] > h->max_blocks)
            return fail(GEMPIC_ERR_ARGUMENT,
                        "autotune: a blocks candidate is negative or exceeds the reduction scratch "
                        "(8 per CU)");
    for (int j = 0; j < n_intervals; ++j)
        if (sort_intervals[j] < 0)
            return fail(GEMPIC_ERR_ARGUMENT, "autotune: a sort interval candidate is negative");

    // snapshot of everything a Strang call changes: particles in their device
    // order, the field slots and the steps since the last sort
    const size_t n = (size_t)h->n, ng = (size_t)NSLOT * (size_t)h->nx;
    const int nv = h->dim_v == 2 ? 2 : 1;
    double *snap = nullptr;
    int64_t *snap_id = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    HIP_TRY(hipStreamSynchronize(h->stream));
    hipError_t e = dalloc(&snap, (2 + (size_t)nv) * n + ng);
    if (e == hipSuccess) e = dalloc(&snap_id, n);
    if (e == hipSuccess) e = hipEventCreate(&ev[0]);
    if (e == hipSuccess) e = hipEventCreate(&ev[1]);
    const int64_t saved_since = h->steps_since_sort;
    const int saved_blocks = h->override_blocks;
    const int64_t saved_interval = h->sort_interval;
    const bool saved_profile = h->profile;
    auto copy_state = [&](bool save) -> hipError_t {
        double *dev[4] = {h->d_x, h->d_v1, h->d_w, h->d_v2};
        hipError_t c = hipSuccess;
        for (int k = 0; k < 2 + nv && c == hipSuccess; ++k) {
            double *s = snap + (size_t)k * n;
            c = hipMemcpyAsync(save ? s : dev[k], save ? dev[k] : s, sizeof(double) * n,
                               hipMemcpyDeviceToDevice, h->stream);
        }
        double *sg = snap + (2 + (size_t)nv) * n;
        if (c == hipSuccess)
            c = hipMemcpyAsync(save ? sg : h->d_grid, save ? h->d_grid : sg, sizeof(double) * ng,
                               hipMemcpyDeviceToDevice, h->stream);
        if (c == hipSuccess)
            c = hipMemcpyAsync(save ? snap_id : h->d_id, save ? h->d_id : snap_id,
                               sizeof(int64_t) * n, hipMemcpyDeviceToDevice, h->stream);
        if (c == hipSuccess) c = hipStreamSynchronize(h->stream);
        h->steps_since_sort = saved_since;
        return c;
    };
    bool saved = false;
    if (e == hipSuccess) {
        e = copy_state(true);
        saved = e == hipSuccess;
    }

    int rc = e == hipSuccess ? GEMPIC_OK
                             : fail(GEMPIC_ERR_DEVICE, std::string("autotune set-up: ") +
                                                           hipGetErrorString(e));
    h->profile = false;
    double best = 0;
    int bi = -1;
    for (int i = 0; i < n_blocks && !rc; ++i) {
        for (int j = 0; j < n_intervals && !rc; ++j) {
            h->override_blocks = blocks[i];
            h->sort_interval = sort_intervals[j];
            // two timed trials from the same state; the faster one counts
            float t = 0;
            for (int r = 0; r < 2 && !rc; ++r) {
                float ms = 0;
                e = hipEventRecord(ev[0], h->stream);
                if (e != hipSuccess) {
                    rc = fail(GEMPIC_ERR_DEVICE, std::string("autotune: ") + hipGetErrorString(e));
                    break;
                }
                // queued without a host round trip, so the events time the GPU
                // work only; the deferred error check follows the timing
                rc = gempic_strang_splitting(h, dt, n_steps, GEMPIC_ASYNC);
                if (!rc) e = hipEventRecord(ev[1], h->stream);
                if (!rc && e == hipSuccess) e = hipEventSynchronize(ev[1]);
                if (!rc && e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
                if (!rc && e == hipSuccess) rc = finish(h);
                if (!rc && e == hipSuccess) e = copy_state(false);
                if (!rc && e != hipSuccess)
                    rc = fail(GEMPIC_ERR_DEVICE, std::string("autotune: ") + hipGetErrorString(e));
                if (r == 0 || ms < t) t = ms;
            }
            if (rc) break;
            const double per = (double)t / (double)n_steps;
            if (ms_per_step) ms_per_step[(size_t)i * n_intervals + j] = per;
            if (bi < 0 || per < best) {
                best = per;
                bi = i * n_intervals + j;
            }
        }
    }
    h->profile = saved_profile;
    if (rc) {
        // a failed trial leaves the caller's state and settings as they were
        const std::string msg = gempic_last_error();
        if (saved) (void)copy_state(false);
        h->override_blocks = saved_blocks;
        h->sort_interval = saved_interval;
        g_last_error = msg;
    } else {
        h->override_blocks = blocks[bi / n_intervals];
        h->sort_interval = sort_intervals[bi % n_intervals];
        if (best_blocks) *best_blocks = h->override_blocks;
        if (best_interval) *best_interval = h->sort_interval;
    }
    if (ev[0]) (void)hipEventDestroy(ev[0]);
    if (ev[1]) (void)hipEventDestroy(ev[1]);
    if (snap) (void)hipFree(snap);
    if (snap_id) (void)hipFree(snap_id);
    return rc;
}

// ---------------------------------------------------------------------------
// batched ParticleMeshCoupling1D verbs
// ---------------------------------------------------------------------------
static hipStream_t pmc_stream()
{
    static thread_local hipStream_t s = nullptr;
    if (!s) (void)hipStreamCreate(&s);
    return s;
}

static int pmc_run(int op, int64_t nx, double xmin, double xmax, int degree, int smoothing,
                   int64_t n, const double *x, const double *x_new, const double *q, double qm,
                   const double *field, int64_t field_len, double *out, double *acc, bool out_in)
{
    if (nx < 1 || nx > kNxMax) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: nx must be in [1, 256]");
    if (degree < 0 || degree > 5) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree must be in 0..5");
    if (smoothing != GEMPIC_GALERKIN && smoothing != GEMPIC_COLLOCATION)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: smoothing type not implemented");
    if (n < 0) return fail(GEMPIC_ERR_ARGUMENT, "n must be >= 0");
    if (!(xmax > xmin)) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: xmax must exceed xmin");
    int rc = check_device();
    if (rc) return rc;
    if (n == 0) return GEMPIC_OK;
    hipStream_t s = pmc_stream();
    PmcArgs a;
    std::memset(&a, 0, sizeof(a));
    a.n = n;
    a.nx = (int)nx;
    a.degree = degree;
    a.xmin = xmin;
    a.dx = (xmax - xmin) / (double)nx;
    a.scaling = smoothing == GEMPIC_COLLOCATION ? 1.0 / a.dx : 1.0;
    gh::gauss_legendre((degree + 2) / 2, a.qx, a.qw);
    if (degree >= 1) gh::splinepp_tables(degree, a.pc, a.pf);
    a.qm = qm;
    const int max_blocks = device_cus() * 4;
    Launch L = plan(n, max_blocks);   // k_pmc: at least 4 workgroups fit per CU
    a.chunk = L.chunk;
    a.iters = L.iters;
    a.ngroups = L.ngroups;
    std::vector<void *> bufs;
    hipError_t e = hipSuccess;
    auto upload = [&](const double *src, size_t cnt) -> double * {
        if (!src) return nullptr;
        double *d = nullptr;
        if (e == hipSuccess) e = dalloc(&d, cnt);
        if (e == hipSuccess) { bufs.push_back(d); e = hipMemcpyAsync(d, src, sizeof(double) * cnt, hipMemcpyHostToDevice, s); }
        return d;
    };
    a.x = upload(x, n);
    a.x_new = upload(x_new, n);
    a.q = upload(q, n);
    a.field = upload(field, (size_t)field_len);
    double *d_out = nullptr, *d_acc = nullptr;
    if (out) {
        if (out_in) d_out = upload(out, n);
        else { if (e == hipSuccess) e = dalloc(&d_out, n); if (e == hipSuccess) bufs.push_back(d_out); }
    }
    if (acc) d_acc = upload(acc, nx);
    a.out = d_out;
    a.acc = d_acc;
    if (e == hipSuccess) e = dalloc(&a.part, (size_t)L.blocks * nx + 8);
    if (e == hipSuccess) bufs.push_back(a.part);
    if (e == hipSuccess) e = dalloc(&a.gpart, (size_t)L.ngroups * nx + 8);
    if (e == hipSuccess) bufs.push_back(a.gpart);
    if (e == hipSuccess) e = dalloc(&a.cnt, (size_t)L.ngroups + 2);
    if (e == hipSuccess) { bufs.push_back(a.cnt); e = hipMemsetAsync(a.cnt, 0, sizeof(unsigned) * (L.ngroups + 2), s); }
    if (e == hipSuccess) e = dalloc(&a.err, 1);
    if (e == hipSuccess) { bufs.push_back(a.err); e = hipMemsetAsync(a.err, 0, sizeof(int), s); }
    if (e == hipSuccess) e = launch_pmc(op, a, L.blocks, s);
    if (e == hipSuccess && out) e = hipMemcpyAsync(out, d_out, sizeof(double) * n, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && acc) e = hipMemcpyAsync(acc, d_acc, sizeof(double) * nx, hipMemcpyDeviceToHost, s);
    int err = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&err, a.err, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipStreamSynchronize(s);
    for (void *p : bufs) (void)hipFree(p);
    if (e != hipSuccess) return fail(GEMPIC_ERR_DEVICE, std::string("particle-mesh coupling: ") + hipGetErrorString(e));
    if (err & E_INEXACT) return fail(GEMPIC_ERR_INEXACT, "InexactError: trunc(Int64, x): non-finite particle position");
    if (err & E_FAR) return fail(GEMPIC_ERR_INEXACT, "a particle crossed more than 65536 cells in one push");
    if (err & E_BOUNDS) return fail(GEMPIC_ERR_ARGUMENT, "BoundsError: position outside the pp matrix");
    return GEMPIC_OK;
}

int gempic_pmc1d_add_charge(int64_t nx, double xmin, double xmax, int degree, int smoothing,
                            int64_t n, const double *x, const double *q, double *rho)
{
    if ((n > 0 && (!x || !q)) || !rho) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    return pmc_run(PMC_CHARGE, nx, xmin, xmax, degree, smoothing, n, x, nullptr, q, 0.0, nullptr,
                   0, nullptr, rho, false);
}

int gempic_pmc1d_add_charge_pp(int64_t nx, double xmin, double xmax, int degree, int smoothing,
                               int64_t n, const double *x, const double *q, double *rho)
{
    if ((n > 0 && (!x || !q)) || !rho) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (degree < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree must be in 1..5 for SplinePP");
    return pmc_run(PMC_CHARGE_PP, nx, xmin, xmax, degree, smoothing, n, x, nullptr, q, 0.0,
                   nullptr, 0, nullptr, rho, false);
}

int gempic_pmc1d_evaluate(int64_t nx, double xmin, double xmax, int degree, int smoothing,
                          int64_t n, const double *x, const double *field, double *out)
{
    if ((n > 0 && (!x || !out)) || !field) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    return pmc_run(PMC_EVAL, nx, xmin, xmax, degree, smoothing, n, x, nullptr, nullptr, 0.0,
                   field, nx, out, nullptr, false);
}

int gempic_pmc1d_evaluate_pp(int64_t nx, double xmin, double xmax, int degree, int smoothing,
                             int64_t n, const double *x, const double *field_pp, double *out)
{
    if ((n > 0 && (!x || !out)) || !field_pp) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (degree < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree must be in 1..5 for SplinePP");
    return pmc_run(PMC_EVAL_PP, nx, xmin, xmax, degree, smoothing, n, x, nullptr, nullptr, 0.0,
                   field_pp, (degree + 1) * nx, out, nullptr, false);
}

int gempic_pmc1d_add_current_update_v(int64_t nx, double xmin, double xmax, int degree,
                                      int smoothing, int64_t n, const double *x_old,
                                      const double *x_new, const double *q, double qm,
                                      const double *bfield, double *v, double *j)
{
    if ((n > 0 && (!x_old || !x_new || !q || !v)) || !j) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (bfield)
        return pmc_run(PMC_CURRENT_B, nx, xmin, xmax, degree, smoothing, n, x_old, x_new, q, qm,
                       bfield, nx, v, j, true);
    return pmc_run(PMC_CURRENT_NOB, nx, xmin, xmax, degree, smoothing, n, x_old, x_new, q, qm,
                   nullptr, 0, nullptr, j, false);
}

int gempic_pmc1d_add_current_update_v_pp(int64_t nx, double xmin, double xmax, int degree,
                                         int smoothing, int64_t n, const double *x_old,
                                         const double *x_new, const double *q, double qm,
                                         const double *bfield, double *v, double *j)
{
    if ((n > 0 && (!x_old || !x_new || !q || !v || !bfield)) || !j)
        return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (degree < 1) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree must be in 1..5 for SplinePP");
    return pmc_run(PMC_CURRENT_PP, nx, xmin, xmax, degree, smoothing, n, x_old, x_new, q, qm,
                   bfield, nx, v, j, true);
}

// b_to_pp (splinepp.jl:241-261): a set-up conversion of nx coefficients,
// done on the host.
int gempic_b_to_pp(int degree, int64_t ncells, const double *b, double *pp)
{
    if (!b || !pp) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (degree < 1 || degree > 5) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree not implemented");
    if (ncells < degree) return fail(GEMPIC_ERR_ASSERTION, "AssertionError: ncells >= degree");
    double pc[36], pf[36];
    gh::splinepp_tables(degree, pc, pf);
    const int dp1 = degree + 1;
    double coeffs[6];
    for (int64_t i = 1; i <= ncells; ++i) {
        if (i <= degree) {
            int c = 0;
            for (int64_t k = ncells - degree + i; k <= ncells; ++k) coeffs[c++] = b[k - 1];
            for (int64_t k = 1; k <= i; ++k) coeffs[c++] = b[k - 1];
        } else {
            for (int k = 0; k < dp1; ++k) coeffs[k] = b[i - degree - 1 + k];
        }
        for (int j = 0; j < dp1; ++j) {
            double s = coeffs[0] * pc[j];
            for (int k = 1; k < dp1; ++k) s = s + coeffs[k] * pc[j + k * dp1];
            pp[j + (i - 1) * dp1] = s;
        }
    }
    return GEMPIC_OK;
}

// ---------------------------------------------------------------------------
// Maxwell1DFEM verbs
// ---------------------------------------------------------------------------
int gempic_maxwell1d_create(int64_t nx, double xmin, double xmax, int degree, gempic_maxwell1d **out)
{
    if (!out) return fail(GEMPIC_ERR_ARGUMENT, "out is NULL");
    *out = nullptr;
    if (degree < 1 || degree > 3) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: Wrong value of degree (1,2 or 3)");
    if (nx < 2 || nx > kNxMax || (nx % 2) != 0) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: nx must be even and in [2, 256]");
    if (!(xmax > xmin)) return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: xmax must exceed xmin");
    int rc = check_device();
    if (rc) return rc;
    gempic_maxwell1d *m = new gempic_maxwell1d();
    m->nx = nx;
    m->xmin = xmin;
    m->xmax = xmax;
    m->dx = (xmax - xmin) / (double)nx;
    m->degree = degree;
    gh::maxwell1d_tables(nx, degree, m->tabs);
    hipError_t e = hipStreamCreate(&m->stream);
    if (e == hipSuccess) e = dalloc(&m->d_grid, (size_t)NSLOT * nx);
    if (e == hipSuccess) e = dalloc(&m->d_tabs, (size_t)NTAB * nx);
    if (e == hipSuccess) e = dalloc(&m->d_scalar, 8);
    if (e == hipSuccess) e = hipMemset(m->d_grid, 0, sizeof(double) * NSLOT * nx);
    if (e == hipSuccess) {
        std::vector<double> T((size_t)NTAB * nx, 0.0);
        auto put = [&](int slot, const std::vector<double> &v) { std::copy(v.begin(), v.end(), T.begin() + (size_t)slot * nx); };
        put(T_COS, m->tabs.cos_tab); put(T_SIN, m->tabs.sin_tab);
        put(T_INVM0, m->tabs.inv_mass0); put(T_INVM1, m->tabs.inv_mass1);
        put(T_AMP, m->tabs.eig_weak_ampere); put(T_POIS, m->tabs.eig_weak_poisson);
        put(T_M0, m->tabs.eig_mass0); put(T_M1, m->tabs.eig_mass1);
        put(T_CM0, m->tabs.circ_m0); put(T_CM1, m->tabs.circ_m1); put(T_CAMP, m->tabs.circ_amp);
        put(T_CMASS1, m->tabs.circ_mass1); put(T_CPOIS, m->tabs.circ_pois);
        e = hipMemcpy(m->d_tabs, T.data(), sizeof(double) * T.size(), hipMemcpyHostToDevice);
    }
    if (e != hipSuccess) {
        gempic_maxwell1d_destroy(m);
        return fail(GEMPIC_ERR_DEVICE, std::string("Maxwell1DFEM allocation: ") + hipGetErrorString(e));
    }
    *out = m;
    return GEMPIC_OK;
}

int gempic_maxwell1d_compute_rhs_from_function(gempic_maxwell1d *m, gempic_fn1d f, void *ctx,
                                               int degree, double *coefs)
{
    if (!m || !f || !coefs) return fail(GEMPIC_ERR_ARGUMENT, "NULL argument");
    if (degree < 0 || degree > 3)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree must be 0..3");
    // gausslegendre(degree + 1) on [0, 1] (closed forms) and the splines there
    double x[4], w[4], bspl[4][4];
    gh::gauss_legendre(degree + 1, x, w);
    for (int k = 0; k <= degree; ++k) {
        x[k] = 0.5 * (x[k] + 1.0);
        w[k] = 0.5 * w[k];
        gh::bspline_host(degree, x[k], bspl[k]);
    }
    for (int64_t i = 1; i <= m->nx; ++i) {
        double coef = 0.0;
        for (int j = 1; j <= degree + 1; ++j)
            for (int k = 1; k <= degree + 1; ++k) {
                const double xq = ((x[k - 1] + (double)i) + (double)j) - 2.0;
                coef = coef + w[k - 1] * f(m->dx * xq, ctx) * bspl[k - 1][degree + 1 - j];
            }
        coefs[i - 1] = coef * m->dx;
    }
    return GEMPIC_OK;
}

int gempic_maxwell1d_l2projection(gempic_maxwell1d *m, gempic_fn1d f, void *ctx, int degree,
                                  double *coefs)
{
    if (!m) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
    if (degree != m->degree && degree != m->degree - 1)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: degree " + std::to_string(degree) + " not available");
    int rc = gempic_maxwell1d_compute_rhs_from_function(m, f, ctx, degree, coefs);
    if (rc) return rc;
    // the reference solves the mass system into its workspace and returns
    // coefs_dofs ./ delta_x, the right-hand side over dx
    for (int64_t i = 0; i < m->nx; ++i) coefs[i] = coefs[i] / m->dx;
    return GEMPIC_OK;
}

int gempic_maxwell1d_destroy(gempic_maxwell1d *m)
{
    if (!m) return GEMPIC_OK;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    if (m->d_grid) (void)hipFree(m->d_grid);
    if (m->d_tabs) (void)hipFree(m->d_tabs);
    if (m->d_scalar) (void)hipFree(m->d_scalar);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return GEMPIC_OK;
}

int gempic_maxwell1d_tables(gempic_maxwell1d *m, double *e0, double *e1, double *ea, double *ep)
{
    if (!m) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
    const size_t nb = sizeof(double) * m->nx;
    if (e0) std::memcpy(e0, m->tabs.eig_mass0.data(), nb);
    if (e1) std::memcpy(e1, m->tabs.eig_mass1.data(), nb);
    if (ea) std::memcpy(ea, m->tabs.eig_weak_ampere.data(), nb);
    if (ep) std::memcpy(ep, m->tabs.eig_weak_poisson.data(), nb);
    return GEMPIC_OK;
}

// run one field op: inputs uploaded to slots a/b/out, output slot downloaded
static int mx_run(gempic_maxwell1d *m, int op, double dt, const double *in_a, const double *in_b,
                  double *inout, double *scalar)
{
    if (!m) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
    const size_t nb = sizeof(double) * m->nx;
    const int64_t nx = m->nx;
    const int SA = S_J1, SB = S_J2, SO = S_E1;
    if (in_a) HIP_TRY(hipMemcpyAsync(m->d_grid + SA * nx, in_a, nb, hipMemcpyHostToDevice, m->stream));
    if (in_b) HIP_TRY(hipMemcpyAsync(m->d_grid + SB * nx, in_b, nb, hipMemcpyHostToDevice, m->stream));
    if (inout) HIP_TRY(hipMemcpyAsync(m->d_grid + SO * nx, inout, nb, hipMemcpyHostToDevice, m->stream));
    GridProg g = prog1(op, dt, SA, SB, SO);
    HIP_TRY(launch_grid(g, (int)nx, m->dx, m->d_grid, m->d_tabs, m->d_scalar, m->stream));
    if (inout) HIP_TRY(hipMemcpyAsync(inout, m->d_grid + SO * nx, nb, hipMemcpyDeviceToHost, m->stream));
    if (scalar) HIP_TRY(hipMemcpyAsync(scalar, m->d_scalar, sizeof(double), hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    return GEMPIC_OK;
}

int gempic_maxwell1d_compute_e_from_rho(gempic_maxwell1d *m, double *e, const double *rho)
{
    if (!e || !rho) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    return mx_run(m, G_E_FROM_RHO, 0.0, rho, nullptr, e, nullptr);
}

int gempic_maxwell1d_compute_e_from_j(gempic_maxwell1d *m, double *e, const double *current, int component)
{
    if (!e || !current) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (component != 1 && component != 2)
        return fail(GEMPIC_ERR_ARGUMENT, "ArgumentError: Component not implemented");
    return mx_run(m, component == 1 ? G_E_FROM_J1 : G_E_FROM_J2, 0.0, current, nullptr, e, nullptr);
}

int gempic_maxwell1d_compute_e_from_b(gempic_maxwell1d *m, double *e, double dt, const double *b)
{
    if (!e || !b) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    return mx_run(m, G_HB, dt, b, nullptr, e, nullptr);
}

int gempic_maxwell1d_compute_b_from_e(gempic_maxwell1d *m, double *b, double dt, const double *e)
{
    if (!e || !b) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    return mx_run(m, G_HE_B, dt, e, nullptr, b, nullptr);
}

int gempic_maxwell1d_inner_product(gempic_maxwell1d *m, const double *c1, const double *c2,
                                   int degree, double *out)
{
    if (!c1 || !c2 || !out) return fail(GEMPIC_ERR_ARGUMENT, "NULL array");
    if (!m) return fail(GEMPIC_ERR_ARGUMENT, "null handle");
    int op;
    if (degree == m->degree) op = G_INNER_M0;
    else if (degree == m->degree - 1) op = G_INNER_M1;
    else return fail(GEMPIC_ERR_ARGUMENT, "degree must be s_deg_0 or s_deg_1");
    return mx_run(m, op, 0.0, c1, c2, nullptr, out);
}

int gempic_maxwell1d_l2norm_squared(gempic_maxwell1d *m, const double *c, int degree, double *out)
{
    return gempic_maxwell1d_inner_product(m, c, c, degree, out);
}

}  // extern "C"
