// ggx.hip -- libggx: device context, arena management and the batched timestep.
//
// Replaces the bodies of the grainhdl phase loops (src/grainhdl.cpp:755-869, 1243-1256,
// 1381-1394) with batched HIP launches.  Per step, with no host round trip:
//   k_reset / k_prep / k_tally (k_schedule for small networks)
//                      deletion of grains that vanished in the previous step, survivor count,
//                      filing of live grains into box-size buckets, allocator reset
//   k_lists            comparison lists (computeSecondOrderNeighbours)
//   k_conv_tiles / k_conv_strip / k_conv_fft
//                      convolution of every live box (executeConvolution)
//   k_compare, k_contour, k_alloc, k_redist
//                      comparison, contour / motion check / new box / neighbours / volume, room for
//                      the new boxes, redistancing (executeComparison .. executeRedistancing), one
//                      launch per range of buckets (level_groups)
// A launch gets the LDS the largest box of its buckets needs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "ggx.h"
#include "ggx_internal.h"
#include "kernels.h"
#include "level.h"
#include "fft.h"
#include "coarsen.h"
#include "adjoint.h"

using namespace ggx;

namespace {

// Built-in box-size buckets (upper edges); ggx_options.bucket_edges replaces them (autotuner).
const int kDefaultEdges[] = {24, 32, 40, 48, 56, 64, 96, 128, 192, 256, 512};
constexpr int kDefaultBuckets = sizeof(kDefaultEdges) / sizeof(kDefaultEdges[0]);
static_assert(kDefaultBuckets <= kMaxBuckets, "bucket table");

template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
};

}  // namespace

struct ggx_ctx {
    ggx_settings s;
    ggx_derived d;
    ggx_options opt;
    std::string err;
    int dev = 0;
    hipStream_t stream = nullptr;
    int lds_max = 65536;
    int cu_count = 0;
    bool loaded = false;
    int max_id = 0;
    int nslots = 0;
    int loop = 0;
    size_t esize = 8;  // sizeof field element

    // arenas (field type erased)
    void* P[2] = {nullptr, nullptr};
    void* Tt = nullptr;
    void* Cf = nullptr;            // compared fields, at the offsets of the step's input layout
    unsigned long long* bits = nullptr;  // sign planes of the compared fields (level.h)
    unsigned long long* gather_part = nullptr;  // running sums of the neighbour pixels compared
    uint32_t* I[2] = {nullptr, nullptr};
    int cur = 0;       // P[cur] holds phi of the current layout
    int icur = 0;      // I[icur] holds the IDLocal written by the previous step
    long long field_cap = 0;       // field-arena elements a step may allocate
    long long field_alloc = 0;     // field-arena elements allocated (>= the initial layout)
    double2* pts = nullptr;
    long long contour_cap = 0;

    // per-grain arrays
    Box *box = nullptr, *box_next = nullptr;
    long long *off = nullptr, *off_next = nullptr, *off_prev = nullptr;
    int* nprev = nullptr;
    int *flags = nullptr, *errs = nullptr;
    int *sec_cnt = nullptr, *sec = nullptr, *cmp_cnt = nullptr, *cmp = nullptr;
    int4* newbox = nullptr;
    long long* coff = nullptr;
    int *ccap = nullptr, *clen = nullptr;
    double *volume = nullptr, *perimeter = nullptr, *energy = nullptr, *meanda = nullptr;
    int *nb_cnt = nullptr, *nb_id = nullptr;
    double* nb_len = nullptr;
    Sched* sched = nullptr;        // device counters of the current step
    Sched* h_sched = nullptr;      // pinned copy, filled at the end of every ggx_step call
    int* blists = nullptr;         // per-bucket work lists (nbuckets x nslots)
    int nbuckets = 0;              // box-size buckets of this context and their upper edges
    int edges[kMaxBuckets] = {};
    unsigned fft_mask = 0;         // bit b: bucket b convolves by FFT (ConvolutionMode 2, engine AUTO)
    int* alist = nullptr;          // all live grains
    int* live = nullptr;
    int* perm = nullptr;                        // grain ids in Z order of their initial box centres
    int *pg_list = nullptr, *pg_one = nullptr;  // per-grain baseline: one-grain work lists
    long long updates_total = 0;
    int lds_per_cu = 163840;
    int static_contour = 0;        // static LDS bytes of k_contour (the largest of its forms)
    int static_redist = 0;         // and of k_redist

    // circulant kernels of every box side 1 .. kMaxBox
    long long* kern_off = nullptr;
    void* kern = nullptr;
    // FFT engine: twiddles of every side 1 .. kMaxBox, global half-spectrum slots for boxes
    // above kFftLdsMax (kFftWideGrid workgroups), static LDS of k_conv_fft<T, LDS>
    double2* tw = nullptr;
    void* fft_work = nullptr;
    int static_fft[2][2] = {{0, 0}, {0, 0}};

    // anisotropic boundaries (K.on): orientations, boundary properties per direct neighbour,
    // junctions of the last contour, origin of the IDLocal window of the last comparison
    AnisoConst K{};
    double4* quat = nullptr;
    double *nb_e = nullptr, *nb_m = nullptr;
    Junc* junc = nullptr;
    int* jcnt = nullptr;
    int2* idl_org = nullptr;
    unsigned char* seg_code = nullptr;  // k_sectors' output for k_aniso, per contour point ...
    double* seg_arc = nullptr;
    SectorRecord* sectors = nullptr;    // ... and per grain
    // grid coarsening: grainhdl::ngrains (the grain count at the last coarsening) and the number of
    // coarsenings so far
    int ngrains = 0;
    int coarsenings = 0;
    int merge_bucket = -1;  // >= 0: a small network's level-set launch over buckets 0..merge_bucket

    // a recorded step (ggx_record_next_step) and what its adjoint reads: snapshots of the state
    // the corrector saw, the convolved fields before the corrector, the set-compared fields and
    // comparison winners of the step, and the adjoint work arrays.  Allocated at the first record.
    struct Record {
        bool armed = false, valid = false;
        int loop = 0;
        int *flags = nullptr, *nprev = nullptr, *clen = nullptr, *jcnt = nullptr, *nb_cnt = nullptr, *nb_id = nullptr;
        Box* box = nullptr;
        long long *off = nullptr, *off_prev = nullptr, *coff = nullptr;
        int2* idl_org = nullptr;
        double2* pts = nullptr;
        Junc* junc = nullptr;
        double *nb_e = nullptr, *nb_m = nullptr;
        double *tilde0 = nullptr, *phi0 = nullptr, *s = nullptr, *lam_s = nullptr, *lam_u = nullptr;
        int *win = nullptr, *area = nullptr;
        double *d_area = nullptr, *d_perim = nullptr, *grad = nullptr;
        const double* phi = nullptr;      // the step's input fields (phi0: the level-set kernel's
                                          // layout without LDS tiles compares in the input slots)
        const uint32_t* idl = nullptr;    // the IDLocal the corrector read
    } rec;

    // host mirrors
    std::vector<double> h_quat;    // orientation quaternion per grain id (q0..q3)
    std::vector<int> h_flags;
    std::vector<Box> h_box;
    std::vector<int> h_live;
    std::vector<int> h_err;

    // frame readback (ggx_frame_begin / ggx_frame_get): device staging of the arrays the next
    // step overwrites, pinned host copies filled on a copy stream
    struct Frame {
        bool copying = false;     // D2H copies of P[cur] / I[icur] in flight: the step after next waits
        bool valid = false;
        int loop = 0;
        long long nfield = 0, nidl = 0, npts = 0;
        size_t small_bytes = 0;
        hipStream_t cs = nullptr;
        hipEvent_t staged = nullptr, done = nullptr;
        void* d_small = nullptr; size_t d_small_cap = 0;
        double2* d_pts = nullptr; size_t d_pts_cap = 0;
        void* h_small = nullptr; size_t h_small_cap = 0;
        void* h_phi = nullptr; size_t h_phi_cap = 0;
        uint32_t* h_idl = nullptr; size_t h_idl_cap = 0;
        double2* h_pts = nullptr; size_t h_pts_cap = 0;
        std::vector<ggx_grain_info> info;
        std::vector<double> phi64;
        std::vector<int64_t> phi_off, idl_off, contour_off;
    } fr;

    hipGraphExec_t graph_exec[2] = {nullptr, nullptr};  // captured step per buffer parity
    std::vector<std::vector<hipEvent_t>> graph_events;  // [start, -, -, end] of replayed steps

    // stats: per-step phase events, read back at ggx_get_stats
    std::vector<std::vector<hipEvent_t>> ev_pending;
    std::vector<std::vector<hipEvent_t>> ev_free;
    ggx_stats st;
};

namespace {

int fail(ggx_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    return code;
}

#define HIPCHK(call)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return fail(ctx, GGX_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_));   \
    } while (0)

template <class X>
int dalloc(ggx_ctx* ctx, X*& p, size_t count) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(X));
    if (e != hipSuccess) return fail(ctx, GGX_E_OOM, std::string("hipMalloc: ") + hipGetErrorString(e));
    p = (X*)q;
    return GGX_OK;
}

template <class X>
void dfree(X*& p) {
    if (p) (void)hipFree((void*)p);
    p = nullptr;
}

int contour_cap_of(int n) { return contour_cap(n); }

long long aligned(long long v) { return (v + kAlign - 1) / kAlign * kAlign; }

// K_n[m] = sum_k g(k) cos(2 pi k m / n), g(k) = exp(-c min(k,n-k)^2) / n with the Gaussian
// exponent of box.cpp:682 split per dimension: c = sqrt(2/pi) 4 dt R^2 pi^2 / n^2.  The cosines
// come from one table of cos(2 pi e / n), e = k m mod n.
void circulant(int n, double dt, int R, std::vector<long double>& K) {
    const long double PI = 3.14159265358979323846264338327950288L;
    K.assign((size_t)n, 0.0L);
    long double c = std::sqrt(2.0L / PI) * 4.0L * (long double)dt * (long double)R * (long double)R * PI * PI /
                    ((long double)n * (long double)n);
    std::vector<long double> g((size_t)n), cs((size_t)n);
    for (int k = 0; k < n; ++k) {
        int k2 = std::min(k, n - k);
        g[k] = std::exp(-c * (long double)k2 * (long double)k2) / (long double)n;
        cs[k] = std::cos(2.0L * PI * (long double)k / (long double)n);
    }
    // four sums at a time: each is a chain of dependent additions in the order of k
    for (int m = 0; m < n; m += 4) {
        long double s[4] = {0.0L, 0.0L, 0.0L, 0.0L};
        int e[4] = {0, 0, 0, 0}, d[4];
        for (int u = 0; u < 4; ++u) d[u] = std::min(m + u, n - 1);
        for (int k = 0; k < n; ++k)
            for (int u = 0; u < 4; ++u) {
                s[u] += g[k] * cs[e[u]];
                e[u] += d[u];
                if (e[u] >= n) e[u] -= n;
            }
        for (int u = 0; u < 4 && m + u < n; ++u) K[m + u] = s[u];
    }
}

// Offset of the table of box side n: sum of ktab_len(m) for m < n.
long long kern_offset(int n) { return (long long)n * (n - 1) + 2LL * kKPad * n; }

// Table of box side n, at its place in the packed tables.
template <class X>
void kernel_table(int n, double dt, int R, std::vector<long double>& K, X* packed) {
    circulant(n, dt, R, K);
    if (sizeof(X) == 4) {
        // FP32: the taps rounded to float no longer sum to one, which would bias every convolved
        // field by (gain - 1) delta at every step and move all interfaces the same way; the
        // centre tap takes up the rounding so that the float taps sum to one
        long double sum = 0.0L;
        for (int m = 1; m < n; ++m) sum += (long double)(float)K[(size_t)m];
        K[0] = 1.0L - sum;
    }
    X* w = packed + kern_offset(n);
    const long long len = ktab_len(n);
    for (long long t = 0; t < len; ++t) w[t] = (X)K[(size_t)(((t - kKPad) % n + n) % n)];
}

// Tables of every box side a step can meet (1 .. min(kMaxBox, ngridpoints)), built once.  The sums
// in 80-bit arithmetic are most of a load's time (sides to 512: 4.5e7 terms, 110 ms on one core), so
// the sides are shared out, the longest first, among up to 16 threads.  A load of 2000 grains 112 -> 9.6 ms, of 100 grains 11.7 -> 2.5 ms.
template <class X>
int build_kernels_of(ggx_ctx* ctx) {
    const int nmax = std::min(kMaxBox, ctx->d.ngridpoints);
    std::vector<X> w((size_t)kern_offset(nmax + 1), X(0));
    std::atomic<int> next{nmax};
    std::atomic<bool> ok{true};
    auto work = [&]() {
        try {
            std::vector<long double> K;
            for (int n; (n = next.fetch_sub(1)) >= 1;) kernel_table(n, ctx->d.dt, ctx->d.real_domain_size, K, w.data());
        } catch (...) {
            ok = false;
        }
    };
    const int helpers = std::min({15, (int)std::thread::hardware_concurrency() - 1, nmax / 32});
    std::vector<std::thread> pool;
    try {
        for (int t = 0; t < helpers; ++t) pool.emplace_back(work);
    } catch (...) {  // fewer helpers, then
    }
    work();
    for (std::thread& t : pool) t.join();
    if (!ok) return fail(ctx, GGX_E_OOM, "circulant tables: out of host memory");
    HIPCHK(hipMemcpy(ctx->kern, w.data(), w.size() * sizeof(X), hipMemcpyHostToDevice));
    return GGX_OK;
}

int build_kernels(ggx_ctx* ctx) { return ctx->esize == 8 ? build_kernels_of<double>(ctx) : build_kernels_of<float>(ctx); }

GridConst grid_const(const ggx_ctx* ctx) {
    GridConst G;
    G.m = ctx->d.ngridpoints;
    G.gb = ctx->d.grid_blowup;
    G.R = ctx->d.real_domain_size;
    G.nslots = ctx->nslots;
    G.h = ctx->d.h;
    G.delta = ctx->d.delta;
    G.dt = ctx->d.dt;
    return G;
}

int raise_lds(ggx_ctx* ctx) {
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, ctx->dev));
    ctx->cu_count = prop.multiProcessorCount;
    int lim = (int)prop.sharedMemPerBlock;
    int smp = (int)prop.maxSharedMemoryPerMultiProcessor;
    if (smp > 0) ctx->lds_per_cu = smp;
    if (smp > lim) lim = smp;
    if (ctx->opt.lds_budget > 0) lim = std::min(lim, ctx->opt.lds_budget);
    // allow the dynamic-LDS kernels to use up to `lim`
    const void* fns[] = {(const void*)k_conv_strip<double, 2>, (const void*)k_conv_strip<float, 2>,
                         (const void*)k_conv_fft<double, true>, (const void*)k_conv_fft<double, false>,
                         (const void*)k_conv_fft<float, true>, (const void*)k_conv_fft<float, false>,
                         (const void*)k_contour<double, false, false, 64>, (const void*)k_contour<double, false, false, 256>,
                         (const void*)k_contour<float, false, false, 64>, (const void*)k_contour<float, false, false, 256>,
                         (const void*)k_contour<double, true, false, 64>, (const void*)k_contour<double, true, false, 256>,
                         (const void*)k_contour<float, true, false, 64>, (const void*)k_contour<float, true, false, 256>,
                         (const void*)k_contour<double, false, true, 256>, (const void*)k_contour<float, false, true, 256>,
                         (const void*)k_contour<double, true, true, 256>, (const void*)k_contour<float, true, true, 256>,
                         (const void*)k_redist<double, 64>, (const void*)k_redist<double, 128>, (const void*)k_redist<double, 256>,
                         (const void*)k_redist<float, 64>, (const void*)k_redist<float, 128>, (const void*)k_redist<float, 256>,
                         (const void*)k_conv_strip<double, 4>, (const void*)k_conv_strip<double, 8>,
                         (const void*)k_conv_strip<float, 4>, (const void*)k_conv_strip<float, 8>,
                         (const void*)k_conv_tiles<double, 2>, (const void*)k_conv_tiles<double, 3>, (const void*)k_conv_tiles<double, 4>,
                         (const void*)k_conv_tiles<float, 2>, (const void*)k_conv_tiles<float, 3>, (const void*)k_conv_tiles<float, 4>};
    constexpr int kFns = (int)(sizeof(fns) / sizeof(fns[0])), kContour0 = 6, kRedist0 = 18, kRedist1 = 24;
    for (const void* f : fns) {
        hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lim);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            lim = std::min(lim, (int)prop.sharedMemPerBlock);
        }
    }
    ctx->lds_max = lim;
    // the strips' launches ask for what their boxes need, within lds_max: one ceiling for every context
    (void)hipFuncSetAttribute((const void*)k_box_rows<StepBoxes>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)box_rows_lds(kMaxBox));
    if (hipFuncSetAttribute((const void*)k_box_columns<StepBoxes>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)box_columns_lds(kMaxBox)) != hipSuccess)
        (void)hipGetLastError();
    // static __shared__ bytes count against the same per-workgroup limit as the dynamic request
    int* dst[] = {&ctx->static_fft[0][1], &ctx->static_fft[0][0], &ctx->static_fft[1][1], &ctx->static_fft[1][0]};
    for (int k = 0; k < kFns; ++k) {
        hipFuncAttributes fa;
        HIPCHK(hipFuncGetAttributes(&fa, fns[k]));
        const int st = (int)fa.sharedSizeBytes;
        if (k >= 2 && k < 6) *dst[k - 2] = st;
        else if (k >= kRedist0 && k < kRedist1) ctx->static_redist = std::max(ctx->static_redist, st);
        else if (k >= kContour0 && k < kRedist0) ctx->static_contour = std::max(ctx->static_contour, st);
    }
    return GGX_OK;
}


void build_live(ggx_ctx* ctx) {
    ctx->h_live.clear();
    for (int g = 1; g < ctx->nslots; ++g)
        if ((ctx->h_flags[g] & kPresent) && (ctx->h_flags[g] & kExists)) ctx->h_live.push_back(g);
}

// Contour points of a slot of bucket b.  A small network's buckets up to kMergeSide share one size.
int slot_cap(const ggx_ctx* ctx, int b) { return contour_cap(ctx->edges[std::max(b, ctx->merge_bucket)]); }

Buckets bucket_table(const ggx_ctx* ctx) {
    Buckets B;
    B.count = ctx->nbuckets;
    for (int b = 0; b < kMaxBuckets; ++b) {
        B.edge[b] = b < ctx->nbuckets ? ctx->edges[b] : 0;
        B.cap[b] = b < ctx->nbuckets ? slot_cap(ctx, b) : 0;
    }
    return B;
}

int per_cu(const ggx_ctx* ctx, long long lds) {
    long long k = lds > 0 ? ctx->lds_per_cu / lds : 8;
    return (int)std::max<long long>(1, std::min<long long>(8, k));
}

// The velocity corrector of anisotropic networks on the convolved fields of a list's grains (items:
// how many at most), before any comparison reads them.
template <class T>
void launch_aniso(ggx_ctx* ctx, hipStream_t st, const int* list, const int* count, int items, const T* P, T* Tt,
                  const uint32_t* Iold) {
    AnisoArgs<T> A;
    A.list = list; A.count = count; A.box = ctx->box; A.off = ctx->off;
    A.phi = P; A.tilde = Tt; A.idl = Iold; A.off_prev = ctx->off_prev; A.n_prev = ctx->nprev;
    A.flags = ctx->flags; A.err = ctx->errs; A.nslots = ctx->nslots;
    A.pts = ctx->pts; A.coff = ctx->coff; A.clen = ctx->clen; A.nb_cnt = ctx->nb_cnt; A.nb_id = ctx->nb_id;
    A.S.quat = ctx->quat; A.S.nb_e = ctx->nb_e; A.S.nb_m = ctx->nb_m; A.S.junc = ctx->junc; A.S.jcnt = ctx->jcnt;
    A.S.idl_org = ctx->idl_org;
    A.K = ctx->K;
    A.loop = &ctx->sched->loop_cur;
    A.h = ctx->d.h;
    A.delta = ctx->d.delta;
    A.seg_code = ctx->seg_code; A.seg_arc = ctx->seg_arc; A.sectors = ctx->sectors;
    const int grid = std::max(1, std::min(items, ctx->cu_count * 64));
    hipLaunchKernelGGL(k_sectors<T>, dim3(grid), dim3(64), 0, st, A);
    hipLaunchKernelGGL(k_aniso<T>, dim3(grid), dim3(256), 0, st, A);
}

AnisoState aniso_state(const ggx_ctx* ctx) {
    AnisoState S;
    S.quat = ctx->quat; S.nb_e = ctx->nb_e; S.nb_m = ctx->nb_m; S.junc = ctx->junc; S.jcnt = ctx->jcnt;
    S.idl_org = ctx->idl_org;
    return S;
}

// The arguments every kernel of the level-set phase shares.
template <class T>
LevelArgs<T> level_args(const ggx_ctx* ctx) {
    LevelArgs<T> A;
    A.box = ctx->box; A.off = ctx->off; A.cmp_cnt = ctx->cmp_cnt; A.cmp = ctx->cmp;
    A.tilde = (const T*)ctx->Tt; A.cfield = (T*)ctx->Cf; A.bits = ctx->bits; A.plane = plane_words(ctx->field_alloc);
    A.idl_old = ctx->I[ctx->icur]; A.idl_new = ctx->I[ctx->icur ^ 1];
    A.off_prev = ctx->off_prev; A.n_prev = ctx->nprev; A.out_field = (T*)ctx->P[ctx->cur ^ 1];
    A.rec_s = nullptr; A.rec_win = nullptr; A.rec_area = nullptr;
    ContourOut& O = A.O;
    O.pts = ctx->pts; O.coff = ctx->coff; O.ccap = ctx->ccap; O.clen = ctx->clen;
    O.volume = ctx->volume; O.perimeter = ctx->perimeter; O.energy = ctx->energy; O.meanda = ctx->meanda;
    O.nb_cnt = ctx->nb_cnt; O.nb_id = ctx->nb_id; O.nb_len = ctx->nb_len;
    O.box_next = ctx->box_next; O.off_next = ctx->off_next; O.flags = ctx->flags; O.err = ctx->errs;
    O.tops = &ctx->sched->tops[0]; O.field_cap = ctx->field_cap; O.contour_cap = ctx->contour_cap;
    A.G = grid_const(ctx); A.loop = &ctx->sched->loop_cur; A.analysis_timestep = ctx->s.analysis_timestep;
    A.gather_part = ctx->gather_part; A.out_total = &ctx->sched->out_total;
    A.contour_base = ctx->sched->contour_base;
    A.K = ctx->K; A.AS = aniso_state(ctx);
    return A;
}

// Buckets b0 .. b1 of the work lists as one launch's items.
Items bucket_items(const ggx_ctx* ctx, int b0, int b1) {
    Items it;
    it.lists = ctx->blists; it.total = ctx->sched->bucket_total; it.stride = ctx->nslots;
    it.b0 = b0; it.b1 = b1;
    for (int b = 0; b < kMaxBuckets; ++b) it.cap[b] = b < ctx->nbuckets ? slot_cap(ctx, b) : 0;
    return it;
}

Items single_item(const int* list, const int* one, int n) {  // a one-grain work list, box side n
    Items it;
    it.lists = list; it.total = one; it.stride = 0;
    it.b0 = it.b1 = 0;
    for (int b = 0; b < kMaxBuckets; ++b) it.cap[b] = b == 0 ? contour_cap(n) : 0;
    return it;
}

template <class T>
void level_items(const ggx_ctx* ctx, LevelArgs<T>& A, int b0, int b1) {
    A.it = bucket_items(ctx, b0, b1);
    A.cap = 0;
    for (int b = b0; b <= b1; ++b) A.cap = std::max(A.cap, A.it.cap[b]);
    A.nb = ctx->edges[b1];
}

// The bucket ranges the level-set kernels are launched over.  Buckets up to side 64 each have a
// launch sized for them, unless the network is small (one launch for all of them: there a launch
// lasts as long as its slowest grain); the buckets up to 128 and those above share one each.
std::vector<std::pair<int, int>> level_groups(const ggx_ctx* ctx) {
    std::vector<std::pair<int, int>> R;
    int b = 0;
    if (ctx->merge_bucket >= 0) {
        R.push_back({0, ctx->merge_bucket});
        b = ctx->merge_bucket + 1;
    }
    while (b < ctx->nbuckets) {
        const int lim = ctx->edges[b] <= 64 ? ctx->edges[b] : (ctx->edges[b] <= 128 ? 128 : kMaxBox);
        int e = b;
        while (e + 1 < ctx->nbuckets && ctx->edges[e + 1] <= lim) ++e;
        R.push_back({b, e});
        b = e + 1;
    }
    return R;
}

// Every live grain as one launch's items, in the spatial order of the list.
Items all_items(const ggx_ctx* ctx) {
    Items it = bucket_items(ctx, 0, 0);
    it.lists = ctx->alist; it.total = &ctx->sched->all_total;
    return it;
}

// One launch over grains of every side (A.nb: the largest).  Six waves per grain, the blocks of a
// common box; more, which leaves a wave fewer blocks to loop over, where that few would not fill
// the chip.  Many more workgroups than fit at a time: their sizes differ, and the ones that wait
// even them out (with 8 per CU, of which 6 fit, the last two ran alone).
template <class T>
int launch_compare(const ggx_ctx* ctx, hipStream_t st, LevelArgs<T>& A, int items, bool coarsen) {
    const int full = ((A.nb + kRows - 1) / kRows) * ((A.nb + 63) / 64);
    A.blocks = std::min({32, full, std::max(6, ctx->cu_count * 64 / std::max(1, items))});
    const long long wgs = ((long long)items * A.blocks + 3) / 4;
    const int grid = (int)std::max<long long>(1, std::min<long long>(wgs, ctx->cu_count * 128));
    if (coarsen) hipLaunchKernelGGL((k_compare<T, true>), dim3(grid), dim3(256), 0, st, A);
    else hipLaunchKernelGGL((k_compare<T, false>), dim3(grid), dim3(256), 0, st, A);
    return GGX_OK;
}

template <class T>
int launch_contour(ggx_ctx* ctx, hipStream_t st, LevelArgs<T>& A, int items, bool coarsen) {
    const bool wide = coarsen || A.nb > 64;
    const long long lds = contour_layout(A.nb, A.cap, wide ? 256 : 64).total;
    if (lds + ctx->static_contour + 256 > ctx->lds_max)
        return fail(ctx, GGX_E_BOUNDS, "box too large for the contour kernel: side " + std::to_string(A.nb) + " needs " +
                                           std::to_string(lds) + " of " + std::to_string(ctx->lds_max) + " LDS bytes");
    const int grid = std::max(1, std::min(items, ctx->cu_count * 128));
    const size_t l = (size_t)lds;
    if (coarsen) {
        if (ctx->K.on) hipLaunchKernelGGL((k_contour<T, true, true, 256>), dim3(grid), dim3(256), l, st, A);
        else hipLaunchKernelGGL((k_contour<T, false, true, 256>), dim3(grid), dim3(256), l, st, A);
    } else if (ctx->K.on) {
        if (wide) hipLaunchKernelGGL((k_contour<T, true, false, 256>), dim3(grid), dim3(256), l, st, A);
        else hipLaunchKernelGGL((k_contour<T, true, false, 64>), dim3(grid), dim3(64), l, st, A);
    } else {
        if (wide) hipLaunchKernelGGL((k_contour<T, false, false, 256>), dim3(grid), dim3(256), l, st, A);
        else hipLaunchKernelGGL((k_contour<T, false, false, 64>), dim3(grid), dim3(64), l, st, A);
    }
    return GGX_OK;
}

template <class T>
int launch_redist(const ggx_ctx* ctx, hipStream_t st, LevelArgs<T>& A, int items) {
    const int room = ctx->lds_max - ctx->static_redist - 256;
    A.tile = A.nb + kTileMargin;
    if (A.tile > 256 || redist_lds<T>(A.tile) > room) A.tile = 0;
    const size_t lds = (size_t)redist_lds<T>(A.tile);
    const int grid = std::max(1, std::min(items, ctx->cu_count * 128));
    if (A.tile > 128 || A.tile == 0) hipLaunchKernelGGL((k_redist<T, 256>), dim3(grid), dim3(256), lds, st, A);
    else if (A.tile > 64) hipLaunchKernelGGL((k_redist<T, 128>), dim3(grid), dim3(128), lds, st, A);
    else hipLaunchKernelGGL((k_redist<T, 64>), dim3(grid), dim3(64), lds, st, A);
    return GGX_OK;
}

std::vector<hipEvent_t> take_events(ggx_ctx* ctx, int count) {
    std::vector<hipEvent_t> ev;
    if (!ctx->ev_free.empty()) {
        ev = ctx->ev_free.back();
        ctx->ev_free.pop_back();
    } else {
        ev.resize(count);
        for (auto& e : ev) (void)hipEventCreate(&e);
    }
    return ev;
}

// Bucket of a box side: the first whose upper edge holds it.
int bucket_of(const ggx_ctx* ctx, int n) {
    for (int b = 0; b < ctx->nbuckets; ++b)
        if (n <= ctx->edges[b]) return b;
    return ctx->nbuckets - 1;
}

// The FFT engine convolves a bucket when the symbol is not the separable Gaussian (modes 0 and
// 1 have no real-space circulant form), when the options ask for it, or when the tuned table
// picks it for that bucket.
bool fft_for(const ggx_ctx* ctx, int nb) {
    if (ctx->s.convolution_mode != 2) return true;
    if (ctx->opt.conv_engine == GGX_CONV_FFT) return true;
    if (ctx->opt.conv_engine == GGX_CONV_CIRCULANT) return false;
    return ((ctx->fft_mask >> bucket_of(ctx, nb)) & 1u) != 0;
}

FftSymbol fft_symbol_of(const ggx_ctx* ctx) {
    FftSymbol sy;
    sy.mode = ctx->s.convolution_mode;
    sy.dt = ctx->d.dt;
    sy.nsq = (double)ctx->d.real_domain_size * (double)ctx->d.real_domain_size;
    return sy;
}

// Workgroups of an FFT launch whose half spectra live in global slots (boxes above kFftLdsMax).
constexpr int kFftWideGrid = 64;

// Whether the half spectra of an FFT launch for boxes up to side nb stay in LDS.
template <class T>
bool fft_in_lds(const ggx_ctx* ctx, int nb) {
    return nb <= kFftLdsMax && fft_lds<T>(nb, true) + ctx->static_fft[sizeof(T) == 8 ? 0 : 1][1] + 256 <= ctx->lds_max;
}

// Whether the strips of boxes up to side nb fit the LDS this context may use.
template <class T>
bool boxes_for(const ggx_ctx* ctx, int nb) { return sizeof(T) == 8 && box_columns_lds(nb) + 256 <= ctx->lds_max; }

// Largest side of the buckets that share a launch of strips with a bucket of this edge.
int strips_limit(int side) { return side <= 64 ? 64 : side <= 128 ? 128 : side <= 256 ? 256 : kMaxBox; }

// Whether any launch of this context's steps runs the FFT (k_conv_fft), and with global slots.
template <class T>
void fft_needs(const ggx_ctx* ctx, bool* engine, bool* slots) {
    *engine = *slots = false;
    auto meet = [&](int nb, int strips_nb) {
        if (!fft_for(ctx, nb) || boxes_for<T>(ctx, strips_nb)) return;
        *engine = true;
        if (!fft_in_lds<T>(ctx, nb)) *slots = true;
    };
    if (ctx->opt.batching == GGX_BATCH_PERGRAIN)
        for (int n = 1; n <= kMaxBox; ++n) meet(n, n);
    else
        for (int b = 0; b < ctx->nbuckets; ++b) meet(ctx->edges[b], strips_limit(ctx->edges[b]));
}

template <class T>
int launch_conv_fft(ggx_ctx* ctx, hipStream_t st, const int* list, const int* count, int nb, int grid,
                    const T* src, T* dst) {
    const int ti = sizeof(T) == 8 ? 0 : 1;
    const bool in_lds = fft_in_lds<T>(ctx, nb);
    const long long lds = fft_lds<T>(nb, in_lds);
    if (lds + ctx->static_fft[ti][in_lds ? 1 : 0] + 256 > ctx->lds_max)
        return fail(ctx, GGX_E_BOUNDS, "box too large for the FFT line buffers: side " + std::to_string(nb));
    if (!ctx->tw || (!ctx->fft_work && !in_lds)) return fail(ctx, GGX_E_STATE, "FFT workspace missing");
    using C = typename Cplx<T>::type;
    if (in_lds) {
        if (grid <= 0) grid = ctx->cu_count * per_cu(ctx, lds + ctx->static_fft[ti][1]);
        hipLaunchKernelGGL((k_conv_fft<T, true>), dim3(grid), dim3(256), (size_t)lds, st, list, count, ctx->box,
                           ctx->off, src, dst, (const double2*)ctx->tw, fft_symbol_of(ctx), nb, (C*)nullptr);
    } else {
        // one global slot per workgroup: the grid is capped at the slots allocated
        grid = grid <= 0 ? kFftWideGrid : std::min(grid, kFftWideGrid);
        hipLaunchKernelGGL((k_conv_fft<T, false>), dim3(grid), dim3(256), (size_t)lds, st, list, count, ctx->box, ctx->off, src, dst, (const double2*)ctx->tw, fft_symbol_of(ctx), nb,
                           (C*)ctx->fft_work);
    }
    return GGX_OK;
}

// The three launches of strip products with the FFT engine's symbol over a launch's items, boxes up to
// side nb (FP64).
int launch_conv_boxes(ggx_ctx* ctx, hipStream_t st, const Items& it, int nb, int items, const double* src, double* dst) {
    StepBoxes B;
    B.it = it; B.strips = (nb + 15) / 16; B.nmax = nb; B.box = ctx->box; B.off = ctx->off;
    // replayed steps launch for the grains there may be: fewer workgroups, as most find none
    const long long cap = (long long)ctx->cu_count * (ctx->opt.persistent ? 16 : 64);
    const dim3 grid((unsigned)std::max<long long>(1, std::min((long long)items * B.strips, cap))), block(256);
    const size_t rows = (size_t)box_rows_lds(nb), columns = (size_t)box_columns_lds(nb);
    hipLaunchKernelGGL(k_box_rows<StepBoxes>, grid, block, rows, st, B, src, dst, 1);
    hipLaunchKernelGGL(k_box_columns<StepBoxes>, grid, block, columns, st, B, dst, fft_symbol_of(ctx));
    hipLaunchKernelGGL(k_box_rows<StepBoxes>, grid, block, rows, st, B, (const double*)dst, dst, 0);
    return GGX_OK;
}

// The circulant convolution of a launch's items, boxes up to side nb: the register tiles of 2, 3 or 4
// times 16 columns, the LDS strip above 64 and where the tiles are above the context's lds_budget.
template <class T>
int launch_conv(ggx_ctx* ctx, hipStream_t st, const Items& it, int nb, int items, const T* src, T* dst) {
    const int nt = (nb + 15) / 16;
    const T* kern = (const T*)ctx->kern;
    const int tiles = std::max(2, nt);
    if (nb <= 64 && conv_tiles_lds<T>(tiles) + 256 <= ctx->lds_max) {
        const size_t lds = (size_t)conv_tiles_lds<T>(tiles);
        const dim3 grid(std::max(1, std::min(items, ctx->cu_count * 64))), block(64 * tiles);
        if (tiles == 2)
            hipLaunchKernelGGL((k_conv_tiles<T, 2>), grid, block, lds, st, it, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
        else if (tiles == 3)
            hipLaunchKernelGGL((k_conv_tiles<T, 3>), grid, block, lds, st, it, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
        else
            hipLaunchKernelGGL((k_conv_tiles<T, 4>), grid, block, lds, st, it, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
        return GGX_OK;
    }
    const long long lds = conv_strip_lds<T>(nb);
    if (lds + 256 > ctx->lds_max) return fail(ctx, GGX_E_BOUNDS, "box too large for LDS strips");
    const dim3 grid((unsigned)std::max<long long>(1, std::min<long long>((long long)items * nt, ctx->cu_count * 64))), block(256);
    if (nb <= 128)
        hipLaunchKernelGGL((k_conv_strip<T, 2>), grid, block, (size_t)lds, st, it, nt, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
    else if (nb <= 256)
        hipLaunchKernelGGL((k_conv_strip<T, 4>), grid, block, (size_t)lds, st, it, nt, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
    else
        hipLaunchKernelGGL((k_conv_strip<T, 8>), grid, block, (size_t)lds, st, it, nt, ctx->box, ctx->off, src, dst, ctx->kern_off, kern);
    return GGX_OK;
}

int snapshot_for_adjoint(ggx_ctx* ctx, hipStream_t st, const void* P, const uint32_t* Iold);

template <class T>
int launch_step(ggx_ctx* ctx, bool timed, bool record = false) {
    hipStream_t st = ctx->stream;
    const int NS = ctx->nslots;
    T* P = (T*)ctx->P[ctx->cur];
    T* Tt = (T*)ctx->Tt;
    uint32_t* Iold = ctx->I[ctx->icur];
    const int cus = ctx->cu_count;
    Sched* S = ctx->sched;
    std::vector<hipEvent_t> ev;
    if (timed) ev = take_events(ctx, 5);

    if (timed) HIPCHK(hipEventRecord(ev[0], st));
    if (NS - 1 <= kSmallNetwork) {
        hipLaunchKernelGGL(k_schedule, dim3(1), dim3(1024), 0, st, NS, ctx->flags, ctx->box, bucket_table(ctx), ctx->blists,
                           ctx->alist, ctx->errs, S, (const int*)ctx->perm);
    } else {
        hipLaunchKernelGGL(k_reset, dim3(1), dim3(32), 0, st, S);
        hipLaunchKernelGGL(k_prep, dim3((NS + 255) / 256), dim3(256), 0, st, NS, ctx->flags, ctx->box, bucket_table(ctx),
                           ctx->blists, ctx->alist, ctx->errs, S, (const int*)ctx->perm);
        hipLaunchKernelGGL(k_tally, dim3(1), dim3(64), 0, st, S, bucket_table(ctx));
    }
    hipLaunchKernelGGL(k_lists, dim3(std::max(1, std::min(NS - 1, cus * 64))), dim3(64), 0, st, (const int*)ctx->alist,
                       (const int*)&S->all_total, ctx->box, ctx->flags, ctx->sec_cnt, ctx->sec, ctx->cmp_cnt, ctx->cmp, ctx->errs);
    if (timed) HIPCHK(hipEventRecord(ev[1], st));
    // grid per bucket: persistent (fixed) or one workgroup per grain (counts read back)
    int counts[kMaxBuckets];
    if (!ctx->opt.persistent) {
        HIPCHK(hipMemcpyAsync(ctx->h_sched, S, sizeof(Sched), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        for (int b = 0; b < ctx->nbuckets; ++b) counts[b] = ctx->h_sched->bucket_count[b];
    }
    // convolution, per range of buckets of one engine and tile count
    for (int b = 0; b < ctx->nbuckets;) {
        const bool fft = fft_for(ctx, ctx->edges[b]);
        int e = b;
        if (!fft) {
            auto tiles = [&](int k) {  // what a launch is sized for
                const int side = ctx->edges[k];
                return side <= 64 ? (ctx->merge_bucket >= 0 ? 4 : std::max(2, (side + 15) / 16)) : (side <= 128 ? 8 : side <= 256 ? 16 : 32);
            };
            while (e + 1 < ctx->nbuckets && !fft_for(ctx, ctx->edges[e + 1]) && tiles(e + 1) == tiles(b)) ++e;
        }
        bool strips = false;
        if (fft) {
            auto limit = [&](int k) { return strips_limit(ctx->edges[k]); };  // strips of one launch share its LDS
            strips = boxes_for<T>(ctx, limit(b));
            while (strips && e + 1 < ctx->nbuckets && fft_for(ctx, ctx->edges[e + 1]) && limit(e + 1) == limit(b)) ++e;
        }
        int items = NS - 1;
        if (!ctx->opt.persistent) {
            items = 0;
            for (int k = b; k <= e; ++k) items += counts[k];
        }
        int rc = GGX_OK;
        if (strips) {
            if (items > 0)
                rc = launch_conv_boxes(ctx, st, bucket_items(ctx, b, e), ctx->edges[e], items, (const double*)P, (double*)Tt);
        } else if (fft && (ctx->opt.persistent || items > 0))
            rc = launch_conv_fft<T>(ctx, st, ctx->blists + (size_t)b * NS, &S->bucket_total[b], ctx->edges[b],
                                    ctx->opt.persistent ? 0 : items, (const T*)P, Tt);
        else if (!fft && items > 0)
            rc = launch_conv<T>(ctx, st, bucket_items(ctx, b, e), ctx->edges[e], items, (const T*)P, Tt);
        if (rc) return rc;
        b = e + 1;
    }
    // a recorded step keeps the convolved fields before the corrector and the corrector's inputs
    if (record) {
        HIPCHK(hipMemcpyAsync(ctx->rec.tilde0, Tt, (size_t)ctx->field_alloc * sizeof(T), hipMemcpyDeviceToDevice, st));
        int rc = snapshot_for_adjoint(ctx, st, P, Iold);
        if (rc) return rc;
        HIPCHK(hipMemsetAsync(ctx->rec.area, 0, (size_t)ctx->nslots * 4, st));
    }
    if (ctx->K.on)
        launch_aniso<T>(ctx, st, ctx->alist, &S->all_total, ctx->opt.persistent ? NS - 1 : std::max(1, ctx->h_sched->all_count),
                        (const T*)P, Tt, Iold);
    if (timed) HIPCHK(hipEventRecord(ev[2], st));
    // comparison, contour, room for the new boxes, redistancing: per range of buckets
    LevelArgs<T> A = level_args<T>(ctx);
    A.rec_s = record ? (T*)ctx->rec.s : nullptr; A.rec_win = record ? ctx->rec.win : nullptr;
    A.rec_area = record ? ctx->rec.area : nullptr;
    const auto groups = level_groups(ctx);
    int all = 0;
    auto items = [&](const std::pair<int, int>& r) {  // grains of a launch: counted, or all the grains there are
        if (ctx->opt.persistent) return NS - 1;
        int c = 0;
        for (int b = r.first; b <= r.second; ++b) c += counts[b];
        return c;
    };
    A.it = all_items(ctx);
    A.nb = ctx->edges[ctx->nbuckets - 1];
    if (const int k = items({0, ctx->nbuckets - 1})) {
        const int rc = launch_compare<T>(ctx, st, A, k, false);
        if (rc) return rc;
    }
    for (int phase = 1; phase < 3; ++phase) {
        for (const auto& r : groups) {
            const int k = items(r);
            if (k == 0) continue;
            level_items(ctx, A, r.first, r.second);
            int rc = GGX_OK;
            if (phase == 1) { rc = launch_contour<T>(ctx, st, A, k, false); all += k; }
            else rc = launch_redist<T>(ctx, st, A, k);
            if (rc) return rc;
        }
        if (phase == 1) {
            const int grid = std::max(1, std::min((std::min(all, NS - 1) + 255) / 256, cus * 8));
            hipLaunchKernelGGL(k_alloc, dim3(grid), dim3(256), 0, st, (const int*)ctx->alist, (const int*)&S->all_total, A.O,
                               &S->out_total);
        }
    }
    if (timed) HIPCHK(hipEventRecord(ev[3], st));
    HIPCHK(hipGetLastError());
    if (timed) ctx->ev_pending.push_back(ev);
    return GGX_OK;
}

// A step as a hipGraph: captured once per buffer parity (the arenas and the per-grain array pairs
// swap every step, so even and odd steps launch with two fixed argument sets; everything else a
// step needs -- loop index, counters, work lists -- lives on the device), replayed afterwards.
// Only the persistent launches are captured: they need no host read-back inside a step.
template <class T>
int launch_step_graph(ggx_ctx* ctx) {
    const int parity = ctx->cur;
    if (!ctx->graph_exec[parity]) {
        hipGraph_t g = nullptr;
        HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        int rc = launch_step<T>(ctx, false);
        hipError_t e = hipStreamEndCapture(ctx->stream, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return fail(ctx, GGX_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
        e = hipGraphInstantiate(&ctx->graph_exec[parity], g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return fail(ctx, GGX_E_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    std::vector<hipEvent_t> ev = take_events(ctx, 5);
    HIPCHK(hipEventRecord(ev[0], ctx->stream));
    HIPCHK(hipGraphLaunch(ctx->graph_exec[parity], ctx->stream));
    HIPCHK(hipEventRecord(ev[3], ctx->stream));
    ctx->graph_events.push_back(ev);  // only [0] and [3]: the phases of a replayed step are not separated
    return GGX_OK;
}

// Reads the counters of the last step (pinned copy) once the stream is idle.
int finish(ggx_ctx* ctx) {
    HIPCHK(hipStreamSynchronize(ctx->stream));
    const Sched& H = *ctx->h_sched;
    if (H.any_err) {
        std::vector<int> e((size_t)ctx->nslots);
        HIPCHK(hipMemcpy(e.data(), ctx->errs, ctx->nslots * sizeof(int), hipMemcpyDeviceToHost));
        for (int g = 1; g < ctx->nslots; ++g)
            if (e[g]) {
                char buf[160];
                std::snprintf(buf, sizeof buf, "grain %d: device error %d before loop %d", g, e[g], ctx->loop);
                return fail(ctx, GGX_E_BOUNDS, buf);
            }
    }
    return GGX_OK;
}

// The per-grain baseline: the same kernels, one launch per grain per kernel, with the work
// lists built on the host (the reference's per-LSbox calls).
template <class T>
int launch_step_pergrain(ggx_ctx* ctx) {
    hipStream_t st = ctx->stream;
    const int NS = ctx->nslots;
    T* P = (T*)ctx->P[ctx->cur];
    T* Tt = (T*)ctx->Tt;
    uint32_t* Iold = ctx->I[ctx->icur];
    Sched* S = ctx->sched;
    std::vector<hipEvent_t> ev = take_events(ctx, 5);
    // host view of the live grains and their boxes
    std::vector<int> f((size_t)NS);
    std::vector<Box> bx((size_t)NS);
    HIPCHK(hipMemcpy(f.data(), ctx->flags, NS * sizeof(int), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(bx.data(), ctx->box, NS * sizeof(Box), hipMemcpyDeviceToHost));
    std::vector<int> live;
    for (int g = 1; g < NS; ++g)
        if ((f[g] & kPresent) && (f[g] & kExists)) live.push_back(g);
    // one-element work lists: grain i at pg_list[i], count 1 at pg_one[i]
    const size_t L = live.size();
    std::vector<int> ones(L, 1);
    HIPCHK(hipMemcpy(ctx->pg_list, live.data(), L * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->pg_one, ones.data(), L * 4, hipMemcpyHostToDevice));
    HIPCHK(hipEventRecord(ev[0], st));
    hipLaunchKernelGGL(k_reset, dim3(1), dim3(32), 0, st, S);
    hipLaunchKernelGGL(k_prep, dim3((NS + 255) / 256), dim3(256), 0, st, NS, ctx->flags, ctx->box, bucket_table(ctx),
                       ctx->blists, ctx->alist, ctx->errs, S, (const int*)nullptr);
    for (size_t i = 0; i < L; ++i)
        hipLaunchKernelGGL(k_lists, dim3(1), dim3(64), 0, st, (const int*)(ctx->pg_list + i), (const int*)(ctx->pg_one + i),
                           ctx->box, ctx->flags, ctx->sec_cnt, ctx->sec, ctx->cmp_cnt, ctx->cmp, ctx->errs);
    HIPCHK(hipEventRecord(ev[1], st));
    for (size_t i = 0; i < live.size(); ++i) {
        const int n = bx[live[i]].n;
        int rc = fft_for(ctx, n) && boxes_for<T>(ctx, n)
                     ? launch_conv_boxes(ctx, st, single_item(ctx->pg_list + i, ctx->pg_one + i, n), n, 1, (const double*)P, (double*)Tt)
                 : fft_for(ctx, n) ? launch_conv_fft<T>(ctx, st, ctx->pg_list + i, ctx->pg_one + i, n, 1, (const T*)P, Tt)
                                 : launch_conv<T>(ctx, st, single_item(ctx->pg_list + i, ctx->pg_one + i, n), n, 1, (const T*)P, Tt);
        if (rc) return rc;
    }
    if (ctx->K.on) {
        for (size_t i = 0; i < live.size(); ++i) {
            launch_aniso<T>(ctx, st, ctx->pg_list + i, ctx->pg_one + i, 1, (const T*)P, Tt, Iold);
        }
    }
    HIPCHK(hipEventRecord(ev[2], st));
    LevelArgs<T> A = level_args<T>(ctx);
    A.contour_base = nullptr;  // contour slots from the bump allocator
    for (size_t i = 0; i < live.size(); ++i) {
        A.nb = bx[live[i]].n;
        A.cap = contour_cap(A.nb);
        A.it = single_item(ctx->pg_list + i, ctx->pg_one + i, A.nb);
        int rc = launch_compare<T>(ctx, st, A, 1, false);
        if (!rc) rc = launch_contour<T>(ctx, st, A, 1, false);
        if (rc) return rc;
        hipLaunchKernelGGL(k_alloc, dim3(1), dim3(256), 0, st, (const int*)(ctx->pg_list + i), (const int*)(ctx->pg_one + i),
                           A.O, &S->out_total);
        if ((rc = launch_redist<T>(ctx, st, A, 1))) return rc;
    }
    HIPCHK(hipEventRecord(ev[3], st));
    HIPCHK(hipGetLastError());
    ctx->ev_pending.push_back(ev);
    return GGX_OK;
}

// resizeToSquare of a box on a grid of m points (dimensionalBuffer.h:123-160)
void square_box(int& xmin, int& ymin, int& xmax, int& ymax, int m) {
    const int grid_size = m - 1;
    const unsigned height = (unsigned)(ymax - ymin), width = (unsigned)(xmax - xmin);
    if (width == height) return;
    if (width > height) {
        const int diff = (int)(width - height);
        ymin -= diff / 2;
        ymax += diff / 2 + diff % 2;
    } else {
        const int diff = (int)(height - width);
        xmin -= diff / 2;
        xmax += diff / 2 + diff % 2;
    }
    if (xmin < 0) { const int dl = -xmin; xmax += dl; xmin += dl; }
    else if (xmax > grid_size) { const int dl = grid_size - xmax; xmax += dl; xmin += dl; }
    if (ymin < 0) { const int dl = -ymin; ymax += dl; ymin += dl; }
    else if (ymax > grid_size) { const int dl = grid_size - ymax; ymax += dl; ymin += dl; }
}

// grainhdl::gridCoarsement (grainhdl.cpp:1396-1477) in place of the step's first buffer switch:
// every grain not deleted moved onto a grid of sqrt(present) * NumberOfPointsPerGrain points
// (k_regrid), the grid constants and the circulant tables of the new grid, then the level-set
// kernel's coarsening pass (IDLocal, contour).  Runs between steps, with the stream idle.
template <class T>
int coarsen(ggx_ctx* ctx, int present) {
    hipStream_t st = ctx->stream;
    const int NS = ctx->nslots;
    HIPCHK(hipStreamSynchronize(st));
    if (ctx->fr.copying) {  // a frame copy of the current arenas may still run
        HIPCHK(hipEventSynchronize(ctx->fr.done));
        ctx->fr.copying = false;
    }
    std::vector<int> f((size_t)NS), er((size_t)NS);
    std::vector<Box> bx((size_t)NS);
    std::vector<long long> off((size_t)NS), offp((size_t)NS);
    HIPCHK(hipMemcpy(f.data(), ctx->flags, NS * sizeof(int), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(er.data(), ctx->errs, NS * sizeof(int), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(bx.data(), ctx->box, NS * sizeof(Box), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(off.data(), ctx->off, NS * sizeof(long long), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(offp.data(), ctx->off_prev, NS * sizeof(long long), hipMemcpyDeviceToHost));
    ggx_derived& D = ctx->d;
    const int newSize = (int)(std::sqrt((double)present) * ctx->s.number_of_points_per_grain);
    if (newSize < 1) return fail(ctx, GGX_E_CONFIG, "grid coarsening to an empty grid");
    const double h = D.h, hn = 1.0 / (double)newSize, delta_old = D.delta;
    const int mnew = newSize + 2 * D.grid_blowup;
    // new boxes, packed into the other arena; the old field of a grain that vanished in the last
    // step is its convolved field (the reference redistances existing grains only)
    std::vector<int> list;
    std::vector<Box> nb((size_t)NS);
    std::vector<long long> noff((size_t)NS, 0), soff((size_t)NS, 0);
    std::vector<int> sflag((size_t)NS, 0);
    long long total = 0;
    int nmax = 1;
    for (int g = 1; g < NS; ++g) {
        nb[g] = bx[g];
        if (!(f[g] & kPresent) || er[g]) continue;
        const Box& b = bx[g];
        int x0 = (int)(b.x0 * (h / hn) + 0.5), x1 = (int)((b.x0 + b.n) * (h / hn) + 0.5);
        int y0 = (int)(b.y0 * (h / hn) + 0.5), y1 = (int)((b.y0 + b.n) * (h / hn) + 0.5);
        square_box(x0, y0, x1, y1, mnew);
        if (x1 - x0 != y1 - y0 || x1 - x0 < 1 || x1 - x0 > kMaxBox)
            return fail(ctx, GGX_E_BOUNDS, "grain " + std::to_string(g) + ": no square box on the coarser grid");
        nb[g] = Box{x0, y0, x1 - x0, y1 - y0};
        noff[g] = total;
        total += aligned((long long)nb[g].n * nb[g].n);
        nmax = std::max(nmax, nb[g].n);
        const bool ex = (f[g] & kExists) != 0;
        sflag[g] = ex ? 0 : 1;
        soff[g] = ex ? off[g] : offp[g];
        list.push_back(g);
    }
    if (total > ctx->field_alloc) return fail(ctx, GGX_E_OOM, "field arena too small for the coarser grid");
    const int count = (int)list.size();
    int *d_flag = nullptr;
    long long* d_soff = nullptr;
    int rc;
    if ((rc = dalloc(ctx, d_flag, NS)) || (rc = dalloc(ctx, d_soff, NS))) return rc;
    HIPCHK(hipMemcpy(d_flag, sflag.data(), NS * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_soff, soff.data(), NS * sizeof(long long), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->box_next, nb.data(), NS * sizeof(Box), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->off_next, noff.data(), NS * sizeof(long long), hipMemcpyHostToDevice));
    if (count > 0) HIPCHK(hipMemcpy(ctx->pg_list, list.data(), count * sizeof(int), hipMemcpyHostToDevice));
    T* Pold = (T*)ctx->P[ctx->cur];
    T* Pnew = (T*)ctx->P[ctx->cur ^ 1];
    T* Tt = (T*)ctx->Tt;
    if (count > 0) {
        RegridArgs<T> R;
        R.list = ctx->pg_list; R.count = count; R.box_old = ctx->box; R.src_off = d_soff; R.src_b_flag = d_flag;
        R.src_a = Pold; R.src_b = Tt; R.box_new = ctx->box_next; R.off_new = ctx->off_next; R.dst = Pnew;
        R.h = h; R.hn = hn; R.delta_old = delta_old;
        hipLaunchKernelGGL(k_regrid<T>, dim3(std::min(count, ctx->cu_count * 8)), dim3(256), 0, st, R);
        HIPCHK(hipGetLastError());
        // the comparison of the pass reads an unedited copy of the new fields (the contours edit
        // their own field)
        HIPCHK(hipMemcpyAsync(Tt, Pnew, (size_t)total * sizeof(T), hipMemcpyDeviceToDevice, st));
    }
    HIPCHK(hipStreamSynchronize(st));
    dfree(d_flag);
    dfree(d_soff);
    std::swap(ctx->box, ctx->box_next);
    std::swap(ctx->off, ctx->off_next);
    ctx->cur ^= 1;
    // the constants of the new grid (grainhdl.cpp:1416-1450; m_Energy_deltaMAX is never set, so
    // the dt correction 0.5 / R / 0 / dt is infinite and clamped to 1)
    D.real_domain_size = newSize;
    D.delta = D.grid_blowup * 1 / double(newSize);
    D.ngridpoints = mnew;
    D.h = 1.0 / newSize;
    D.dt = 0.8 / double(newSize * newSize) * ctx->s.number_of_points_per_grain / 2 / 5.0;
    if ((rc = build_kernels(ctx))) return rc;
    // the pass: work lists per bucket of the new boxes, contour slots from the bucket bases
    Sched* S = ctx->sched;
    Sched hs;
    HIPCHK(hipMemcpy(&hs, S, sizeof(Sched), hipMemcpyDeviceToHost));
    std::vector<std::vector<int>> bl((size_t)ctx->nbuckets);
    for (int g : list) {
        int b = 0;
        while (b < ctx->nbuckets - 1 && nb[g].n > ctx->edges[b]) ++b;
        bl[(size_t)b].push_back(g);
    }
    long long cbase = 0;
    for (int b = 0; b < ctx->nbuckets; ++b) {
        hs.bucket_total[b] = (int)bl[(size_t)b].size();
        hs.contour_base[b] = cbase;
        cbase += (long long)bl[(size_t)b].size() * (long long)slot_cap(ctx, b);
        if (!bl[(size_t)b].empty())
            HIPCHK(hipMemcpy(ctx->blists + (size_t)b * NS, bl[(size_t)b].data(), bl[(size_t)b].size() * sizeof(int),
                             hipMemcpyHostToDevice));
    }
    hs.tops[0] = (unsigned long long)total;  // the next step's input layout
    hs.tops[1] = 0ull;
    HIPCHK(hipMemcpy(S, &hs, sizeof(Sched), hipMemcpyHostToDevice));
    // the comparison writes IDLocal, then the contours are traced in (and may edit) the new fields
    LevelArgs<T> A = level_args<T>(ctx);
    A.cmp_cnt = ctx->sec_cnt; A.cmp = ctx->sec;  // the last step's lists
    A.cfield = (T*)ctx->P[ctx->cur];
    if (!list.empty()) {
        level_items(ctx, A, 0, ctx->nbuckets - 1);
        if ((rc = launch_compare<T>(ctx, st, A, (int)list.size(), true))) return rc;
    }
    for (const auto& r : level_groups(ctx)) {
        int k = 0;
        for (int b = r.first; b <= r.second; ++b) k += (int)bl[(size_t)b].size();
        if (k == 0) continue;
        level_items(ctx, A, r.first, r.second);
        if ((rc = launch_contour<T>(ctx, st, A, k, true))) return rc;
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    ctx->icur ^= 1;
    ctx->ngrains = present;
    ctx->coarsenings++;
    return GGX_OK;
}

}  // namespace

extern "C" int ggx_options_default(ggx_options* o) {
    if (!o) return GGX_E_ARG;
    std::memset(o, 0, sizeof(*o));
    o->precision = GGX_PREC_FP64;
    o->batching = GGX_BATCH_FUSED;
    o->conv_engine = GGX_CONV_AUTO;
    o->device = 0;
    o->lds_budget = 0;
    o->use_graph = 0;
    o->persistent = 1;
    o->arena_headroom = 1.5;
    return GGX_OK;
}

extern "C" int ggx_create(const ggx_settings* s, const ggx_options* o, ggx_ctx** out) {
    if (!s || !out) return GGX_E_ARG;
    ggx_ctx* ctx = new ggx_ctx();
    ctx->s = *s;
    if (o) ctx->opt = *o; else ggx_options_default(&ctx->opt);
    int rc = ggx_settings_derive(s, &ctx->d);
    if (rc != GGX_OK) { delete ctx; return rc; }
    if (s->is_isotropic_network == 0) {
        // anisotropic boundaries as the reference computes them for microstructures read from file
        // or generated (MicrostructureGenMode 0/1): cubic lattice, no twin identification,
        // ResearchProject 0 or unset, mobility models 0-2 or the 16-bin model 4 (model 3 reads
        // other grains' volumes while they change), runs that start at loop 0
        const bool ok = s->lattice_type == 0 && s->identify_twins == 0 &&
                        (s->research_project == 0 || s->research_project == 3) &&
                        (s->use_mobility_model == 0 || s->use_mobility_model == 1 || s->use_mobility_model == 2 ||
                         s->use_mobility_model == 4) &&
                        (s->microstructure_gen_mode == 0 || s->microstructure_gen_mode == 1) && s->start_time == 0;
        if (!ok) { delete ctx; return GGX_E_CONFIG; }
        AnisoConst& K = ctx->K;
        K.on = 1;
        K.research_mode = s->research_mode != 0 ? 1 : 0;
        K.mobility_model = s->use_mobility_model;
        K.tpd = s->triple_point_drag;
        K.ds = ctx->d.ds;
        K.csr = s->constant_sector_radius * ctx->d.h;
        K.isr = s->interpolating_sector_radius * ctx->d.h;
        for (int b = 0; b < 16; ++b) K.bins[b] = 1.0;
    }
    if (s->convolution_mode < 0 || s->convolution_mode > 2) { delete ctx; return GGX_E_CONFIG; }
    if (s->decouple_grains || s->use_magnetic_field || s->use_stored_elastic_energy) {
        delete ctx;
        return GGX_E_CONFIG;
    }
    {
        const ggx_options& q = ctx->opt;
        const char* bad = nullptr;
        if (q.precision != GGX_PREC_FP64 && q.precision != GGX_PREC_FP32) bad = "precision";
        else if (q.batching != GGX_BATCH_FUSED && q.batching != GGX_BATCH_PERGRAIN) bad = "batching";
        else if (q.conv_engine != GGX_CONV_AUTO && q.conv_engine != GGX_CONV_CIRCULANT && q.conv_engine != GGX_CONV_FFT)
            bad = "conv_engine";
        else if (q.conv_engine == GGX_CONV_CIRCULANT && s->convolution_mode != 2)
            bad = "the circulant engine convolves the separable Gaussian (ConvolutionMode 2) only";
        else if (q.use_graph != 0 && q.use_graph != 1) bad = "use_graph";
        else if (q.persistent != 0 && q.persistent != 1) bad = "persistent";
        else if (q.use_graph && (!q.persistent || q.batching != GGX_BATCH_FUSED))
            bad = "use_graph needs persistent, batched launches";
        else if (q.use_graph && s->grid_coarsement)
            bad = "grid coarsening changes the grid between steps: no captured step";
        else if (q.lds_budget < 0 || !(q.arena_headroom > 0.0)) bad = "lds_budget / arena_headroom";
        else if (q.bucket_edges[0] != 0) {
            // ascending edges, each in [1, kMaxBox], the last one kMaxBox, then zeros
            int c = 0;
            while (c < 16 && q.bucket_edges[c] != 0) ++c;
            bool ok = c <= kMaxBuckets && q.bucket_edges[c - 1] == kMaxBox;
            for (int b = 0; ok && b < c; ++b)
                ok = q.bucket_edges[b] >= 1 && q.bucket_edges[b] <= kMaxBox && (b == 0 || q.bucket_edges[b] > q.bucket_edges[b - 1]);
            for (int b = c; ok && b < 16; ++b) ok = q.bucket_edges[b] == 0;
            if (!ok) bad = "bucket_edges";
        }
        if (bad) {
            delete ctx;
            return GGX_E_CONFIG;
        }
    }
    ctx->esize = ctx->opt.precision == GGX_PREC_FP32 ? 4 : 8;
    if (ctx->opt.bucket_edges[0] != 0) {
        while (ctx->nbuckets < 16 && ctx->opt.bucket_edges[ctx->nbuckets] != 0) {
            ctx->edges[ctx->nbuckets] = ctx->opt.bucket_edges[ctx->nbuckets];
            ++ctx->nbuckets;
        }
    } else {
        ctx->nbuckets = kDefaultBuckets;
        for (int b = 0; b < kDefaultBuckets; ++b) ctx->edges[b] = kDefaultEdges[b];
    }
    ctx->fft_mask = (unsigned)ctx->opt.fft_buckets;
    ctx->dev = ctx->opt.device;
    hipError_t e = hipSetDevice(ctx->dev);
    if (e != hipSuccess) { delete ctx; return GGX_E_HIP; }
    if (hipStreamCreate(&ctx->stream) != hipSuccess) { delete ctx; return GGX_E_HIP; }
    if (raise_lds(ctx) != GGX_OK) { delete ctx; return GGX_E_HIP; }
    std::memset(&ctx->st, 0, sizeof(ctx->st));
    ctx->loop = s->start_time;
    ctx->ngrains = s->number_of_particles;
    *out = ctx;
    return GGX_OK;
}

extern "C" void ggx_destroy(ggx_ctx* ctx) {
    if (!ctx) return;
    (void)hipDeviceSynchronize();
    for (int k = 0; k < 2; ++k) { dfree(ctx->P[k]); dfree(ctx->I[k]); }
    dfree(ctx->Tt); dfree(ctx->Cf); dfree(ctx->bits); dfree(ctx->gather_part); dfree(ctx->pts);
    dfree(ctx->box); dfree(ctx->box_next); dfree(ctx->off); dfree(ctx->off_next); dfree(ctx->off_prev);
    dfree(ctx->nprev); dfree(ctx->flags); dfree(ctx->errs); dfree(ctx->sec_cnt); dfree(ctx->sec);
    dfree(ctx->cmp_cnt); dfree(ctx->cmp); dfree(ctx->newbox); dfree(ctx->coff); dfree(ctx->ccap); dfree(ctx->clen);
    dfree(ctx->volume); dfree(ctx->perimeter); dfree(ctx->energy); dfree(ctx->meanda); dfree(ctx->nb_cnt);
    dfree(ctx->nb_id); dfree(ctx->nb_len);
    dfree(ctx->quat); dfree(ctx->nb_e); dfree(ctx->nb_m); dfree(ctx->junc); dfree(ctx->jcnt); dfree(ctx->idl_org); dfree(ctx->seg_code); dfree(ctx->seg_arc); dfree(ctx->sectors); dfree(ctx->sched); dfree(ctx->live); dfree(ctx->perm); dfree(ctx->kern_off); dfree(ctx->kern);
    dfree(ctx->tw); dfree(ctx->fft_work);
    dfree(ctx->blists); dfree(ctx->alist); dfree(ctx->pg_list); dfree(ctx->pg_one);
    {
        auto& R = ctx->rec;
        dfree(R.flags); dfree(R.nprev); dfree(R.clen); dfree(R.jcnt); dfree(R.nb_cnt); dfree(R.nb_id); dfree(R.box);
        dfree(R.off); dfree(R.off_prev); dfree(R.coff); dfree(R.idl_org); dfree(R.pts); dfree(R.junc); dfree(R.nb_e);
        dfree(R.nb_m); dfree(R.tilde0); dfree(R.phi0); dfree(R.s); dfree(R.lam_s); dfree(R.lam_u); dfree(R.win); dfree(R.d_area);
        dfree(R.d_perim); dfree(R.grad); dfree(R.area);
    }
    for (auto& ge : ctx->graph_exec)
        if (ge) (void)hipGraphExecDestroy(ge);
    for (auto& v : ctx->graph_events) for (auto e : v) (void)hipEventDestroy(e);
    if (ctx->h_sched) (void)hipHostFree(ctx->h_sched);
    {
        auto& F = ctx->fr;
        if (F.cs) (void)hipStreamSynchronize(F.cs);
        dfree(F.d_small); dfree(F.d_pts);
        if (F.h_small) (void)hipHostFree(F.h_small);
        if (F.h_phi) (void)hipHostFree(F.h_phi);
        if (F.h_idl) (void)hipHostFree(F.h_idl);
        if (F.h_pts) (void)hipHostFree(F.h_pts);
        if (F.staged) (void)hipEventDestroy(F.staged);
        if (F.done) (void)hipEventDestroy(F.done);
        if (F.cs) (void)hipStreamDestroy(F.cs);
    }
    for (auto& v : ctx->ev_pending) for (auto e : v) (void)hipEventDestroy(e);
    for (auto& v : ctx->ev_free) for (auto e : v) (void)hipEventDestroy(e);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

namespace {
thread_local std::string t_last_error = "no error";  // last failure of a context-free call, per thread
int fail_free(int code, const std::string& msg) {
    t_last_error = msg;
    return code;
}
}  // namespace

extern "C" const char* ggx_last_error(const ggx_ctx* ctx) { return ctx ? ctx->err.c_str() : t_last_error.c_str(); }

extern "C" int ggx_load_network(ggx_ctx* ctx, const ggx_network* net) {
    if (!ctx || !net) return GGX_E_ARG;
    if (ctx->loaded) return fail(ctx, GGX_E_STATE, "network already loaded");
    const ggx_derived& D = ctx->d;
    HostGrains HG;
    int rc0 = build_host_grains(*net, D, ctx->s.number_of_particles, HG, ctx->err);
    if (rc0 != GGX_OK) return rc0;
    ctx->max_id = HG.max_id;
    ctx->nslots = HG.nslots;
    const int NS = ctx->nslots;
    ctx->h_quat.assign((size_t)NS * 4, 0.0);
    for (int g = 0; g < NS; ++g) ctx->h_quat[(size_t)g * 4] = 1.0;
    for (size_t i = 0; i < net->ids.size(); ++i)
        for (int k = 0; k < 4; ++k) ctx->h_quat[(size_t)net->ids[i] * 4 + k] = net->q[i][k];
    const std::vector<Box>& hbox = HG.box;
    const std::vector<int>& hflags = HG.flags;
    const std::vector<double>& hvol = HG.volume;
    const std::vector<int>& hclen = HG.clen;
    const std::vector<int>& voff = HG.voff;
    const std::vector<int>& vcnt = HG.vcnt;
    std::vector<double2> verts(HG.verts.size() / 2);
    for (size_t k = 0; k < verts.size(); ++k) verts[k] = make_double2(HG.verts[2 * k], HG.verts[2 * k + 1]);
    // layout
    std::vector<long long> hoff((size_t)NS, 0);
    long long total = 0, ctotal = 0;
    const int nmax = HG.nmax;
    for (int g = 1; g < NS; ++g) {
        if (!(hflags[g] & kPresent)) continue;
        hoff[g] = total;
        total += aligned((long long)hbox[g].n * hbox[g].n);
        ctotal += contour_cap_of(hbox[g].n);
    }
    // arena capacity = headroom x the initial layout (+ 64K elements of slack above 1.0).  Below
    // 1.0 the initial layout still loads, but a step's output cannot fit: the grains that find no
    // room leave the step and GGX_E_BOUNDS is reported (the overflow paths, exercised by tests).
    const double hr = ctx->opt.arena_headroom;
    const long long slack = hr > 1.0 ? 64LL * 1024 : 0;
    ctx->field_cap = (long long)(hr * (double)total) + slack;
    ctx->contour_cap = (long long)(hr * (double)ctotal) + slack;
    // a small network steps its level-set kernel with every grain up to kMergeSide in one launch,
    // each of those taking a contour slot of the merged bucket's size
    ctx->merge_bucket = -1;
    if (ctx->opt.persistent && ctx->opt.batching == GGX_BATCH_FUSED && NS - 1 <= kSmallNetwork)
        for (int b = 0; b < ctx->nbuckets && ctx->edges[b] <= kMergeSide; ++b) ctx->merge_bucket = b;
    if (ctx->merge_bucket >= 0)
        ctx->contour_cap += (long long)NS * contour_cap_of(ctx->edges[ctx->merge_bucket]);
    const long long field_alloc = std::max(ctx->field_cap, total);
    ctx->field_alloc = field_alloc;
    // initial neighbour lists in the reference's R-tree order (find_neighbors)
    std::vector<int> hsec_cnt, hsec;
    if ((rc0 = initial_lists(HG, kCmpCap, hsec_cnt, hsec, ctx->err)) != GGX_OK) return rc0;
    // the initial direct-neighbour list holds the same grains with zero length
    // (LSbox::computeDirectNeighbours -> addDirectNeighbourManual, box.cpp:2220-2237)
    std::vector<int> hnb_cnt((size_t)NS, 0), hnb_id((size_t)NS * kNbCap, 0);
    for (int g = 1; g < NS; ++g) {
        int c = std::min(hsec_cnt[g], kNbCap);
        hnb_cnt[g] = c;
        for (int k = 0; k < c; ++k) hnb_id[(size_t)g * kNbCap + k] = hsec[(size_t)g * kCmpCap + k];
    }

    // device allocations
    size_t es = ctx->esize;
    void* p;
    for (int k = 0; k < 2; ++k) {
        HIPCHK(hipMalloc(&p, (size_t)field_alloc * es)); ctx->P[k] = p;
        HIPCHK(hipMalloc(&p, (size_t)field_alloc * 4)); ctx->I[k] = (uint32_t*)p;
        HIPCHK(hipMemset(ctx->I[k], 0, (size_t)field_alloc * 4));
    }
    HIPCHK(hipMalloc(&p, (size_t)field_alloc * es)); ctx->Tt = p;
    HIPCHK(hipMalloc(&p, (size_t)field_alloc * es)); ctx->Cf = p;
    int rc;
    if ((rc = dalloc(ctx, ctx->bits, (size_t)(kPlanes * plane_words(field_alloc)))) ||
        (rc = dalloc(ctx, ctx->gather_part, (size_t)kCountSlots * kCountStride)))
        return rc;
    HIPCHK(hipMemset(ctx->gather_part, 0, (size_t)kCountSlots * kCountStride * 8));
    if ((rc = dalloc(ctx, ctx->pts, (size_t)std::max(1LL, ctx->contour_cap)))) return rc;
    if ((rc = dalloc(ctx, ctx->box, NS)) || (rc = dalloc(ctx, ctx->box_next, NS)) || (rc = dalloc(ctx, ctx->off, NS)) ||
        (rc = dalloc(ctx, ctx->off_next, NS)) || (rc = dalloc(ctx, ctx->off_prev, NS)) || (rc = dalloc(ctx, ctx->nprev, NS)) ||
        (rc = dalloc(ctx, ctx->flags, NS)) || (rc = dalloc(ctx, ctx->errs, NS)) || (rc = dalloc(ctx, ctx->sec_cnt, NS)) ||
        (rc = dalloc(ctx, ctx->sec, (size_t)NS * kCmpCap)) || (rc = dalloc(ctx, ctx->cmp_cnt, NS)) ||
        (rc = dalloc(ctx, ctx->cmp, (size_t)NS * kCmpCap)) || (rc = dalloc(ctx, ctx->newbox, NS)) ||
        (rc = dalloc(ctx, ctx->coff, NS)) || (rc = dalloc(ctx, ctx->ccap, NS)) || (rc = dalloc(ctx, ctx->clen, NS)) ||
        (rc = dalloc(ctx, ctx->volume, NS)) || (rc = dalloc(ctx, ctx->perimeter, NS)) || (rc = dalloc(ctx, ctx->energy, NS)) ||
        (rc = dalloc(ctx, ctx->meanda, NS)) || (rc = dalloc(ctx, ctx->nb_cnt, NS)) ||
        (rc = dalloc(ctx, ctx->nb_id, (size_t)NS * kNbCap)) || (rc = dalloc(ctx, ctx->nb_len, (size_t)NS * kNbCap)) ||
        (rc = dalloc(ctx, ctx->sched, 1)) || (rc = dalloc(ctx, ctx->live, NS)) ||
        (rc = dalloc(ctx, ctx->blists, (size_t)ctx->nbuckets * NS)) || (rc = dalloc(ctx, ctx->alist, NS)) ||
        (rc = dalloc(ctx, ctx->pg_list, NS)) || (rc = dalloc(ctx, ctx->pg_one, NS)) ||
        (rc = dalloc(ctx, ctx->perm, NS)) || (rc = dalloc(ctx, ctx->kern_off, kMaxBox + 1)))
        return rc;
    {
        // the order in which k_prep files grains into the work lists: Z order (bit-interleaved
        // coordinates) of the initial box centres, so consecutive list items are neighbours on the
        // grid.  Grains move little between steps and coarsening scales all coordinates alike, so
        // the order stays spatial for the run.
        auto spread = [](unsigned long long v) {
            v &= 0xffffffffull;
            v = (v | (v << 16)) & 0x0000ffff0000ffffull;
            v = (v | (v << 8)) & 0x00ff00ff00ff00ffull;
            v = (v | (v << 4)) & 0x0f0f0f0f0f0f0f0full;
            v = (v | (v << 2)) & 0x3333333333333333ull;
            v = (v | (v << 1)) & 0x5555555555555555ull;
            return v;
        };
        std::vector<std::pair<unsigned long long, int>> key;
        key.reserve((size_t)NS);
        for (int g = 1; g < NS; ++g) {
            const unsigned cx = (unsigned)std::max(0, hbox[g].x0 + hbox[g].n / 2);
            const unsigned cy = (unsigned)std::max(0, hbox[g].y0 + hbox[g].n / 2);
            key.push_back({spread(cx) | (spread(cy) << 1), g});
        }
        std::sort(key.begin(), key.end());
        std::vector<int> hperm((size_t)NS, 0);
        for (size_t k = 0; k < key.size(); ++k) hperm[k] = key[k].second;
        HIPCHK(hipMemcpy(ctx->perm, hperm.data(), NS * 4, hipMemcpyHostToDevice));
    }
    {
        // the device counters are initialised in stream order on the context's stream; the pinned
        // host copy is only ever written by device copies and read by the host
        hipLaunchKernelGGL(k_sched_init, dim3(1), dim3(64), 0, ctx->stream, ctx->sched, (unsigned long long)total,
                           ctx->loop);
        HIPCHK(hipGetLastError());
        void* hp = nullptr;
        HIPCHK(hipHostMalloc(&hp, sizeof(Sched), 0));
        ctx->h_sched = (Sched*)hp;
        HIPCHK(hipMemcpyAsync(ctx->h_sched, ctx->sched, sizeof(Sched), hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(hipStreamSynchronize(ctx->stream));
    }
    HIPCHK(hipMalloc(&p, (size_t)kern_offset(kMaxBox + 1) * es + 64)); ctx->kern = p;
    {
        std::vector<long long> ko(kMaxBox + 1);
        for (int n = 0; n <= kMaxBox; ++n) ko[n] = kern_offset(n);
        HIPCHK(hipMemcpy(ctx->kern_off, ko.data(), ko.size() * 8, hipMemcpyHostToDevice));
    }
    if ((rc = build_kernels(ctx))) return rc;
    {
        // what the FFT engine reads, where a launch of this context runs it: twiddles of every side up
        // to kMaxBox (built on the device), and the global half-spectrum slots
        bool engine, slots;
        if (es == 8) fft_needs<double>(ctx, &engine, &slots);
        else fft_needs<float>(ctx, &engine, &slots);
        if (engine) {
            if ((rc = dalloc(ctx, ctx->tw, (size_t)tw_offset(kMaxBox + 1)))) return rc;
            hipLaunchKernelGGL(k_fft_twiddles, dim3(kMaxBox), dim3(256), 0, ctx->stream, ctx->tw, 1, kMaxBox);
            HIPCHK(hipGetLastError());
        }
        if (slots) {
            HIPCHK(hipMalloc(&p, (size_t)kFftWideGrid * (size_t)fft_slot(kMaxBox) * 2 * es + 256));
            ctx->fft_work = p;
        }
    }
    if (nmax > kMaxBox) return fail(ctx, GGX_E_BOUNDS, "box side above the supported maximum");

    std::vector<int> hnprev((size_t)NS);
    for (int g = 0; g < NS; ++g) hnprev[g] = hbox[g].n;
    std::vector<double> zeros((size_t)NS * kNbCap, 0.0);
    std::vector<int> izeros((size_t)NS, 0);
    HIPCHK(hipMemcpy(ctx->box, hbox.data(), NS * sizeof(Box), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->box_next, hbox.data(), NS * sizeof(Box), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->off, hoff.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->off_prev, hoff.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->off_next, hoff.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->nprev, hnprev.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->flags, hflags.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->errs, izeros.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->sec_cnt, hsec_cnt.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->sec, hsec.data(), hsec.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->cmp_cnt, izeros.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->clen, hclen.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->ccap, izeros.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->volume, hvol.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->perimeter, zeros.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->energy, zeros.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->meanda, zeros.data(), NS * 8, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->nb_cnt, hnb_cnt.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->nb_id, hnb_id.data(), hnb_id.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->nb_len, zeros.data(), zeros.size() * 8, hipMemcpyHostToDevice));
    if (ctx->K.on) {
        // the initial direct neighbours are characteristics(neighbour, 0, 0, 0, 0): energy and
        // mobility 0 (grainBoundary.h:68)
        if ((rc = dalloc(ctx, ctx->quat, NS)) || (rc = dalloc(ctx, ctx->nb_e, (size_t)NS * kNbCap)) ||
            (rc = dalloc(ctx, ctx->nb_m, (size_t)NS * kNbCap)) || (rc = dalloc(ctx, ctx->junc, (size_t)NS * kJuncCap)) ||
            (rc = dalloc(ctx, ctx->jcnt, NS)) || (rc = dalloc(ctx, ctx->idl_org, NS)) ||
            (rc = dalloc(ctx, ctx->seg_code, (size_t)std::max(1LL, ctx->contour_cap))) ||
            (rc = dalloc(ctx, ctx->seg_arc, (size_t)std::max(1LL, ctx->contour_cap))) || (rc = dalloc(ctx, ctx->sectors, NS)))
            return rc;
        std::vector<double4> hq((size_t)NS);
        std::vector<int2> horg((size_t)NS);
        for (int g = 0; g < NS; ++g) {
            hq[g] = make_double4(ctx->h_quat[(size_t)g * 4], ctx->h_quat[(size_t)g * 4 + 1], ctx->h_quat[(size_t)g * 4 + 2],
                                 ctx->h_quat[(size_t)g * 4 + 3]);
            horg[g] = make_int2(hbox[g].x0, hbox[g].y0);
        }
        HIPCHK(hipMemcpy(ctx->quat, hq.data(), NS * sizeof(double4), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(ctx->idl_org, horg.data(), NS * sizeof(int2), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(ctx->nb_e, zeros.data(), zeros.size() * 8, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(ctx->nb_m, zeros.data(), zeros.size() * 8, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(ctx->jcnt, izeros.data(), NS * 4, hipMemcpyHostToDevice));
    }

    // initial signed distance (distanceInitialisation, grainhdl.cpp:728-753)
    ctx->h_flags = hflags;
    ctx->h_box = hbox;
    ctx->h_err.assign((size_t)NS, 0);
    build_live(ctx);
    int nlive = (int)ctx->h_live.size();
    int *d_voff = nullptr, *d_vcnt = nullptr;
    double2* d_verts = nullptr;
    if ((rc = dalloc(ctx, d_voff, NS)) || (rc = dalloc(ctx, d_vcnt, NS)) || (rc = dalloc(ctx, d_verts, verts.size())))
        return rc;
    HIPCHK(hipMemcpy(d_voff, voff.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_vcnt, vcnt.data(), NS * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_verts, verts.data(), verts.size() * sizeof(double2), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(ctx->live, ctx->h_live.data(), nlive * 4, hipMemcpyHostToDevice));
    GridConst G = grid_const(ctx);
    if (nlive > 0) {
        if (es == 8)
            hipLaunchKernelGGL(k_init_sdf<double>, dim3(nlive), dim3(256), 0, ctx->stream, ctx->live, ctx->box, ctx->off,
                               d_voff, d_vcnt, d_verts, (double*)ctx->P[ctx->cur], G);
        else
            hipLaunchKernelGGL(k_init_sdf<float>, dim3(nlive), dim3(256), 0, ctx->stream, ctx->live, ctx->box, ctx->off,
                               d_voff, d_vcnt, d_verts, (float*)ctx->P[ctx->cur], G);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    dfree(d_voff); dfree(d_vcnt); dfree(d_verts);
    ctx->loaded = true;
    return GGX_OK;
}

// Steps are queued without waiting for the device; deferred device errors are collected every
// 8 steps and by ggx_sync.
extern "C" int ggx_step(ggx_ctx* ctx, int32_t nsteps) {
    if (!ctx) return GGX_E_ARG;
    if (!ctx->loaded) return fail(ctx, GGX_E_STATE, "ggx_step before ggx_load_network");
    for (int s = 0; s < nsteps; ++s) {
        int rc;
        const bool record = ctx->rec.armed && s == 0;  // the first step after ggx_record_next_step
        ctx->rec.valid = false;                        // a recorded step stays valid until the next one
        if (s > 0 && s % 8 == 0) {
            if ((rc = finish(ctx))) return rc;
        }
        if (ctx->s.grid_coarsement && ctx->loop != 0) {
            // gridCoarsement (grainhdl.cpp:1398-1400): currentNrGrains of the last step against
            // ngrains of the last coarsening
            HIPCHK(hipStreamSynchronize(ctx->stream));
            const int present = ctx->h_sched->present;
            if ((double)present / (double)ctx->ngrains < ctx->s.grid_coarsement_gradient) {
                // the new fields, boxes and IDLocal become the step's input layout
                rc = (ctx->esize == 8) ? coarsen<double>(ctx, present) : coarsen<float>(ctx, present);
                if (rc) return rc;
            }
        }
        if (ctx->fr.copying && ctx->loop >= ctx->fr.loop + 1) {  // this step overwrites the copied arenas
            HIPCHK(hipStreamWaitEvent(ctx->stream, ctx->fr.done, 0));
            ctx->fr.copying = false;
        }
        if (record)
            rc = launch_step<double>(ctx, true, true);
        else if (ctx->opt.batching == GGX_BATCH_PERGRAIN)
            rc = (ctx->esize == 8) ? launch_step_pergrain<double>(ctx) : launch_step_pergrain<float>(ctx);
        else if (ctx->opt.use_graph)
            rc = (ctx->esize == 8) ? launch_step_graph<double>(ctx) : launch_step_graph<float>(ctx);
        else
            rc = (ctx->esize == 8) ? launch_step<double>(ctx, true) : launch_step<float>(ctx, true);
        if (record) {
            ctx->rec.armed = false;
            if (!rc) { ctx->rec.valid = true; ctx->rec.loop = ctx->loop; }
        }
        if (rc) return rc;
        // layout switch: the next arena becomes current, this step's IDLocal the stale source
        std::swap(ctx->box, ctx->box_next);
        std::swap(ctx->off, ctx->off_next);
        std::swap(ctx->sec, ctx->cmp);
        std::swap(ctx->sec_cnt, ctx->cmp_cnt);
        ctx->cur ^= 1;
        ctx->icur ^= 1;
        ctx->loop += 1;
        HIPCHK(hipMemcpyAsync(ctx->h_sched, ctx->sched, sizeof(Sched), hipMemcpyDeviceToHost, ctx->stream));
    }
    return GGX_OK;
}

extern "C" int ggx_sync(ggx_ctx* ctx) {
    if (!ctx) return GGX_E_ARG;
    if (!ctx->loaded) {
        if (ctx->stream) HIPCHK(hipStreamSynchronize(ctx->stream));
        return GGX_OK;
    }
    return finish(ctx);
}

extern "C" int ggx_loop(const ggx_ctx* ctx) { return ctx ? ctx->loop : GGX_E_ARG; }

extern "C" int ggx_get_grid(const ggx_ctx* ctx, ggx_derived* out) {
    if (!ctx || !out) return GGX_E_ARG;
    *out = ctx->d;
    return ctx->coarsenings;
}
extern "C" int ggx_max_id(const ggx_ctx* ctx) { return ctx ? ctx->max_id : GGX_E_ARG; }

extern "C" int ggx_current_grains(ggx_ctx* ctx) {
    if (!ctx || !ctx->loaded) return GGX_E_STATE;
    int rc = finish(ctx);
    if (rc) return rc;
    if (ctx->h_sched->steps_total == 0) {
        int c = 0;
        for (int g = 1; g < ctx->nslots; ++g) c += (ctx->h_flags[g] & kPresent) ? 1 : 0;
        return c;
    }
    return ctx->h_sched->present;
}

namespace {
template <class X>
int fetch(ggx_ctx* ctx, const X* dsrc, X* h, size_t count) {
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(hipMemcpy(h, dsrc, count * sizeof(X), hipMemcpyDeviceToHost));
    return GGX_OK;
}
}  // namespace

extern "C" int ggx_get_info(ggx_ctx* ctx, int32_t id, ggx_grain_info* o) {
    if (!ctx || !o || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    std::memset(o, 0, sizeof(*o));
    int f, e, cl, nbc, cc;
    Box b;
    double v, p, en, md;
    int rc;
    if ((rc = fetch(ctx, ctx->flags + id, &f, 1)) || (rc = fetch(ctx, ctx->errs + id, &e, 1)) ||
        (rc = fetch(ctx, ctx->box + id, &b, 1)) || (rc = fetch(ctx, ctx->clen + id, &cl, 1)) ||
        (rc = fetch(ctx, ctx->nb_cnt + id, &nbc, 1)) || (rc = fetch(ctx, ctx->sec_cnt + id, &cc, 1)) ||
        (rc = fetch(ctx, ctx->volume + id, &v, 1)) || (rc = fetch(ctx, ctx->perimeter + id, &p, 1)) ||
        (rc = fetch(ctx, ctx->energy + id, &en, 1)) || (rc = fetch(ctx, ctx->meanda + id, &md, 1)))
        return rc;
    Box bi;
    if ((rc = fetch(ctx, ctx->box_next + id, &bi, 1))) return rc;  // the box the last step compared on
    o->present = (f & kPresent) != 0;
    o->exists = (f & kExists) != 0;
    o->motion_regular = (f & kRegular) != 0;
    o->intersects_boundary = (f & kBoundary) != 0;
    o->xmin = b.x0; o->xmax = b.x0 + b.n; o->ymin = b.y0; o->ymax = b.y0 + b.n;
    o->id_xmin = bi.x0; o->id_xmax = bi.x0 + bi.n; o->id_ymin = bi.y0; o->id_ymax = bi.y0 + bi.n;
    o->contour_len = cl;
    o->n_neighbours = nbc;
    o->n_compare = cc;
    o->error = e;
    o->volume = v; o->perimeter = p; o->energy = en; o->mean_da = md;
    return GGX_OK;
}

extern "C" int ggx_get_info_all(ggx_ctx* ctx, ggx_grain_info* out, int32_t count) {
    if (!ctx || !out || !ctx->loaded) return GGX_E_ARG;
    int NS = std::min(count, ctx->nslots);
    std::vector<int> f(NS), e(NS), cl(NS), nbc(NS), cc(NS);
    std::vector<Box> b(NS), bi(NS);
    std::vector<double> v(NS), p(NS), en(NS), md(NS);
    int rc;
    if ((rc = fetch(ctx, ctx->flags, f.data(), NS)) || (rc = fetch(ctx, ctx->errs, e.data(), NS)) ||
        (rc = fetch(ctx, ctx->box, b.data(), NS)) || (rc = fetch(ctx, ctx->box_next, bi.data(), NS)) ||
        (rc = fetch(ctx, ctx->clen, cl.data(), NS)) || (rc = fetch(ctx, ctx->nb_cnt, nbc.data(), NS)) ||
        (rc = fetch(ctx, ctx->sec_cnt, cc.data(), NS)) || (rc = fetch(ctx, ctx->volume, v.data(), NS)) ||
        (rc = fetch(ctx, ctx->perimeter, p.data(), NS)) || (rc = fetch(ctx, ctx->energy, en.data(), NS)) ||
        (rc = fetch(ctx, ctx->meanda, md.data(), NS)))
        return rc;
    for (int id = 0; id < NS; ++id) {
        ggx_grain_info& o = out[id];
        std::memset(&o, 0, sizeof(o));
        o.present = (f[id] & kPresent) != 0;
        o.exists = (f[id] & kExists) != 0;
        o.motion_regular = (f[id] & kRegular) != 0;
        o.intersects_boundary = (f[id] & kBoundary) != 0;
        o.xmin = b[id].x0; o.xmax = b[id].x0 + b[id].n; o.ymin = b[id].y0; o.ymax = b[id].y0 + b[id].n;
        o.id_xmin = bi[id].x0; o.id_xmax = bi[id].x0 + bi[id].n; o.id_ymin = bi[id].y0; o.id_ymax = bi[id].y0 + bi[id].n;
        o.contour_len = cl[id];
        o.n_neighbours = nbc[id];
        o.n_compare = cc[id];
        o.error = e[id];
        o.volume = v[id]; o.perimeter = p[id]; o.energy = en[id]; o.mean_da = md[id];
    }
    return NS;
}

extern "C" int ggx_get_phi(ggx_ctx* ctx, int32_t id, double* out, int32_t cap) {
    if (!ctx || !out || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    Box b;
    long long o;
    int rc;
    if ((rc = fetch(ctx, ctx->box + id, &b, 1)) || (rc = fetch(ctx, ctx->off + id, &o, 1))) return rc;
    int cnt = b.n * b.n;
    if (cnt > cap) return GGX_E_ARG;
    if (ctx->esize == 8) {
        if ((rc = fetch(ctx, (const double*)ctx->P[ctx->cur] + o, out, cnt))) return rc;
    } else {
        std::vector<float> tmp(cnt);
        if ((rc = fetch(ctx, (const float*)ctx->P[ctx->cur] + o, tmp.data(), cnt))) return rc;
        for (int k = 0; k < cnt; ++k) out[k] = tmp[k];
    }
    return cnt;
}

extern "C" int ggx_get_idlocal(ggx_ctx* ctx, int32_t id, uint32_t* out, int32_t cap) {
    if (!ctx || !out || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    // IDLocal of the last step lives in I[icur] with the layout of that step (off_prev, box_next)
    Box b;
    long long o;
    int rc;
    if ((rc = fetch(ctx, ctx->box_next + id, &b, 1)) || (rc = fetch(ctx, ctx->off_prev + id, &o, 1))) return rc;
    int cnt = b.n * b.n;
    if (cnt > cap) return GGX_E_ARG;
    if ((rc = fetch(ctx, ctx->I[ctx->icur] + o, out, cnt))) return rc;
    return cnt;
}

extern "C" int ggx_get_contour(ggx_ctx* ctx, int32_t id, double* xy, int32_t cap_points) {
    if (!ctx || !xy || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    int len;
    long long co;
    int rc;
    if ((rc = fetch(ctx, ctx->clen + id, &len, 1)) || (rc = fetch(ctx, ctx->coff + id, &co, 1))) return rc;
    if (len > cap_points) return GGX_E_ARG;
    if ((rc = fetch(ctx, ctx->pts + co, (double2*)xy, len))) return rc;
    return len;
}

extern "C" int ggx_get_neighbours(ggx_ctx* ctx, int32_t id, int32_t* ids, double* lengths, int32_t cap) {
    if (!ctx || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    int c;
    int rc;
    if ((rc = fetch(ctx, ctx->nb_cnt + id, &c, 1))) return rc;
    if (c > cap) return GGX_E_ARG;
    if (ids && (rc = fetch(ctx, ctx->nb_id + (size_t)id * kNbCap, ids, c))) return rc;
    if (lengths && (rc = fetch(ctx, ctx->nb_len + (size_t)id * kNbCap, lengths, c))) return rc;
    return c;
}

extern "C" int ggx_get_neighbour_props(ggx_ctx* ctx, int32_t id, double* energy, double* mobility, int32_t cap) {
    if (!ctx || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    if (!ctx->K.on) return fail(ctx, GGX_E_STATE, "boundary properties are recorded for anisotropic networks only");
    int c;
    int rc;
    if ((rc = fetch(ctx, ctx->nb_cnt + id, &c, 1))) return rc;
    if (c > cap) return GGX_E_ARG;
    if (energy && (rc = fetch(ctx, ctx->nb_e + (size_t)id * kNbCap, energy, c))) return rc;
    if (mobility && (rc = fetch(ctx, ctx->nb_m + (size_t)id * kNbCap, mobility, c))) return rc;
    return c;
}

extern "C" int ggx_get_junctions(ggx_ctx* ctx, int32_t id, int32_t* ints, double* dbls, int32_t cap) {
    if (!ctx || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    if (!ctx->K.on) return fail(ctx, GGX_E_STATE, "junctions are recorded for anisotropic networks only");
    int c;
    int rc;
    if ((rc = fetch(ctx, ctx->jcnt + id, &c, 1))) return rc;
    if (c > cap) return GGX_E_ARG;
    std::vector<Junc> J((size_t)c);
    if (c > 0 && (rc = fetch(ctx, ctx->junc + (size_t)id * kJuncCap, J.data(), (size_t)c))) return rc;
    for (int k = 0; k < c; ++k) {
        if (ints) {
            ints[6 * k] = J[k].order;
            ints[6 * k + 1] = J[k].seg;
            for (int q = 0; q < 4; ++q) ints[6 * k + 2 + q] = (int32_t)J[k].gr[q];
        }
        if (dbls) {
            dbls[3 * k] = J[k].x;
            dbls[3 * k + 1] = J[k].y;
            dbls[3 * k + 2] = J[k].lambda;
        }
    }
    return c;
}

// ------------------------------------------------------------------------------------------
// The adjoint of a recorded step (adjoint.h).
// ------------------------------------------------------------------------------------------
namespace {
int snapshot_for_adjoint(ggx_ctx* ctx, hipStream_t st, const void* P, const uint32_t* Iold) {
    auto& R = ctx->rec;
    const size_t NS = (size_t)ctx->nslots;
    auto cp = [&](void* dst, const void* src, size_t bytes) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, st);
    };
    HIPCHK(cp(R.flags, ctx->flags, NS * 4));
    HIPCHK(cp(R.nprev, ctx->nprev, NS * 4));
    HIPCHK(cp(R.clen, ctx->clen, NS * 4));
    HIPCHK(cp(R.jcnt, ctx->jcnt, NS * 4));
    HIPCHK(cp(R.nb_cnt, ctx->nb_cnt, NS * 4));
    HIPCHK(cp(R.nb_id, ctx->nb_id, NS * kNbCap * 4));
    HIPCHK(cp(R.box, ctx->box, NS * sizeof(Box)));
    HIPCHK(cp(R.off, ctx->off, NS * 8));
    HIPCHK(cp(R.off_prev, ctx->off_prev, NS * 8));
    HIPCHK(cp(R.coff, ctx->coff, NS * 8));
    HIPCHK(cp(R.idl_org, ctx->idl_org, NS * sizeof(int2)));
    HIPCHK(cp(R.pts, ctx->pts, (size_t)std::max(1LL, ctx->contour_cap) * sizeof(double2)));
    HIPCHK(cp(R.junc, ctx->junc, NS * kJuncCap * sizeof(Junc)));
    HIPCHK(cp(R.nb_e, ctx->nb_e, NS * kNbCap * 8));
    HIPCHK(cp(R.nb_m, ctx->nb_m, NS * kNbCap * 8));
    HIPCHK(cp(R.phi0, P, (size_t)ctx->field_alloc * 8));
    R.phi = R.phi0;
    R.idl = Iold;
    return GGX_OK;
}
}  // namespace

extern "C" int ggx_record_next_step(ggx_ctx* ctx) {
    if (!ctx) return GGX_E_ARG;
    if (!ctx->loaded) return fail(ctx, GGX_E_STATE, "ggx_record_next_step before ggx_load_network");
    if (ctx->esize != 8 || !ctx->K.on || ctx->K.mobility_model != 4 || ctx->K.research_mode != 0 ||
        ctx->opt.batching != GGX_BATCH_FUSED || ctx->s.grid_coarsement)
        return fail(ctx, GGX_E_CONFIG, "the adjoint covers FP64 batched steps of anisotropic networks with "
                                       "UseMobilityModel 4, ResearchMode 0 and no grid coarsening");
    auto& R = ctx->rec;
    if (!R.flags) {
        const size_t NS = (size_t)ctx->nslots, F = (size_t)ctx->field_alloc;
        int rc;
        if ((rc = dalloc(ctx, R.flags, NS)) || (rc = dalloc(ctx, R.nprev, NS)) || (rc = dalloc(ctx, R.clen, NS)) ||
            (rc = dalloc(ctx, R.jcnt, NS)) || (rc = dalloc(ctx, R.nb_cnt, NS)) || (rc = dalloc(ctx, R.nb_id, NS * kNbCap)) ||
            (rc = dalloc(ctx, R.box, NS)) || (rc = dalloc(ctx, R.off, NS)) || (rc = dalloc(ctx, R.off_prev, NS)) ||
            (rc = dalloc(ctx, R.coff, NS)) || (rc = dalloc(ctx, R.idl_org, NS)) ||
            (rc = dalloc(ctx, R.pts, (size_t)std::max(1LL, ctx->contour_cap))) ||
            (rc = dalloc(ctx, R.junc, NS * kJuncCap)) || (rc = dalloc(ctx, R.nb_e, NS * kNbCap)) ||
            (rc = dalloc(ctx, R.nb_m, NS * kNbCap)) || (rc = dalloc(ctx, R.tilde0, F)) || (rc = dalloc(ctx, R.s, F)) ||
            (rc = dalloc(ctx, R.phi0, F)) ||
            (rc = dalloc(ctx, R.lam_s, F)) || (rc = dalloc(ctx, R.lam_u, F)) || (rc = dalloc(ctx, R.win, F)) ||
            (rc = dalloc(ctx, R.area, NS)) ||
            (rc = dalloc(ctx, R.d_area, NS)) || (rc = dalloc(ctx, R.d_perim, NS)) || (rc = dalloc(ctx, R.grad, 16)))
            return rc;
    }
    R.armed = true;
    return GGX_OK;
}

extern "C" int ggx_step_adjoint(ggx_ctx* ctx, const double* d_area, const double* d_perimeter, double* grad_bins) {
    if (!ctx || !d_area || !d_perimeter || !grad_bins) return GGX_E_ARG;
    auto& R = ctx->rec;
    if (!R.valid) return fail(ctx, GGX_E_STATE, "no recorded step: ggx_record_next_step, then one ggx_step");
    int rc = finish(ctx);
    if (rc) return rc;
    hipStream_t st = ctx->stream;
    const int NS = ctx->nslots;
    std::vector<double> ha((size_t)NS, 0.0), hp((size_t)NS, 0.0);
    for (int g = 1; g <= ctx->max_id && g < NS; ++g) { ha[g] = d_area[g]; hp[g] = d_perimeter[g]; }
    HIPCHK(hipMemcpyAsync(R.d_area, ha.data(), (size_t)NS * 8, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(R.d_perim, hp.data(), (size_t)NS * 8, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemsetAsync(R.lam_s, 0, (size_t)ctx->field_alloc * 8, st));
    HIPCHK(hipMemsetAsync(R.lam_u, 0, (size_t)ctx->field_alloc * 8, st));
    HIPCHK(hipMemsetAsync(R.grad, 0, 16 * 8, st));
    AdjContourArgs C;
    C.nslots = NS; C.flags_conv = R.flags; C.flags_out = ctx->flags; C.box = R.box; C.off = R.off;
    C.pts = ctx->pts; C.coff = ctx->coff; C.clen = ctx->clen; C.s = R.s; C.win = R.win; C.u = (const double*)ctx->Tt;
    C.d_area = R.d_area; C.d_perim = R.d_perim; C.lam_s = R.lam_s; C.lam_u = R.lam_u; C.area_set = R.area;
    C.h = ctx->d.h; C.band = 0.7 * ctx->d.delta;
    const int grid = std::max(1, std::min(NS, ctx->cu_count * 8));
    hipLaunchKernelGGL(k_adj_contour, dim3(grid), dim3(64), 0, st, C);
    hipLaunchKernelGGL(k_adj_route, dim3(grid), dim3(256), 0, st, C);
    AdjWeightArgs W;
    AnisoArgs<double>& A = W.A;
    A.list = nullptr; A.count = nullptr; A.box = R.box; A.off = R.off; A.phi = R.phi; A.tilde = nullptr;
    A.idl = R.idl; A.off_prev = R.off_prev; A.n_prev = R.nprev; A.flags = R.flags; A.err = nullptr; A.nslots = NS;
    A.pts = R.pts; A.coff = R.coff; A.clen = R.clen; A.nb_cnt = R.nb_cnt; A.nb_id = R.nb_id;
    A.S.quat = ctx->quat; A.S.nb_e = R.nb_e; A.S.nb_m = R.nb_m; A.S.junc = R.junc; A.S.jcnt = R.jcnt;
    A.S.idl_org = R.idl_org; A.K = ctx->K; A.loop = nullptr; A.h = ctx->d.h; A.delta = ctx->d.delta;
    A.seg_code = nullptr; A.seg_arc = nullptr; A.sectors = nullptr;
    W.tilde0 = R.tilde0; W.lam_u = R.lam_u; W.grad = R.grad; W.loop = R.loop;
    hipLaunchKernelGGL(k_adj_weight, dim3(grid), dim3(256), 0, st, W);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(grad_bins, R.grad, 16 * 8, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return GGX_OK;
}

extern "C" int ggx_set_mobility_bins(ggx_ctx* ctx, const double* bins) {
    if (!ctx || !bins) return GGX_E_ARG;
    if (!ctx->K.on || ctx->K.mobility_model != 4)
        return fail(ctx, GGX_E_STATE, "mobility bins belong to anisotropic networks with UseMobilityModel 4");
    for (int b = 0; b < 16; ++b) {
        if (!(bins[b] >= 0.0)) return fail(ctx, GGX_E_ARG, "mobility bins must be non-negative numbers");
        ctx->K.bins[b] = bins[b];
    }
    // captured steps carry the constants in their kernel arguments: capture again
    for (int k = 0; k < 2; ++k) {
        if (ctx->graph_exec[k]) {
            (void)hipStreamSynchronize(ctx->stream);
            (void)hipGraphExecDestroy(ctx->graph_exec[k]);
            ctx->graph_exec[k] = nullptr;
        }
    }
    // the recorded boundary mobilities are those of the new bins from here on
    ctx->rec.valid = false;
    if (ctx->loaded) {
        hipLaunchKernelGGL(k_refresh_mobility, dim3((ctx->nslots + 255) / 256), dim3(256), 0, ctx->stream, ctx->nslots,
                           (const int*)ctx->nb_cnt, (const int*)ctx->nb_id, (const double*)ctx->nb_e, ctx->nb_m,
                           (const double4*)ctx->quat, ctx->K);
        HIPCHK(hipGetLastError());
    }
    return GGX_OK;
}

extern "C" int ggx_get_compare_list(ggx_ctx* ctx, int32_t id, int32_t* ids, int32_t cap) {
    if (!ctx || !ctx->loaded || id < 1 || id >= ctx->nslots) return GGX_E_ARG;
    int c;
    int rc;
    if ((rc = fetch(ctx, ctx->sec_cnt + id, &c, 1))) return rc;
    if (c > cap) return GGX_E_ARG;
    if (ids && (rc = fetch(ctx, ctx->sec + (size_t)id * kCmpCap, ids, c))) return rc;
    return c;
}

namespace {

template <class X>
int grow_pinned(ggx_ctx* ctx, X*& p, size_t& cap, size_t bytes) {
    if (bytes <= cap) return GGX_OK;
    if (p) HIPCHK(hipHostFree((void*)p));
    p = nullptr;
    cap = 0;
    void* q = nullptr;
    size_t want = bytes + bytes / 4 + 4096;
    HIPCHK(hipHostMalloc(&q, want, 0));
    p = (X*)q;
    cap = want;
    return GGX_OK;
}

template <class X>
int grow_device(ggx_ctx* ctx, X*& p, size_t& cap, size_t bytes) {
    if (bytes <= cap) return GGX_OK;
    dfree(p);
    cap = 0;
    size_t want = bytes + bytes / 4 + 4096;
    void* q = nullptr;
    HIPCHK(hipMalloc(&q, want));
    p = (X*)q;
    cap = want;
    return GGX_OK;
}

// The per-grain arrays a frame needs, in staging order: (device pointer, bytes per grain).
struct SmallPart {
    const void* src;
    size_t per;
};

std::vector<SmallPart> small_parts(const ggx_ctx* ctx) {
    return {{ctx->flags, 4}, {ctx->errs, 4}, {ctx->box, sizeof(Box)}, {ctx->box_next, sizeof(Box)},
            {ctx->off, 8}, {ctx->off_prev, 8}, {ctx->coff, 8}, {ctx->clen, 4}, {ctx->volume, 8},
            {ctx->perimeter, 8}, {ctx->energy, 8}, {ctx->meanda, 8}, {ctx->nb_cnt, 4},
            {ctx->nb_id, 4 * (size_t)kNbCap}, {ctx->nb_len, 8 * (size_t)kNbCap}, {ctx->sec_cnt, 4},
            {ctx->sec, 4 * (size_t)kCmpCap}};
}

}  // namespace

extern "C" int ggx_frame_begin(ggx_ctx* ctx) {
    if (!ctx) return GGX_E_ARG;
    if (!ctx->loaded) return fail(ctx, GGX_E_STATE, "ggx_frame_begin before ggx_load_network");
    auto& F = ctx->fr;
    int rc;
    if ((rc = finish(ctx))) return rc;  // the last step is done; its counters are on the host
    if (!F.cs) {
        HIPCHK(hipStreamCreate(&F.cs));
        HIPCHK(hipEventCreateWithFlags(&F.staged, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&F.done, hipEventDisableTiming));
    }
    HIPCHK(hipStreamSynchronize(F.cs));  // the staging buffers of the previous frame are free
    const int NS = ctx->nslots;
    const Sched& H = *ctx->h_sched;
    const bool stepped = H.steps_total > 0;
    // the bump counters keep counting past a full arena (the grains that overflowed left the step)
    F.nfield = std::min((long long)H.tops[0], ctx->field_alloc);
    F.nidl = std::min((long long)H.in_top, ctx->field_alloc);
    F.npts = stepped ? std::min((long long)H.tops[1], ctx->contour_cap) : 0;
    const std::vector<SmallPart> parts = small_parts(ctx);
    auto part_bytes = [&](const SmallPart& q) { return (q.per * (size_t)NS + 7) & ~(size_t)7; };
    size_t small = 0;
    for (const auto& q : parts) small += part_bytes(q);
    F.small_bytes = small;
    if ((rc = grow_device(ctx, F.d_small, F.d_small_cap, small)) ||
        (rc = grow_device(ctx, F.d_pts, F.d_pts_cap, (size_t)F.npts * sizeof(double2))) ||
        (rc = grow_pinned(ctx, F.h_small, F.h_small_cap, small)) ||
        (rc = grow_pinned(ctx, F.h_phi, F.h_phi_cap, (size_t)F.nfield * ctx->esize)) ||
        (rc = grow_pinned(ctx, F.h_idl, F.h_idl_cap, (size_t)F.nidl * 4)) ||
        (rc = grow_pinned(ctx, F.h_pts, F.h_pts_cap, (size_t)F.npts * sizeof(double2))))
        return rc;
    // stage what the next step overwrites, in stream order on the main stream
    size_t o = 0;
    for (const auto& q : parts) {
        HIPCHK(hipMemcpyAsync((char*)F.d_small + o, q.src, q.per * NS, hipMemcpyDeviceToDevice, ctx->stream));
        o += part_bytes(q);
    }
    if (F.npts)
        HIPCHK(hipMemcpyAsync(F.d_pts, ctx->pts, (size_t)F.npts * sizeof(double2), hipMemcpyDeviceToDevice, ctx->stream));
    HIPCHK(hipEventRecord(F.staged, ctx->stream));
    // device -> host on the copy stream; P[cur] and I[icur] stay intact through the next step
    HIPCHK(hipStreamWaitEvent(F.cs, F.staged, 0));
    HIPCHK(hipMemcpyAsync(F.h_small, F.d_small, small, hipMemcpyDeviceToHost, F.cs));
    if (F.npts) HIPCHK(hipMemcpyAsync(F.h_pts, F.d_pts, (size_t)F.npts * sizeof(double2), hipMemcpyDeviceToHost, F.cs));
    if (F.nfield)
        HIPCHK(hipMemcpyAsync(F.h_phi, ctx->P[ctx->cur], (size_t)F.nfield * ctx->esize, hipMemcpyDeviceToHost, F.cs));
    if (F.nidl) HIPCHK(hipMemcpyAsync(F.h_idl, ctx->I[ctx->icur], (size_t)F.nidl * 4, hipMemcpyDeviceToHost, F.cs));
    HIPCHK(hipEventRecord(F.done, F.cs));
    F.copying = true;
    F.valid = true;
    F.loop = ctx->loop;
    return GGX_OK;
}

extern "C" int ggx_frame_get(ggx_ctx* ctx, ggx_frame* out) {
    if (!ctx || !out) return GGX_E_ARG;
    auto& F = ctx->fr;
    if (!F.valid) return fail(ctx, GGX_E_STATE, "ggx_frame_get without ggx_frame_begin");
    HIPCHK(hipEventSynchronize(F.done));
    const int NS = ctx->nslots;
    // the parts of the staged block, each padded to 8 bytes, in small_parts() order
    std::vector<const char*> at;
    {
        const char* b = (const char*)F.h_small;
        for (const auto& q : small_parts(ctx)) {
            at.push_back(b);
            b += (q.per * (size_t)NS + 7) & ~(size_t)7;
        }
    }
    const int* f = (const int*)at[0];
    const int* e = (const int*)at[1];
    const Box* bx = (const Box*)at[2];
    const Box* bi = (const Box*)at[3];
    const long long* off = (const long long*)at[4];
    const long long* offp = (const long long*)at[5];
    const long long* coff = (const long long*)at[6];
    const int* cl = (const int*)at[7];
    const double* v = (const double*)at[8];
    const double* p = (const double*)at[9];
    const double* en = (const double*)at[10];
    const double* md = (const double*)at[11];
    const int* nbc = (const int*)at[12];
    const int* nbid = (const int*)at[13];
    const double* nbl = (const double*)at[14];
    const int* cc = (const int*)at[15];
    const int* cmp = (const int*)at[16];
    F.info.assign((size_t)NS, ggx_grain_info{});
    F.phi_off.assign((size_t)NS, 0);
    F.idl_off.assign((size_t)NS, 0);
    F.contour_off.assign((size_t)NS, 0);
    for (int id = 0; id < NS; ++id) {
        ggx_grain_info& o = F.info[id];
        o.present = (f[id] & kPresent) != 0;
        o.exists = (f[id] & kExists) != 0;
        o.motion_regular = (f[id] & kRegular) != 0;
        o.intersects_boundary = (f[id] & kBoundary) != 0;
        o.xmin = bx[id].x0; o.xmax = bx[id].x0 + bx[id].n; o.ymin = bx[id].y0; o.ymax = bx[id].y0 + bx[id].n;
        o.id_xmin = bi[id].x0; o.id_xmax = bi[id].x0 + bi[id].n; o.id_ymin = bi[id].y0; o.id_ymax = bi[id].y0 + bi[id].n;
        o.contour_len = cl[id];
        o.n_neighbours = nbc[id];
        o.n_compare = cc[id];
        o.error = e[id];
        o.volume = v[id]; o.perimeter = p[id]; o.energy = en[id]; o.mean_da = md[id];
        F.phi_off[id] = off[id];
        F.idl_off[id] = offp[id];
        F.contour_off[id] = coff[id];
    }
    const double* phi;
    if (ctx->esize == 8) {
        phi = (const double*)F.h_phi;
    } else {
        F.phi64.resize((size_t)F.nfield);
        const float* q = (const float*)F.h_phi;
        for (long long k = 0; k < F.nfield; ++k) F.phi64[(size_t)k] = q[k];
        phi = F.phi64.data();
    }
    std::memset(out, 0, sizeof(*out));
    out->nslots = NS;
    out->loop = F.loop;
    out->precision = ctx->esize == 8 ? GGX_PREC_FP64 : GGX_PREC_FP32;
    out->nb_stride = kNbCap;
    out->list_stride = kCmpCap;
    out->real_domain_size = ctx->d.real_domain_size;
    out->field_elems = F.nfield;
    out->idl_elems = F.nidl;
    out->contour_points = F.npts;
    out->info = F.info.data();
    out->phi_off = F.phi_off.data();
    out->phi = phi;
    out->idl_off = F.idl_off.data();
    out->idl = F.h_idl;
    out->contour_off = F.contour_off.data();
    out->contour = (const double*)F.h_pts;
    out->nb_id = nbid;
    out->nb_len = nbl;
    out->cmp = cmp;
    out->quat = ctx->h_quat.data();
    return GGX_OK;
}

extern "C" int ggx_get_stats(ggx_ctx* ctx, ggx_stats* out) {
    if (!ctx || !out) return GGX_E_ARG;
    if (ctx->loaded) {
        int rc = finish(ctx);
        if (rc) return rc;
        for (auto& ev : ctx->ev_pending) {
            float ms[3];
            for (int k = 0; k < 3; ++k) HIPCHK(hipEventElapsedTime(&ms[k], ev[k], ev[k + 1]));
            ctx->st.comparison_ms += ms[0];   // scheduling + comparison lists
            ctx->st.convolution_ms += ms[1];
            ctx->st.levelset_ms += ms[2];     // fused comparison / level set / redistancing
            ctx->st.total_ms += ms[0] + ms[1] + ms[2];
            ctx->st.steps += 1;
            ctx->ev_free.push_back(ev);
        }
        ctx->ev_pending.clear();
        for (auto& ev : ctx->graph_events) {
            float ms;
            HIPCHK(hipEventElapsedTime(&ms, ev[0], ev[3]));
            ctx->st.total_ms += ms;
            ctx->st.steps += 1;
            ctx->ev_free.push_back(ev);
        }
        ctx->graph_events.clear();
        unsigned long long part[kCountSlots * kCountStride], gathered = 0;
        HIPCHK(hipMemcpy(part, ctx->gather_part, sizeof(part), hipMemcpyDeviceToHost));
        for (int k = 0; k < kCountSlots; ++k) gathered += part[k * kCountStride];
        const Sched& H = *ctx->h_sched;
        ctx->st.grid_point_updates = (int64_t)H.updates_total;
        const int64_t S = ctx->esize;
        ctx->st.conv_bytes = 2 * S * (int64_t)H.updates_total;
        // comparison: own phi~ + neighbour gathers; IDLocal written on the box; phi' on the new box
        ctx->st.algorithmic_bytes = ctx->st.conv_bytes + S * (int64_t)(H.updates_total + gathered + H.out_total) +
                                    4 * (int64_t)H.updates_total;
        ctx->st.live_grains = H.all_count;
        ctx->st.max_box = H.max_n;
    }
    *out = ctx->st;
    return GGX_OK;
}

// ------------------------------------------------------------------------------------------
// Standalone batched convolution (the FFT engine without a context).
// ------------------------------------------------------------------------------------------
namespace {

int check_batch_args(int32_t count, const int32_t* n, const int64_t* off, const double* in, const double* out,
                     int32_t max_n, int32_t mode, int32_t R) {
    if (count < 0 || mode < 0 || mode > 2 || R < 1 || max_n < 1) return GGX_E_ARG;
    if (count > 0 && (!n || !off || !in || !out)) return GGX_E_ARG;
    if (max_n > kMaxBox) return GGX_E_BOUNDS;
    return GGX_OK;
}

// The three launches of a batch, queued on st; *bad collects sides outside [1, max_n].
int run_batch(int32_t count, const int32_t* n, const int64_t* off, const double* in, double* out, int32_t max_n,
              const FftSymbol& sy, hipStream_t st, int* bad) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return fail_free(GGX_E_HIP, std::string("ggx_convolve_boxes: device: ") + hipGetErrorString(e));
    const size_t rows = (size_t)box_rows_lds(max_n), columns = (size_t)box_columns_lds(max_n);
    const struct { const void* f; size_t lds, most; } need[] = {
        {(const void*)k_box_rows<BoxBatch>, rows, (size_t)box_rows_lds(kMaxBox)},
        {(const void*)k_box_columns<BoxBatch>, columns, (size_t)box_columns_lds(kMaxBox)}};
    for (const auto& k : need)  // above the default limit: one value for every call, so that threads agree
        if (k.lds > 65536 && hipFuncSetAttribute(k.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.most) != hipSuccess) {
            (void)hipGetLastError();
            return GGX_E_BOUNDS;
        }
    BoxBatch B;
    B.count = count; B.strips = (max_n + 15) / 16;
    B.ns = n; B.offs = off; B.nmax = max_n; B.bad = bad;
    // an odd stride, so that a workgroup's items differ in their strip (50000 boxes of side 4 to 8 with
    // max_n 128: 1.69 ms with cus * 64, 0.78)
    const dim3 grid((unsigned)std::min<long long>((long long)count * B.strips, (long long)cus * 64 - 1)), block(256);
    hipLaunchKernelGGL(k_box_rows<BoxBatch>, grid, block, rows, st, B, in, out, 1);
    hipLaunchKernelGGL(k_box_columns<BoxBatch>, grid, block, columns, st, B, out, sy);
    hipLaunchKernelGGL(k_box_rows<BoxBatch>, grid, block, rows, st, B, (const double*)out, out, 0);
    if (hipGetLastError() != hipSuccess) return GGX_E_HIP;
    return GGX_OK;
}

FftSymbol batch_symbol(int32_t mode, double dt, int32_t R) {
    FftSymbol sy;
    sy.mode = mode;
    sy.dt = dt;
    sy.nsq = (double)R * (double)R;
    return sy;
}

}  // namespace

extern "C" int ggx_convolve_boxes(int32_t count, const int32_t* n, const int64_t* off, const double* in,
                                  double* out, int32_t max_n, int32_t mode, double dt, int32_t R, void* stream) {
    int rc = check_batch_args(count, n, off, in, out, max_n, mode, R);
    if (rc != GGX_OK) return fail_free(rc, "ggx_convolve_boxes: bad arguments");
    if (count == 0) return GGX_OK;
    hipStream_t st = (hipStream_t)stream;
    int* bad = nullptr;
    if (hipMalloc((void**)&bad, sizeof(int)) != hipSuccess) return GGX_E_OOM;
    rc = run_batch(count, n, off, in, out, max_n, batch_symbol(mode, dt, R), st, bad);
    int hbad = 0;
    if (rc == GGX_OK) {
        if (hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            rc = GGX_E_HIP;
    } else {
        (void)hipStreamSynchronize(st);
    }
    (void)hipFree(bad);
    if (rc == GGX_OK && hbad) return fail_free(GGX_E_BOUNDS, "ggx_convolve_boxes: a box side is outside [1, max_n]");
    if (rc != GGX_OK) return fail_free(rc, "ggx_convolve_boxes: device error");
    return rc;
}

// ------------------------------------------------------------------------------------------
// The same batch without any allocation: its bounds flag is the static device word `scratch` (one
// copy per GPU, alive until the process ends).  Host code never passes the word's name to a kernel
// or a copy: it uses the device address taken once per device with hipGetSymbolAddress.  Calls that
// overlap on one GPU share the word and race.
// ------------------------------------------------------------------------------------------
constexpr int kNoAllocMaxN = 256;

static __device__ int scratch;

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up on the first call per device).
int scratch_address(void** out) {
    int dev = 0;
    hipError_t ge = hipGetDevice(&dev);
    if (ge != hipSuccess)
        return fail_free(GGX_E_HIP, std::string("ggx_convolve_boxes_noalloc: hipGetDevice: ") + hipGetErrorString(ge));
    if (dev < 0 || dev >= kMaxDevices) return fail_free(GGX_E_ARG, "ggx_convolve_boxes_noalloc: device ordinal above 63");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail_free(GGX_E_HIP, std::string("ggx_convolve_boxes_noalloc: hipGetSymbolAddress: ") +
                                            hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return GGX_OK;
}

}  // namespace

extern "C" int ggx_convolve_boxes_noalloc(int32_t count, const int32_t* n, const int64_t* off, const double* in,
                                          double* out, int32_t max_n, int32_t mode, double dt, int32_t R,
                                          void* stream) {
    int rc = check_batch_args(count, n, off, in, out, max_n, mode, R);
    if (rc != GGX_OK) return fail_free(rc, "ggx_convolve_boxes_noalloc: bad arguments");
    if (max_n > kNoAllocMaxN)
        return fail_free(GGX_E_BOUNDS, "ggx_convolve_boxes_noalloc: max_n " + std::to_string(max_n) +
                                           " is above the largest side " +
                                           std::to_string(kNoAllocMaxN));
    if (count == 0) return GGX_OK;
    void* base = nullptr;
    if ((rc = scratch_address(&base)) != GGX_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    int* bad = (int*)base;
    rc = run_batch(count, n, off, in, out, max_n, batch_symbol(mode, dt, R), st, bad);
    if (rc != GGX_OK) {
        (void)hipStreamSynchronize(st);
        return fail_free(rc, "ggx_convolve_boxes_noalloc: launch failed");
    }
    int hbad = 0;
    if (hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return fail_free(GGX_E_HIP, "ggx_convolve_boxes_noalloc: device error");
    if (hbad) return fail_free(GGX_E_BOUNDS, "ggx_convolve_boxes_noalloc: a box side is outside [1, max_n]");
    return GGX_OK;
}
