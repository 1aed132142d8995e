// CPU execution of the libggx HIP sources, for tests only.
//
// This header stands in for <hip/hip_runtime.h> when tests/emu/Makefile compiles the product
// sources with g++.  Each workgroup runs its lanes as cooperative fibers (ucontext): a lane
// runs until __syncthreads() or its end, then the next lane runs, so barrier semantics and
// LDS sharing are those of the device.  Workgroups run one after another; LDS is poisoned at
// every launch.  Nothing here is linked into libggx.so.
#pragma once
#include <ucontext.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <tuple>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...)
#define __shared__ static
#define __align__(n) alignas(n)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct alignas(16) double2 { double x, y; };
struct int4 { int x, y, z, w; };
struct int2 { int x, y; };
struct double4 { double x, y, z, w; };
inline double2 make_double2(double a, double b) { return double2{a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return int4{a, b, c, d}; }
inline int2 make_int2(int a, int b) { return int2{a, b}; }
inline double4 make_double4(double a, double b, double c, double d) { return double4{a, b, c, d}; }
struct alignas(8) float2 { float x, y; };
inline float2 make_float2(float a, float b) { return float2{a, b}; }
struct alignas(16) float4 { float x, y, z, w; };
inline float4 make_float4(float a, float b, float c, float d) { return float4{a, b, c, d}; }

inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }
inline long long min(long long a, long long b) { return a < b ? a : b; }
inline long long max(long long a, long long b) { return a > b ? a : b; }

namespace emu {
struct Fiber {
    ucontext_t ctx;
    bool done;
};
inline ucontext_t g_main;
inline std::vector<Fiber> g_fibers;
inline std::vector<char*> g_stacks;
inline int g_cur = 0;
inline dim3 g_tid, g_bid, g_bdim, g_gdim;
inline std::function<void()>* g_body = nullptr;
inline unsigned char* g_dyn = nullptr;
inline size_t g_lds_most = 0;  // largest dynamic LDS of any launch so far
inline unsigned long long g_die_barriers[8];  // workgroup barriers passed so far, by workgroup mod 8 (its die)
constexpr size_t kStack = 256 * 1024;

// Barriers: a workgroup barrier waits until every live lane of the block has arrived; a wave
// barrier (used by the cross-lane operations) until every lane of the caller's 64-lane wave has.
inline unsigned g_nt = 0, g_done = 0;
inline unsigned g_bar_count = 0, g_bar_gen = 0;
inline unsigned g_wave_count[16], g_wave_gen[16];
inline unsigned long long g_wave_val[16][64];
inline void yield() { swapcontext(&g_fibers[g_cur].ctx, &g_main); }
inline void entry() {
    (*g_body)();
    g_fibers[g_cur].done = true;
    g_done++;
    if (g_bar_count > 0 && g_bar_count == g_nt - g_done) { g_bar_count = 0; g_bar_gen++; }
    swapcontext(&g_fibers[g_cur].ctx, &g_main);
}
inline void sync() {
    unsigned gen = g_bar_gen;
    if (++g_bar_count == g_nt - g_done) { g_bar_count = 0; g_bar_gen++; }
    while (g_bar_gen == gen) yield();
}
inline void wave_sync() {
    unsigned w = (unsigned)g_cur / 64u, lanes = std::min(64u, g_nt - 64u * w);
    unsigned gen = g_wave_gen[w];
    if (++g_wave_count[w] == lanes) { g_wave_count[w] = 0; g_wave_gen[w]++; }
    while (g_wave_gen[w] == gen) yield();
}
inline unsigned long long wave_exchange(unsigned long long v, int src, bool ballot) {
    unsigned w = (unsigned)g_cur / 64u, lanes = std::min(64u, g_nt - 64u * w);
    g_wave_val[w][g_cur % 64] = v;
    wave_sync();
    unsigned long long r = 0;
    if (ballot) {
        for (unsigned l = 0; l < lanes; ++l)
            if (g_wave_val[w][l]) r |= 1ull << l;
    } else {
        r = g_wave_val[w][src & 63];
    }
    wave_sync();
    return r;
}

// Frees the fiber stacks and the LDS stand-in at exit (no leak reports from the sanitizer).
struct Cleanup {
    ~Cleanup() {
        for (char* p : g_stacks) std::free(p);
        g_stacks.clear();
        std::free(g_dyn);
        g_dyn = nullptr;
    }
};
inline Cleanup g_cleanup;

// Stream capture: while a stream captures, launches are recorded (arguments already bound) and
// run when the instantiated graph is launched.
inline bool g_capturing = false;
inline std::vector<std::function<void()>>* g_capture = nullptr;

inline void run_launch(dim3 grid, dim3 block, size_t shmem, std::function<void()> body);
inline void launch(dim3 grid, dim3 block, size_t shmem, std::function<void()> body) {
    if (g_capturing) {
        g_capture->push_back([=]() { run_launch(grid, block, shmem, body); });
        return;
    }
    run_launch(grid, block, shmem, body);
}

inline void run_launch(dim3 grid, dim3 block, size_t shmem, std::function<void()> body) {
    unsigned nt = block.x * block.y * block.z;
    g_lds_most = std::max(g_lds_most, shmem);
    if (std::getenv("EMU_TRACE")) std::fprintf(stderr, "[emu] launch grid %u block %u lds %zu\n", grid.x, nt, shmem);
    while (g_stacks.size() < nt) g_stacks.push_back((char*)std::malloc(kStack));
    g_fibers.assign(nt, Fiber{});
    g_nt = nt;
    g_body = &body;
    g_gdim = grid;
    g_bdim = block;
    for (unsigned b = 0; b < grid.x; ++b) {
        g_bid = dim3(b, 0, 0);
        std::free(g_dyn);
        g_dyn = (unsigned char*)std::malloc(shmem ? shmem : 1);
        std::memset(g_dyn, 0xCD, shmem ? shmem : 1);
        g_done = 0;
        g_bar_count = 0;
        const unsigned gen = g_bar_gen;
        for (unsigned w = 0; w < 16; ++w) g_wave_count[w] = 0;
        for (unsigned t = 0; t < nt; ++t) {
            getcontext(&g_fibers[t].ctx);
            g_fibers[t].ctx.uc_stack.ss_sp = g_stacks[t];
            g_fibers[t].ctx.uc_stack.ss_size = kStack;
            g_fibers[t].ctx.uc_link = &g_main;
            g_fibers[t].done = false;
            makecontext(&g_fibers[t].ctx, (void (*)())entry, 0);
        }
        bool any = true;
        while (any) {
            any = false;
            for (unsigned t = 0; t < nt; ++t) {
                if (g_fibers[t].done) continue;
                g_cur = (int)t;
                g_tid = dim3(t, 0, 0);
                swapcontext(&g_main, &g_fibers[t].ctx);
                if (!g_fibers[t].done) any = true;
            }
        }
        g_die_barriers[b & 7u] += g_bar_gen - gen;
    }
    g_body = nullptr;
}
}  // namespace emu

inline void __builtin_amdgcn_wave_barrier() { emu::wave_sync(); }
inline void __builtin_amdgcn_fence(int, const char*) {}  // fibers see each other's writes at once
inline double cospi(double x) { return (double)std::cos(3.14159265358979323846264338327950288L * (long double)x); }
inline void sincospi(double x, double* s, double* c) {
    const long double a = 3.14159265358979323846264338327950288L * (long double)x;
    *s = (double)std::sin(a);
    *c = (double)std::cos(a);
}
inline int __builtin_amdgcn_readfirstlane(int v) { return (int)emu::wave_exchange((unsigned)v, 0, false); }
inline int __builtin_amdgcn_readlane(int v, int src) { return (int)emu::wave_exchange((unsigned)v, src, false); }
inline unsigned long long __ballot(int p) { return emu::wave_exchange(p ? 1ull : 0ull, 0, true); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __popc(unsigned v) { return __builtin_popcount(v); }
inline long long __double_as_longlong(double d) { long long r; std::memcpy(&r, &d, 8); return r; }
inline double __longlong_as_double(long long v) { double r; std::memcpy(&r, &v, 8); return r; }
inline int __shfl_up(int v, unsigned d) {
    const int lane = emu::g_cur % 64;
    return (int)emu::wave_exchange((unsigned)v, lane >= (int)d ? lane - (int)d : lane, false);
}
inline double __shfl_xor(double v, int mask) {
    return __longlong_as_double((long long)emu::wave_exchange((unsigned long long)__double_as_longlong(v),
                                                             (emu::g_cur % 64) ^ mask, false));
}
inline int __float_as_int(float f) { int r; std::memcpy(&r, &f, 4); return r; }
inline float __int_as_float(int v) { float r; std::memcpy(&r, &v, 4); return r; }
inline float __shfl_xor(float v, int mask) { return (float)__shfl_xor((double)v, mask); }
// Matrix products of a wave: 16 x 16 results, four fused multiply-adds in ascending order each.
// Operands a: row lane % 16, term lane / 16; b: column lane % 16, term lane / 16.
namespace emu {
// Two buffers in turn: a lane fills a buffer again only after every lane has met the barrier of the
// product between, so one barrier per product is enough.
inline double g_ma[2][16][64], g_mb[2][16][64];
inline unsigned g_mturn[16][64];
template <class V, class X, class Row>
inline V mfma(X a, X b, V c, Row row) {
    const unsigned w = (unsigned)g_cur / 64u, l = (unsigned)g_cur % 64u, t = g_mturn[w][l]++ & 1u;
    g_ma[t][w][l] = a;
    g_mb[t][w][l] = b;
    wave_sync();
    for (int r = 0; r < 4; ++r) {
        X s = c[r];
        for (int k = 0; k < 4; ++k)
            s = std::fma((X)g_ma[t][w][row((int)(l / 16), r) + 16 * k], (X)g_mb[t][w][l % 16 + 16 * k], s);
        c[r] = s;
    }
    return c;
}
typedef double v4d __attribute__((vector_size(32)));
typedef float v4f __attribute__((vector_size(16)));
}  // namespace emu
inline emu::v4d __builtin_amdgcn_mfma_f64_16x16x4f64(double a, double b, emu::v4d c, int, int, int) {
    return emu::mfma(a, b, c, [](int q, int r) { return q + 4 * r; });
}
inline emu::v4f __builtin_amdgcn_mfma_f32_16x16x4f32(float a, float b, emu::v4f c, int, int, int) {
    return emu::mfma(a, b, c, [](int q, int r) { return 4 * q + r; });
}

#define threadIdx (emu::g_tid)
#define blockIdx (emu::g_bid)
#define blockDim (emu::g_bdim)
#define gridDim (emu::g_gdim)
#define HIP_DYNAMIC_SHARED(type, var) type* var = (type*)emu::g_dyn;
inline void __syncthreads() { emu::sync(); }
inline void __threadfence() {}
inline void __threadfence_block() {}
inline int __ffs(unsigned int v) { return __builtin_ffs((int)v); }
inline unsigned long long atomicAdd(unsigned long long* p, unsigned long long v) { auto o = *p; *p += v; return o; }
inline int atomicAdd(int* p, int v) { int o = *p; *p += v; return o; }
inline double atomicAdd(double* p, double v) { double o = *p; *p += v; return o; }
inline unsigned atomicAdd(unsigned* p, unsigned v) { unsigned o = *p; *p += v; return o; }
inline int atomicMin(int* p, int v) { int o = *p; if (v < o) *p = v; return o; }
inline int atomicMax(int* p, int v) { int o = *p; if (v > o) *p = v; return o; }
inline int atomicOr(int* p, int v) { int o = *p; *p |= v; return o; }
inline int atomicCAS(int* p, int cmp, int v) { int o = *p; if (o == cmp) *p = v; return o; }
inline unsigned atomicAnd(unsigned* p, unsigned v) { unsigned o = *p; *p &= v; return o; }
inline unsigned long long atomicExch(unsigned long long* p, unsigned long long v) { auto o = *p; *p = v; return o; }
#define __HIP_MEMORY_SCOPE_AGENT 3
template <class X>
inline X __hip_atomic_load(const X* p, int, int) { return *p; }

#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) \
    emu::launch(grid, block, shmem, [args_ = std::make_tuple(__VA_ARGS__)]() { std::apply(kernel, args_); })

typedef int hipError_t;
typedef int hipStream_t_;
typedef hipStream_t_* hipStream_t;
typedef double* hipEvent_t;
constexpr hipError_t hipSuccess = 0;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyHostToHost };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize };
struct hipDeviceProp_t {
    int multiProcessorCount;
    size_t sharedMemPerBlock;
    size_t maxSharedMemoryPerMultiProcessor;
};
inline const char* hipGetErrorString(hipError_t) { return "emu error"; }
// device and pinned allocations come back filled with a junk pattern (as reused device memory
// does), so a read of memory no kernel or copy has written shows up as a difference
inline size_t g_device_bytes = 0;  // allocated by hipMalloc so far
inline hipError_t hipMalloc(void** p, size_t n) {
    g_device_bytes += n;
    *p = std::malloc(n ? n : 1);
    if (*p) std::memset(*p, 0xA5, n ? n : 1);
    return *p ? 0 : 2;
}
inline hipError_t hipFree(void* p) { std::free(p); return 0; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n ? n : 1);
    if (*p) std::memset(*p, 0x5A, n ? n : 1);
    return *p ? 0 : 2;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return 0; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memmove(d, s, n); return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memmove(d, s, n); return 0; }
inline hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return 0; }
inline hipError_t hipSetDevice(int) { return 0; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return 0; }
#define HIP_SYMBOL(x) (&(x))
enum { hipDeviceAttributeMultiprocessorCount = 1 };
inline hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 4; return 0; }
inline hipError_t hipGetSymbolAddress(void** p, const void* sym) { *p = const_cast<void*>(sym); return 0; }
inline hipError_t hipStreamCreate(hipStream_t* s) { *s = new int(0); return 0; }
inline hipError_t hipStreamDestroy(hipStream_t s) { delete s; return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipDeviceSynchronize() { return 0; }
inline hipError_t hipEventCreate(hipEvent_t* e) { *e = new double(0); return 0; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return 0; }
constexpr unsigned hipEventDisableTiming = 2;
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new double(0); return 0; }
inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
typedef std::vector<std::function<void()>>* hipGraph_t;
typedef std::vector<std::function<void()>>* hipGraphExec_t;
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    emu::g_capture = new std::vector<std::function<void()>>();
    emu::g_capturing = true;
    return 0;
}
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    emu::g_capturing = false;
    *g = emu::g_capture;
    emu::g_capture = nullptr;
    return 0;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t) {
    *e = new std::vector<std::function<void()>>(*g);
    return 0;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (auto& f : *e) f();
    return 0;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return 0; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete e; return 0; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    *e = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
    return 0;
}
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { *ms = (float)(*b - *a); return 0; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    p->multiProcessorCount = 4;
    p->sharedMemPerBlock = 65536;
    p->maxSharedMemoryPerMultiProcessor = 163840;
    return 0;
}
inline hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return 0; }
inline hipError_t hipGetLastError() { return 0; }
struct hipFuncAttributes {
    size_t sharedSizeBytes;
};
inline hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { a->sharedSizeBytes = 0; return 0; }
