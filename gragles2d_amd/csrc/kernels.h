// kernels.h -- CDNA4 (gfx950) kernels of the per-grain level-set timestep.
//
// Every kernel is batched: a launch covers all live grains of a step (one workgroup per
// grain unless stated otherwise); the per-grain launch mode of the baseline issues the same
// kernels with a one-grain work list.  Boxes live in device arenas addressed by per-grain
// offsets; T is the field type (double for the FP64 path, float for the FP32 path).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "ggx_internal.h"

namespace ggx {

struct GridConst {
    int m;        // ngridpoints
    int gb;       // grid_blowup
    int R;        // realDomainSize
    int nslots;   // max grain id + 1 (grains.size())
    double h, delta, dt;
};

// Contour points reserved per grain of box side n: a convex grain's contour has about pi * n
// points; longer contours are reported as GGX_E_BOUNDS instead of being truncated.
__host__ __device__ inline int contour_cap(int n) { return 8 * n + 64; }

template <class T>
__device__ __forceinline__ int sgn_of(T v) {  // utilities.h:27-30
    return (T(0) < v) - (v < T(0));
}

// Flat index of DimensionalBuffer::getValueAt (dimensionalBuffer.h:68-73): 32-bit unsigned
// arithmetic, checked against the element count only.  Returns -1 when the reference would
// throw std::out_of_range.
__device__ __forceinline__ long long flat_index(int row, int col, int x0, int y0, int w, long long size) {
    uint32_t k = (uint32_t)row - (uint32_t)y0;
    k *= (uint32_t)w;
    k += (uint32_t)col - (uint32_t)x0;
    return ((long long)k < size) ? (long long)k : -1;
}

// Orders the wave's LDS writes before its following reads (the other waves are not waited for).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------------------------------------
// Per-step scheduling, all on the device so that a step needs no host round trip.
// Sched holds the counters of one step; k_reset clears them, k_prep deletes the grains that
// vanished in the previous step (grainhdl::level_set, grainhdl.cpp:840-843), counts the
// survivors (get_biggestGrainVol, 1744-1754) and files every live grain into the work list
// of its box-size bucket.
// ------------------------------------------------------------------------------------------
constexpr int kMaxBuckets = 16;
// Networks up to this many grain ids are launch-latency bound (a launch lasts about as long as its
// slowest grain): the scheduling runs in one workgroup, and the circulant convolution, contour and
// redistancing as one launch for every grain up to kMergeSide, the larger buckets keeping their own.
// Set below the break-even: a lognormal network takes 0.61 ms per step with 4000 grains and, launched
// per bucket, 0.83 with 4200.
constexpr int kSmallNetwork = 4096;
constexpr int kMergeSide = 64;

struct Sched {
    int bucket_count[kMaxBuckets];   // live grains per bucket (advanced by k_prep's atomics)
    int bucket_total[kMaxBuckets];   // the same, written by k_tally for the later kernels
    long long contour_base[kMaxBuckets];  // first contour point of each bucket's slots (k_tally)
    int all_count;                   // live grains (advanced by k_prep's atomics)
    int all_total;                   // the same, written by k_tally
    int present;                     // grains not deleted (currentNrGrains)
    int max_n;                       // largest box side this step
    int any_err;
    int loop_cur;                    // loop index of the running step (set by k_reset)
    int loop_next;                   // loop index of the next step
    unsigned long long updates;      // sum of n^2 over live grains, this step
    unsigned long long tops[2];      // bump allocators: field arena, contour arena
    unsigned long long in_top;       // field-arena elements used by the step's input layout
    unsigned long long updates_total;  // sum of n^2 over all steps (never reset)
    unsigned long long steps_total;
    unsigned long long out_total;      // sum over steps and grains of the redistanced box areas
};

struct Buckets {
    int count;
    int edge[kMaxBuckets];           // bucket b holds edge[b-1] < n <= edge[b]
    int cap[kMaxBuckets];            // contour points of a slot of bucket b
};

// Counters of a freshly loaded network: everything zero except the field-arena layout of the
// initial boxes (the input layout of the first step).
__global__ void k_sched_init(Sched* __restrict__ S, unsigned long long initial_top, int start_loop) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        unsigned char* b = (unsigned char*)S;
        for (unsigned k = 0; k < sizeof(Sched); ++k) b[k] = 0;
        S->tops[0] = initial_top;
        S->in_top = initial_top;
        S->loop_next = start_loop;
    }
}

// A counter that other workgroups of earlier kernels advanced with device-scope atomics is read
// with an atomic load: a plain load may be served by a cache line of this XCD's L2 that those
// atomics never touched.
__device__ __forceinline__ int load_counter(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_reset(Sched* __restrict__ S) {
    int t = threadIdx.x;
    if (t < kMaxBuckets) S->bucket_count[t] = 0;
    if (t == 0) {
        S->all_count = 0; S->present = 0; S->max_n = 0; S->any_err = 0;
        // the previous step's output layout is this step's input; its bump counters were advanced
        // by atomics, so they are taken (and cleared) by atomics too
        S->in_top = atomicExch(&S->tops[0], 0ull);
        (void)atomicExch(&S->tops[1], 0ull);
        S->loop_cur = S->loop_next;
        S->loop_next = S->loop_next + 1;
        S->updates = 0ull;
    }
}

// After k_prep: the bucket sizes k_prep's atomics produced, read once with atomic loads and
// written with plain stores for the kernels that follow (every workgroup of those reads them),
// and each bucket's first contour slot: bucket b's grains take consecutive slots of
// cap[b] points after the lower buckets' slots (no per-grain allocation).
__global__ void k_tally(Sched* __restrict__ S, Buckets B) {
    const int t = threadIdx.x;
    if (t < kMaxBuckets) S->bucket_total[t] = t < B.count ? load_counter(&S->bucket_count[t]) : 0;
    if (t == 0) {
        S->all_total = load_counter(&S->all_count);
        long long base = 0;
        for (int b = 0; b < B.count; ++b) {
            S->contour_base[b] = base;
            base += (long long)load_counter(&S->bucket_count[b]) * (long long)B.cap[b];
        }
        S->tops[1] = (unsigned long long)base;
    }
}

// The flags of grain g at the start of a step: deletion of a grain that vanished in the last one.  A
// grain that carries an error (or a box above the largest bucket) is taken out of the step: its
// existence flag is cleared, so no list, gather or launch touches its slots again, and it is deleted
// at the next step like a vanished grain; the host reports the error.
__device__ __forceinline__ int schedule_flags(int g, int* flags, const Box* box, int* err, const Buckets& B, bool* bad) {
    int f = flags[g];
    if (f & kGone) { f &= ~kGone; flags[g] = f; }
    if ((f & kPresent) && !(f & kExists)) { f = (f & ~kPresent) | kGone; flags[g] = f; }
    if ((f & kPresent) && (f & kExists) && !err[g] && box[g].n > B.edge[B.count - 1]) err[g] = kErrBoxCap;
    *bad = err[g] != 0;
    if (*bad && (f & kExists)) { f &= ~kExists; flags[g] = f; }
    return f;
}

// perm: the grain ids in a spatial order (the work lists come out in that order), or null.
__global__ void __launch_bounds__(256) k_prep(int nslots, int* __restrict__ flags, const Box* __restrict__ box,
                                              Buckets B, int* __restrict__ blists, int* __restrict__ alist,
                                              int* __restrict__ err, Sched* __restrict__ S, const int* __restrict__ perm) {
    // per-workgroup histogram, then one reservation per bucket per workgroup
    __shared__ int s_cnt[kMaxBuckets], s_base[kMaxBuckets];
    __shared__ int s_all, s_allbase, s_present, s_err, s_maxn;
    __shared__ unsigned long long s_upd;
    const int t = threadIdx.x;
    if (t < kMaxBuckets) s_cnt[t] = 0;
    if (t == 0) { s_all = 0; s_present = 0; s_err = 0; s_maxn = 0; s_upd = 0ull; }
    __syncthreads();
    const int idx = blockIdx.x * blockDim.x + t;
    const int g = perm ? (idx < nslots - 1 ? perm[idx] : 0) : idx;
    int bk = -1, lpos = -1, apos = -1, n = 0;
    if (g > 0 && g < nslots) {
        bool bad;
        const int f = schedule_flags(g, flags, box, err, B, &bad);
        if (bad) s_err = 1;
        if (f & kPresent) {
            atomicAdd(&s_present, 1);
            if (f & kExists) {
                n = box[g].n;
                bk = 0;
                while (n > B.edge[bk]) bk++;
                lpos = atomicAdd(&s_cnt[bk], 1);
                apos = atomicAdd(&s_all, 1);
                atomicMax(&s_maxn, n);
                atomicAdd(&s_upd, (unsigned long long)n * (unsigned long long)n);
            }
        }
    }
    __syncthreads();
    if (t < B.count && s_cnt[t] > 0) s_base[t] = atomicAdd(&S->bucket_count[t], s_cnt[t]);
    if (t == 0) {
        if (blockIdx.x == 0) S->steps_total += 1ull;
        s_allbase = s_all ? atomicAdd(&S->all_count, s_all) : 0;
        if (s_present) atomicAdd(&S->present, s_present);
        if (s_err) atomicOr(&S->any_err, 1);
        if (s_maxn) atomicMax(&S->max_n, s_maxn);
        if (s_upd) { atomicAdd(&S->updates, s_upd); atomicAdd(&S->updates_total, s_upd); }
    }
    __syncthreads();
    if (bk >= 0) {
        blists[(size_t)bk * nslots + s_base[bk] + lpos] = g;
        alist[s_allbase + apos] = g;
    }
}

// A wave-uniform read of data no lane of this kernel writes (lists, boxes, offsets): through the
// scalar cache into scalar registers, so that the chain list -> box -> field costs a scalar load's
// latency per link and no lane waits for a broadcast.
template <class X>
__device__ __forceinline__ X sload(const X* p) {
    return *(const __attribute__((address_space(4))) X*)p;
}
__device__ __forceinline__ Box sload_box(const Box* p) { return Box{sload(&p->x0), sload(&p->y0), sload(&p->n), 0}; }

// Work items of a launch: the grains of buckets b0 .. b1, bucket after bucket.
struct Items {
    const int* lists;        // work list of bucket b at lists + b * stride
    const int* total;        // grains per bucket (device)
    int stride, b0, b1;
    int cap[kMaxBuckets];    // contour points a grain of each bucket has room for
};

__device__ __forceinline__ int items_total(const Items& it) {
    int n = 0;
    for (int b = it.b0; b <= it.b1; ++b) n += sload(it.total + b);
    return n;
}

// Grain of item `item`, with its bucket and its position in the bucket's list.
__device__ __forceinline__ int item_grain(const Items& it, int item, int* bucket, int* pos) {
    int b = it.b0;
    while (b < it.b1) {
        const int t = sload(it.total + b);
        if (item < t) break;
        item -= t;
        ++b;
    }
    *bucket = b;
    *pos = item;
    return sload(it.lists + (size_t)b * it.stride + item);
}

// k_reset, k_prep and k_tally in one workgroup, for small networks: three dependent launches take
// 15 us there, one takes 5 us.
__global__ void __launch_bounds__(1024) k_schedule(int nslots, int* __restrict__ flags, const Box* __restrict__ box,
                                                   Buckets B, int* __restrict__ blists, int* __restrict__ alist,
                                                   int* __restrict__ err, Sched* __restrict__ S, const int* __restrict__ perm) {
    __shared__ int s_cnt[kMaxBuckets];
    __shared__ int s_all, s_present, s_err, s_maxn;
    __shared__ unsigned long long s_upd;
    const int t = (int)threadIdx.x;
    if (t < kMaxBuckets) s_cnt[t] = 0;
    if (t == 0) { s_all = 0; s_present = 0; s_err = 0; s_maxn = 0; s_upd = 0ull; }
    __syncthreads();
    int present = 0, maxn = 0;
    double upd = 0.0;  // sums of n^2 are exact
    for (int i = t; i < nslots - 1; i += (int)blockDim.x) {
        const int g = perm[i];
        if (g <= 0 || g >= nslots) continue;
        bool bad;
        const int f = schedule_flags(g, flags, box, err, B, &bad);
        if (bad) s_err = 1;
        if (!(f & kPresent)) continue;
        present++;
        if (!(f & kExists)) continue;
        const int n = box[g].n;
        int bk = 0;
        while (n > B.edge[bk]) bk++;
        blists[(size_t)bk * nslots + atomicAdd(&s_cnt[bk], 1)] = g;
        alist[atomicAdd(&s_all, 1)] = g;
        maxn = max(maxn, n);
        upd += (double)n * n;
    }
    double p = present, m = maxn;
    for (int d = 32; d >= 1; d >>= 1) {
        p += __shfl_xor(p, d);
        m = fmax(m, __shfl_xor(m, d));
        upd += __shfl_xor(upd, d);
    }
    if ((t & 63) == 0) {
        atomicAdd(&s_present, (int)p);
        atomicMax(&s_maxn, (int)m);
        atomicAdd(&s_upd, (unsigned long long)upd);
    }
    __syncthreads();
    if (t < kMaxBuckets) {
        S->bucket_count[t] = s_cnt[t];
        S->bucket_total[t] = t < B.count ? s_cnt[t] : 0;
    }
    if (t == 0) {
        S->all_count = s_all; S->all_total = s_all; S->present = s_present; S->max_n = s_maxn; S->any_err = s_err;
        // the previous step's output layout is this step's input; k_alloc's atomics advanced its counter
        S->in_top = atomicExch(&S->tops[0], 0ull);
        S->loop_cur = S->loop_next;
        S->loop_next = S->loop_next + 1;
        S->updates = s_upd;
        S->updates_total += s_upd;
        S->steps_total += 1ull;
        long long base = 0;
        for (int b = 0; b < B.count; ++b) {
            S->contour_base[b] = base;
            base += (long long)s_cnt[b] * (long long)B.cap[b];
        }
        (void)atomicExch(&S->tops[1], (unsigned long long)base);
    }
}

// Block-wide exclusive scan of one int per lane; returns the exclusive prefix, *total gets the sum.
// Shuffles within each wave, one exchange of wave totals through LDS (s_tmp: one int per wave).
__device__ __forceinline__ int block_scan(int v, int* s_tmp, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) s_tmp[wave] = x;
    __syncthreads();
    int base = 0, tot = 0;
    for (int w = 0; w < nw; ++w) {
        const int c = s_tmp[w];
        if (w < wave) base += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return base + x - v;
}

// ------------------------------------------------------------------------------------------
// Comparison lists, LSbox::computeSecondOrderNeighbours (box.cpp:1027-1068).  cmp = the existing
// entries of the previous list, then every existing neighbour-of-neighbour whose input box
// intersects (closed intervals, checkIntersection, box.cpp:881-888), first occurrence only,
// excluding self and the boundary grain.
//
// One wave per grain.  Bound by latency: list -> its entries' lists -> their flags and boxes, three
// dependent reads, so the wave takes 256 candidates at a time (four reads in flight per lane) and
// meets no workgroup barrier.  The first-occurrence test is an LDS hash (grain id -> smallest
// candidate index): the candidates of a pass are entered together, and a candidate whose index the
// table then holds is a first occurrence, since the later passes' indices are larger.  A 256-lane
// workgroup per grain, pulled from a cursor with two passes over the candidates, took 1.10 ms for
// 100k grains and 60 to 70 us for 100; this takes 0.21 ms and 10 us.
// ------------------------------------------------------------------------------------------
constexpr int kHash = 512;       // LDS hash slots (grain id -> smallest candidate index)
constexpr int kHashFill = 320;   // distinct keys allowed per grain (> 2 kCmpCap: beyond it the list overflows anyway)
static_assert(kHashFill > 2 * kCmpCap && kHashFill + 64 < kHash, "hash capacity");

// Open-addressing insert (key-CAS): returns the slot holding `key`, or -1 when the table holds
// kHashFill keys already (the caller reports an error; probing stays bounded: the lanes that pass
// the test together enter at most one key each).
__device__ __forceinline__ int hash_insert(int* h_key, int* fill, int key) {
    unsigned hs = ((unsigned)key * 2654435761u) >> 23;
    for (int probe = 0; probe < kHash; ++probe) {
        const int cur = h_key[hs];
        if (cur == key) return (int)hs;
        if (cur == -1) {
            if (*fill >= kHashFill) return -1;
            const int old = atomicCAS(&h_key[hs], -1, key);
            if (old == -1) { atomicAdd(fill, 1); return (int)hs; }
            if (old == key) return (int)hs;
        }
        hs = (hs + 1) & (kHash - 1);
    }
    return -1;
}

__global__ void __launch_bounds__(64) k_lists(const int* __restrict__ list, const int* __restrict__ count,
                                              const Box* __restrict__ box, const int* __restrict__ flags,
                                              const int* __restrict__ sec_cnt, const int* __restrict__ sec,
                                              int* __restrict__ cmp_cnt, int* __restrict__ cmp, int* __restrict__ err) {
    __shared__ int h_key[kHash], h_min[kHash];
    __shared__ int s_sec[kCmpCap], s_off[kCmpCap + 1];
    __shared__ int s_fill;
    constexpr int kU = 4;  // candidates per lane and pass
    const int lane = (int)threadIdx.x;
    const unsigned long long below = (1ull << lane) - 1ull;
    const int total = sload(count);
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        wave_lds_sync();  // the previous grain's shared state is free
        const int g = sload(list + item);
        const Box bg = sload_box(box + g);
        const int ns = sload(sec_cnt + g);
        int* out = cmp + (size_t)g * kCmpCap;
        for (int k = lane; k < kHash; k += 64) { h_key[k] = -1; h_min[k] = 0x7fffffff; }
        if (lane == 0) s_fill = 0;
        wave_lds_sync();
        // part 1: existing entries of the previous list, in order (box.cpp:1038-1041), and the offset of
        // each entry's candidates
        int written = 0, ntot = 0;
        bool bad = false;
        for (int e0 = 0; e0 < ns; e0 += 64) {
            const int e = e0 + lane;
            int nb = 0, len = 0;
            bool ex = false;
            if (e < ns) {
                nb = sec[(size_t)g * kCmpCap + e];
                ex = (flags[nb] & kExists) != 0;
                len = sec_cnt[nb];
                s_sec[e] = nb;
            }
            int x = len;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int y = __shfl_up(x, d);
                if (lane >= d) x += y;
            }
            if (e < ns) s_off[e] = ntot + x - len;
            ntot += __builtin_amdgcn_readlane(x, 63);
            const unsigned long long m = __ballot(ex);
            if (ex) {
                out[written + __popcll(m & below)] = nb;
                const int hs = hash_insert(h_key, &s_fill, nb);
                if (hs >= 0) h_min[hs] = -1;  // already in the list
                else bad = true;
            }
            written += __popcll(m);
        }
        if (lane == 0) s_off[ns] = ntot;
        wave_lds_sync();
        // candidates in (entry, entry's entry) order (box.cpp:1042-1048)
        for (int c0 = 0; c0 < ntot; c0 += 64 * kU) {
            int c[kU], hs[kU], f[kU];
            Box bc[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int q = c0 + 64 * u + lane;
                c[u] = -1;
                if (q < ntot) {
                    int lo = 0, hi = ns;  // the entry a with s_off[a] <= q < s_off[a + 1]
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (s_off[mid] <= q) lo = mid;
                        else hi = mid;
                    }
                    c[u] = sec[(size_t)s_sec[lo] * kCmpCap + (q - s_off[lo])];
                }
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                f[u] = 0;
                bc[u] = Box{0, 0, 0, 0};
                if (c[u] > 0 && c[u] != g) { f[u] = flags[c[u]]; bc[u] = box[c[u]]; }
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const bool valid = (f[u] & kExists) && !(bg.x0 > bc[u].x0 + bc[u].n || bg.x0 + bg.n < bc[u].x0 ||
                                                         bg.y0 > bc[u].y0 + bc[u].n || bg.y0 + bg.n < bc[u].y0);
                hs[u] = -1;
                if (valid) {
                    hs[u] = hash_insert(h_key, &s_fill, c[u]);
                    if (hs[u] >= 0) atomicMin(&h_min[hs[u]], c0 + 64 * u + lane);  // stays -1 for part-1 entries
                    else bad = true;
                }
            }
            wave_lds_sync();
            // ordered compaction of first occurrences (box.cpp:1050-1066)
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const bool keep = hs[u] >= 0 && h_min[hs[u]] == c0 + 64 * u + lane;
                const unsigned long long m = __ballot(keep);
                const int at = written + __popcll(m & below);
                if (keep && at < kCmpCap) out[at] = c[u];
                written += __popcll(m);
            }
        }
        const bool over = __ballot(bad) != 0ull || written > kCmpCap;
        if (lane == 0) {
            if (over) err[g] = kErrCmpCap;
            cmp_cnt[g] = min(written, kCmpCap);
        }
    }
}

// ------------------------------------------------------------------------------------------
// Circulant tables: the table of box side n holds K_n[(t - kKPad) mod n] for
// t in [0, 2n + 2 kKPad), so that every index a tile needs is in range without a modulo (a step's
// padding reaches three taps beyond the box).
constexpr int kKPad = 8;
__host__ __device__ inline long long ktab_len(int n) { return 2LL * n + 2 * kKPad; }

// Convolution as an exact dense circulant (LSbox::convolutionGeneratorFFTW, box.cpp:622-695,
// Gaussian mode).  The Gaussian symbol G(i,j) = g(i) g(j) is separable and even, so
// IDFT(G . DFT(phi)) = K_n phi K_n with the symmetric circulant
// K_n[m] = sum_k g(k) cos(2 pi k m / n) computed on the host per box size with all n taps
// (the symbol is cut at Nyquist, so K_n has a slowly decaying tail and cannot be banded).
//
// Two contractions, so they run on the matrix cores: 16 x 16 x 4 products, whose sums are the
// ascending chain of fused multiply-adds a scalar loop over the taps makes, bit for bit (FP64 and
// FP32).  Rows first, B = phi K for all n rows of 16 columns, then columns, D = K B.  An FP64
// product's result lies in the registers as the next product's operand does (row lane / 16 + 4 r of
// the tile in register r, operand row lane / 16 of step r), so B need not leave them; an FP32 one
// holds rows 4 (lane / 16) + r and is turned through LDS.  The operands come from LDS, where the
// field lies zero-padded to whole tiles at a pitch that spreads a product's 16 rows over all banks
// (read from global memory instead, a product's 16 row pieces take as long as the product), and the
// coefficients of a step are 19 consecutive table entries.  Both kernels ask for two waves per SIMD or
// more: within 256 registers the compiler keeps the accumulators in vector registers, else it moves
// them to and from accumulation registers around every product (three times the time).  The strips of
// sides above 256 hold too many for that in FP64: 496 bytes per lane lie in scratch there.
//
// On the 100k-grain network in FP64 (4 n flops and 16 bytes per point: floor 0.6 ms, the products at
// the 77 TFLOP/s the matrix cores reach) this takes 1.2 ms per step, where register-blocked VALU
// products with both tiles in LDS took 1.85 ms (five output blocks on four waves, 40 of 64 lanes
// active).  Boxes of 70 to 300 points among 200 fine grains, most of whose tiles did not fit LDS before,
// go from 1.7 to 0.1 ms.  What is left is the latency of reading and writing each box.
// ------------------------------------------------------------------------------------------
template <class T> struct Mma;
template <> struct Mma<double> {
    typedef double V __attribute__((vector_size(32)));
    static __device__ __forceinline__ V run(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int r) { return q + 4 * r; }  // of register r, lanes 16 q ..
};
template <> struct Mma<float> {
    typedef float V __attribute__((vector_size(16)));
    static __device__ __forceinline__ V run(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int r) { return 4 * q + r; }
};

// Smallest pitch >= w at which lanes (row lane % 16, column lane / 16) meet every LDS bank once:
// 2 mod 4 doubles, 4 mod 8 floats.
template <class T>
__host__ __device__ inline int tile_pitch(int w) {
    constexpr int m = sizeof(T) == 8 ? 4 : 8;
    return w + (m / 2 - w % m + m) % m;
}

template <class T>
__host__ __device__ inline long long conv_tiles_lds(int tiles) {
    const int side = 16 * tiles;
    // an FP32 wave turns its tiles through 16 x 17 floats
    return ((long long)side * tile_pitch<T>(side) + ktab_len(side) + (sizeof(T) == 4 ? tiles * 16 * 17 : 0)) * (long long)sizeof(T);
}

// Boxes up to side 16 NT: a workgroup of NT waves per box, a wave per 16 columns, B in registers.  All
// NT row tiles are multiplied, those beyond the box as zeros: a test per product costs more.
template <class T, int NT>
__global__ void __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(NT == 2 ? 5 : NT == 3 ? 4 : 3))) k_conv_tiles(Items it, const Box* __restrict__ box,
                                                        const long long* __restrict__ off, const T* __restrict__ src,
                                                        T* __restrict__ dst, const long long* __restrict__ kern_off,
                                                        const T* __restrict__ kern) {
    using V = typename Mma<T>::V;
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    const int tid = (int)threadIdx.x, lane = tid & 63, j = lane & 15, q = lane >> 4;
    const int xt = __builtin_amdgcn_readfirstlane(tid >> 6);
    T* field = (T*)smem;
    const int total = items_total(it);
    // The next box is read while this one's products run: wave xt carries rows xt, xt + NT, .. (lane =
    // column), thread tid the table's entry tid; its list entry was read one box earlier still.
    T carry[16], coef;
    int next_n = 0, next_g = 0;
    long long next_o = 0;
    auto grain_of = [&](int i) {
        int bucket, pos;
        return i < total ? item_grain(it, i, &bucket, &pos) : 0;
    };
    auto fetch = [&](int g) {
        next_n = sload(&box[g].n);
        next_o = sload(off + g);
        const T* s = src + next_o;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int y = xt + NT * u;
            carry[u] = y < next_n && lane < next_n ? s[y * next_n + lane] : T(0);
        }
        const T* kg = kern + sload(kern_off + next_n);
        coef = tid < (int)ktab_len(next_n) ? kg[tid] : T(0);
    };
    if ((int)blockIdx.x < total) fetch(grain_of((int)blockIdx.x));
    next_g = grain_of((int)blockIdx.x + (int)gridDim.x);
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        const int n = next_n;
        const long long o = next_o;
        const int nt = (n + 15) >> 4, pairs = (n + 7) >> 3, pitch = tile_pitch<T>(8 * pairs);
        T* table = field + 16 * NT * pitch;
        __syncthreads();  // the previous box's LDS is free
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int y = xt + NT * u;
            if (lane < 8 * pairs) field[y * pitch + lane] = carry[u];
        }
        if (tid < (int)ktab_len(n)) table[tid] = coef;
        __syncthreads();
        if (item + (int)gridDim.x < total) {
            fetch(next_g);
            next_g = grain_of(item + 2 * (int)gridDim.x);
        }
        if (xt >= nt) continue;
        const T* kt = table + n + kKPad;         // K_n[m] at m, -n - kKPad <= m < n + kKPad
        const int x = min(16 * xt + j, n - 1);  // columns beyond the box repeat the last one
        V acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] = T(0);
        // rows: B[y][x] = sum_k phi[y][k] K[x - k], two steps at a time
        for (int p = 0; p < pairs; ++p) {
            T v[2][NT], kb[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int k = 8 * p + 4 * u + q;
                kb[u] = kt[x - k];
#pragma unroll
                for (int t = 0; t < NT; ++t) v[u][t] = field[(16 * t + j) * pitch + k];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = Mma<T>::run(v[u][t], kb[u], acc[t]);
        }
        if constexpr (sizeof(T) == 4) {  // register r of lanes 16 q ..: row 4 q + r -> row q + 4 r
            T* turn = table + ktab_len(n) + xt * 16 * 17;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) turn[(4 * q + r) * 17 + j] = acc[t][r];
                wave_lds_sync();
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][r] = turn[(q + 4 * r) * 17 + j];
                wave_lds_sync();
            }
        }
        // columns: D[y][x] = sum_i K[y - i] B[i][x]; the rows of B beyond the box are zero, and the rows
        // of D beyond it (clamped coefficients) are not stored
        V out[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[t][r] = T(0);
#pragma unroll
        for (int p = 0; p < 2 * NT; ++p) {
            if (p < pairs) {
                T k[2][NT];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int t = 0; t < NT; ++t) k[u][t] = kt[min(16 * t + j, n - 1) - (8 * p + 4 * u + q)];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int t = 0; t < NT; ++t) out[t] = Mma<T>::run(k[u][t], acc[p >> 1][2 * (p & 1) + u], out[t]);
            }
        }
        T* d = dst + o;
        if (16 * xt + j < n) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int y = 16 * t + Mma<T>::row(q, r);
                    if (y < n) d[y * n + 16 * xt + j] = out[t][r];
                }
        }
    }
}

// Larger boxes, up to side 64 TU: four waves share 16 columns, each takes every fourth 16-row tile;
// B in LDS, the field through LDS 16 columns at a time (the next 16 on their way meanwhile).  Takes a
// box of any side n at about 160 n bytes of LDS, so where the lds_budget is too small for the tiles of
// a smaller box it is convolved here, with the same bits.
constexpr int kStripCols = 16;

template <class T>
__host__ __device__ inline long long conv_strip_lds(int nb) {
    const int rows = (nb + 15) & ~15;
    return ((long long)rows * tile_pitch<T>(kStripCols) + ktab_len(nb)) * (long long)sizeof(T);
}

// Calls f with the tile count as a constant: 1 .. N.
template <int N, class F>
__device__ __forceinline__ void by_tiles(int count, F f) {
    if constexpr (N > 0) {
        if (count == N) f(std::integral_constant<int, N>());
        else by_tiles<N - 1>(count, f);
    }
}

template <class T, int TU>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_conv_strip(Items it, int blocks, const Box* __restrict__ box,
                                                    const long long* __restrict__ off, const T* __restrict__ src,
                                                    T* __restrict__ dst, const long long* __restrict__ kern_off,
                                                    const T* __restrict__ kern) {
    using V = typename Mma<T>::V;
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    constexpr int kU = TU >= 8 ? 1 : 2;  // steps whose operands are read together
    const int pitch = tile_pitch<T>(kStripCols);
    const int total = items_total(it);
    int item = (int)(blockIdx.x / (unsigned)blocks), xt = (int)(blockIdx.x % (unsigned)blocks);
    const int item_step = (int)(gridDim.x / (unsigned)blocks), xt_step = (int)(gridDim.x % (unsigned)blocks);
    for (; item < total; item += item_step, xt += xt_step) {
        if (xt >= blocks) {
            xt -= blocks;
            if (++item >= total) break;
        }
        int bucket, pos;
        const int g = item_grain(it, item, &bucket, &pos);
        const int n = sload(&box[g].n);
        const int nt = (n + 15) >> 4;
        if (xt >= nt) continue;
        const long long o = sload(off + g);
        const T* s = src + o;
        T* chunk = (T*)smem;                      // the field's columns k0 .. k0 + 15, all rows
        T* strip = chunk;                         // then B: row i, 16 columns (no chunk is read any more)
        T* table = chunk + 16 * nt * pitch;
        const T* kg = kern + sload(kern_off + n);
        const T* kt = table + n + kKPad;
        const int x = min(16 * xt + j, n - 1), low = -n - kKPad;  // the table's first tap: for the zeros beyond the box
        // thread tid carries column tid % 16 of rows tid / 16 + 16 u
        const int cx = tid & 15, cy = tid >> 4;
        T carry[4 * TU];
        auto fetch = [&](int k0) {
#pragma unroll
            for (int u = 0; u < 4 * TU; ++u) {
                const int y = cy + 16 * u;
                carry[u] = u < nt && y < n && k0 + cx < n ? s[y * n + k0 + cx] : T(0);
            }
        };
        fetch(0);
        __syncthreads();  // the previous strip is free
        for (int t = tid; t < (int)ktab_len(n); t += 256) table[t] = kg[t];
        V acc[TU];
#pragma unroll
        for (int u = 0; u < TU; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[u][r] = T(0);
        // the products of this wave's U tiles (the count fixed at compile time: a test per product costs
        // more than the product)
        const int mine = (nt - wave + 3) >> 2;
        auto rows_of = [&](auto tiles, int k0) {
            constexpr int U = decltype(tiles)::value;
#pragma unroll
            for (int p0 = 0; p0 < 4; p0 += kU) {
                T v[kU][U], kb[kU];
#pragma unroll
                for (int p = 0; p < kU; ++p) {
                    const int k = 4 * (p0 + p) + q;
                    kb[p] = kt[max(x - (k0 + k), low)];
#pragma unroll
                    for (int u = 0; u < U; ++u) v[p][u] = chunk[(16 * (wave + 4 * u) + j) * pitch + k];
                }
#pragma unroll
                for (int p = 0; p < kU; ++p)
#pragma unroll
                    for (int u = 0; u < U; ++u) acc[u] = Mma<T>::run(v[p][u], kb[p], acc[u]);
            }
        };
        auto columns_of = [&](auto tiles) {
            constexpr int U = decltype(tiles)::value;
            for (int p0 = 0; p0 < 4 * nt; p0 += kU) {
                T v[kU], k[kU][U];
#pragma unroll
                for (int p = 0; p < kU; ++p) {
                    const int i = 4 * (p0 + p) + q;
                    v[p] = strip[i * 16 + j];
#pragma unroll
                    for (int u = 0; u < U; ++u) k[p][u] = kt[max(min(16 * (wave + 4 * u) + j, n - 1) - i, low)];
                }
#pragma unroll
                for (int p = 0; p < kU; ++p)
#pragma unroll
                    for (int u = 0; u < U; ++u) acc[u] = Mma<T>::run(k[p][u], v[p], acc[u]);
            }
        };
        auto rows = [&](int k0) { by_tiles<TU>(mine, [&](auto tiles) { rows_of(tiles, k0); }); };
        auto columns = [&]() { by_tiles<TU>(mine, [&](auto tiles) { columns_of(tiles); }); };
        for (int k0 = 0; k0 < n; k0 += kStripCols) {
#pragma unroll
            for (int u = 0; u < 4 * TU; ++u)
                if (u < nt) chunk[(cy + 16 * u) * pitch + cx] = carry[u];
            __syncthreads();
            if (k0 + kStripCols < n) fetch(k0 + kStripCols);
            rows(k0);
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < TU; ++u)
            if (wave + 4 * u < nt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    strip[(16 * (wave + 4 * u) + Mma<T>::row(q, r)) * 16 + j] = acc[u][r];
                    acc[u][r] = T(0);
                }
            }
        __syncthreads();
        columns();
        T* d = dst + o;
        if (16 * xt + j < n) {
#pragma unroll
            for (int u = 0; u < TU; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int y = 16 * (wave + 4 * u) + Mma<T>::row(q, r);
                    if (y < n) d[y * n + 16 * xt + j] = acc[u][r];
                }
        }
    }
}

// ------------------------------------------------------------------------------------------
// Contour, volume, motion check, new box and direct neighbours:
// LSbox::extractContour (box.cpp:1089-1153) with MarchingSquaresAlgorithm::generateContour
// (marchingSquares.cpp:28-188), isMotionRegular (box.cpp:1155-1190), clearContourGrainArea
// (1883-1904), then computeVolumeAndEnergy (1201-1228) -> buildDirectNeighbours
// (grainBoundary.cpp:85-199).  What k_contour and k_alloc (level.h) leave per grain, and the cases and
// directions of the marching squares.
// ------------------------------------------------------------------------------------------
struct ContourOut {
    double2* pts;             // contour arena
    long long* coff;          // per grain: offset into pts
    int* ccap;                // per grain: capacity reserved this step
    int* clen;                // per grain: contour length (in: old, out: new)
    double* volume;
    double* perimeter;
    double* energy;
    double* meanda;
    int* nb_cnt;
    int* nb_id;
    double* nb_len;
    Box* box_next;
    long long* off_next;
    int* flags;
    int* err;
    unsigned long long* tops;  // [0] field arena top (elements), [1] contour arena top
    long long field_cap;
    long long contour_cap;
};

enum { MS_TL = 1, MS_TR = 2, MS_BL = 4, MS_BR = 8 };
enum { D_UP = 0, D_DOWN = 1, D_LEFT = 2, D_RIGHT = 3, D_NONE = 4 };

// ------------------------------------------------------------------------------------------
// Initial signed distance, LSbox::calculateDistanceFunction (box.cpp:342-401): crossing-number
// point-in-polygon and the minimum point-segment distance, clamped to delta.  One workgroup
// per grain, one lane per pixel.  Contraction is off so the values match a scalar CPU build.
// ------------------------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(256) k_init_sdf(const int* __restrict__ live, const Box* __restrict__ box,
                                                  const long long* __restrict__ off, const int* __restrict__ voff,
                                                  const int* __restrict__ vcnt, const double2* __restrict__ verts,
                                                  T* __restrict__ field, GridConst G) {
#pragma clang fp contract(off)
    int g = live[blockIdx.x];
    Box b = box[g];
    int n = b.n;
    const double2* cg = verts + voff[g];
    int cs = vcnt[g];
    T* o = field + off[g];
    double h = G.h;
    int gb = G.gb;
    for (int p = threadIdx.x; p < n * n; p += blockDim.x) {
        int yy = p / n, xx = p - yy * n;
        int i = b.y0 + yy, j = b.x0 + xx;
        double tx = (j - gb) * h, ty = (i - gb) * h;
        bool inside = false;
        for (int k = 1, l = 0; k < cs; k++) {
            double2 L = cg[l], K = cg[k];
            if (((L.y > ty) != (K.y > ty)) && (tx < (K.x - L.x) * (ty - L.y) / (K.y - L.y) + L.x)) inside = !inside;
            l = k;
        }
        double minDist = 1000000.0;
        for (int k = 1, l = 0; k < cs; k++) {
            double2 L = cg[l], K = cg[k];
            double ux = K.x - L.x, uy = K.y - L.y;
            double lambda = (tx - L.x) * ux + (ty - L.y) * uy;
            lambda /= ux * ux + uy * uy;
            double dist;
            if (lambda <= 0) {
                double dx = tx - L.x, dy = ty - L.y;
                dist = sqrt(dx * dx + dy * dy);
            } else if (lambda >= 1) {
                double dx = K.x - tx, dy = K.y - ty;
                dist = sqrt(dx * dx + dy * dy);
            } else {
                double px = L.x + ux * lambda, py = L.y + uy * lambda;
                double dx = tx - px, dy = ty - py;
                dist = sqrt(dx * dx + dy * dy);
            }
            minDist = (dist < minDist) ? dist : minDist;
            l = k;
        }
        if (minDist > G.delta) minDist = G.delta;
        o[p] = (T)(inside ? minDist : -minDist);
    }
}

}  // namespace ggx
