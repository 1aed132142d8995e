// kernels.h -- CDNA4 (gfx950) kernels of the per-grain level-set timestep.
//
// Every kernel is batched: a launch covers all live grains of a step (one workgroup per
// grain unless stated otherwise); the per-grain launch mode of the baseline issues the same
// kernels with a one-grain work list.  Boxes live in device arenas addressed by per-grain
// offsets; T is the field type (double for the FP64 path, float for the FP32 path).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

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
// slowest grain): the corrector runs as one launch, and the level-set kernel as one launch for
// every grain up to kMergeSide, the larger buckets keeping their own.
constexpr int kSmallNetwork = 4096;
constexpr int kMergeSide = 64;

struct Sched {
    int cursor[kMaxBuckets + 1];     // work cursors: level-set kernel per bucket, then the lists
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
    if (t <= kMaxBuckets) S->cursor[t] = 0;
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

// A grain that carries an error (or a box above the largest bucket) is taken out of the step:
// its existence flag is cleared, so no list, gather or launch touches its slots again, and it
// is deleted at the next step like a vanished grain; the host reports the error.
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
        int f = flags[g];
        if (f & kGone) { f &= ~kGone; flags[g] = f; }
        if ((f & kPresent) && !(f & kExists)) { f = (f & ~kPresent) | kGone; flags[g] = f; }
        if ((f & kPresent) && (f & kExists) && !err[g] && box[g].n > B.edge[B.count - 1]) err[g] = kErrBoxCap;
        if (err[g]) {
            s_err = 1;
            if (f & kExists) { f &= ~kExists; flags[g] = f; }
        }
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

// Work-list items.  Kernels whose per-item work is uniform (the convolutions: boxes of one bucket)
// take them statically, workgroup i taking items i, i + grid, ...: a shared cursor costs one
// same-address atomic per item, and those serialise across the chip at about 12 ns each.
// Kernels whose per-item work varies with the grain (lists, level set) pull items from a cursor
// when one is given (dynamic balance), else statically; with a cursor, one atomic takes a chunk
// of `chunk` consecutive items (chunk c covers items c * chunk ... c * chunk + chunk - 1).
__device__ __forceinline__ int take_item(int* cursor, int* s_slot, int prev, int chunk = 1) {
    if (!cursor) return prev < 0 ? (int)blockIdx.x : prev + (int)gridDim.x;
    if (prev >= 0 && (prev + 1) % chunk != 0) return prev + 1;
    __syncthreads();
    if (threadIdx.x == 0) *s_slot = atomicAdd(cursor, 1) * chunk;
    __syncthreads();
    return *s_slot;
}

// ------------------------------------------------------------------------------------------
// Comparison lists, LSbox::computeSecondOrderNeighbours (box.cpp:1027-1068).  One 64-lane
// workgroup per grain.  cmp = the existing entries of the previous list, then every existing
// neighbour-of-neighbour whose input box intersects (closed intervals, checkIntersection,
// box.cpp:881-888), first occurrence only, excluding self and the boundary grain.  The
// first-occurrence test is an LDS hash (grain id -> smallest candidate index), so the
// candidates are examined in parallel and compacted in their original order.
// ------------------------------------------------------------------------------------------
constexpr int kHash = 1024;      // LDS hash slots (grain id -> smallest candidate index)
constexpr int kHashFill = 768;   // distinct keys allowed per grain (> 2 kCmpCap: beyond it the list overflows anyway)
constexpr int kCandChunk = 2048; // neighbours-of-neighbours staged in LDS at a time

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

// Open-addressing insert (key-CAS): returns the slot holding `key`, or -1 when the table holds
// kHashFill keys already (the caller reports an error; probing stays bounded).
__device__ __forceinline__ int hash_insert(int* h_key, int* fill, int key) {
    unsigned hs = ((unsigned)key * 2654435761u) & (kHash - 1);
    while (true) {
        int cur = h_key[hs];
        if (cur == key) return (int)hs;
        if (cur == -1) {
            if (*fill >= kHashFill) return -1;
            int old = atomicCAS(&h_key[hs], -1, key);
            if (old == -1) { atomicAdd(fill, 1); return (int)hs; }
            if (old == key) return (int)hs;
        }
        hs = (hs + 1) & (kHash - 1);
    }
}

__device__ __forceinline__ int hash_find(const int* h_key, int key) {
    unsigned hs = ((unsigned)key * 2654435761u) & (kHash - 1);
    while (h_key[hs] != key) hs = (hs + 1) & (kHash - 1);
    return (int)hs;
}

__global__ void __launch_bounds__(256) k_lists(const int* __restrict__ alist, const int* __restrict__ count,
                                               int* __restrict__ cursor, const Box* __restrict__ box,
                                               const int* __restrict__ flags, const int* __restrict__ sec_cnt,
                                               const int* __restrict__ sec, int* __restrict__ cmp_cnt,
                                               int* __restrict__ cmp, int* __restrict__ err) {
    __shared__ int h_key[kHash];
    __shared__ int h_min[kHash];
    __shared__ int s_cand[kCandChunk];
    __shared__ int s_sec[kCmpCap];
    __shared__ int s_off[kCmpCap + 1];
    __shared__ int s_tmp[256];
    __shared__ int s_slot, s_fill, s_bad;
    const int t = threadIdx.x;
    const int total = *count;  // written by k_tally (or the host) before this kernel
    constexpr int kChunk = 4;  // items per cursor atomic: the list work of a grain is light
    for (int item = take_item(cursor, &s_slot, -1, kChunk); item < total;
         item = take_item(cursor, &s_slot, item, kChunk)) {
        __syncthreads();  // the previous item's shared state is free
        const int g = alist[item];
        const Box bg = box[g];
        const int ns = sec_cnt[g];
        int* out = cmp + (size_t)g * kCmpCap;
        for (int k = t; k < kHash; k += blockDim.x) { h_key[k] = -1; h_min[k] = 0x7fffffff; }
        if (t == 0) { s_fill = 0; s_bad = 0; }
        int ex = 0, len = 0;
        if (t < ns) {
            int nb = sec[(size_t)g * kCmpCap + t];
            s_sec[t] = nb;
            ex = (flags[nb] & kExists) ? 1 : 0;
            len = sec_cnt[nb];
        }
        int ntot;
        int koff = block_scan(len, s_tmp, &ntot);   // candidate offset of entry t
        if (t < ns) s_off[t] = koff;
        if (t == 0) s_off[ns] = ntot;
        int n1;
        int pos1 = block_scan(ex, s_tmp, &n1);      // rank among existing entries
        // part 1: existing entries of the previous list, in order (box.cpp:1038-1041)
        if (t < ns && ex) {
            out[pos1] = s_sec[t];
            int hs = hash_insert(h_key, &s_fill, s_sec[t]);
            if (hs >= 0) h_min[hs] = -1;  // already in the list
            else s_bad = 1;
        }
        __syncthreads();
        // candidates, flattened in (entry, entry's entry) order (box.cpp:1042-1048), staged in
        // chunks; pass 0 records each id's first valid index, pass 1 compacts first occurrences
        int written = n1;
        bool over = false;
        for (int pass = 0; pass < 2; ++pass) {
            for (int c0 = 0; c0 < ntot; c0 += kCandChunk) {
                const int cl = min(kCandChunk, ntot - c0);
                for (int a = 0; a < ns; ++a) {
                    const int lo = max(s_off[a], c0), hi = min(s_off[a + 1], c0 + cl);
                    const int* snb = sec + (size_t)s_sec[a] * kCmpCap - s_off[a];
                    for (int k = lo + t; k < hi; k += blockDim.x) s_cand[k - c0] = snb[k];
                }
                __syncthreads();
                for (int q = t; q < cl; q += blockDim.x) {
                    int c = s_cand[q];
                    bool valid = (flags[c] & kExists) && c != g && c != 0;
                    if (valid) {
                        Box bc = box[c];
                        valid = !(bg.x0 > bc.x0 + bc.n || bg.x0 + bg.n < bc.x0 || bg.y0 > bc.y0 + bc.n ||
                                  bg.y0 + bg.n < bc.y0);
                    }
                    if (!valid) { s_cand[q] = -1; continue; }
                    if (pass == 0) {
                        int hs = hash_insert(h_key, &s_fill, c);
                        if (hs >= 0) atomicMin(&h_min[hs], c0 + q);  // stays -1 for part-1 entries
                        else s_bad = 1;
                    }
                }
                __syncthreads();
                if (pass == 1 && !s_bad) {
                    // ordered compaction of first occurrences (box.cpp:1050-1066)
                    const int per = (cl + (int)blockDim.x - 1) / (int)blockDim.x;
                    const int q0 = t * per, q1 = min(cl, q0 + per);
                    int keep = 0;
                    for (int q = q0; q < q1; ++q) {
                        int c = s_cand[q];
                        if (c >= 0 && h_min[hash_find(h_key, c)] == c0 + q) keep++;
                    }
                    int nk;
                    int w = written + block_scan(keep, s_tmp, &nk);
                    for (int q = q0; q < q1; ++q) {
                        int c = s_cand[q];
                        if (c >= 0 && h_min[hash_find(h_key, c)] == c0 + q) {
                            if (w < kCmpCap) out[w] = c; else over = true;
                            w++;
                        }
                    }
                    written += nk;
                }
                __syncthreads();
            }
        }
        if (over) err[g] = kErrCmpCap;
        if (t == 0) {
            if (written > kCmpCap || s_bad) err[g] = kErrCmpCap;
            cmp_cnt[g] = min(written, kCmpCap);
        }
    }
}

// ------------------------------------------------------------------------------------------
// Circulant tables: the table of box side n holds K_n[(t - kKPad) mod n] for
// t in [0, 2n + 2 kKPad), so that every index a register block needs is in range without a
// modulo.
constexpr int kKPad = 8;
__host__ __device__ inline long long ktab_len(int n) { return 2LL * n + 2 * kKPad; }

// Convolution as an exact dense circulant (LSbox::convolutionGeneratorFFTW, box.cpp:622-695,
// Gaussian mode).  The Gaussian symbol G(i,j) = g(i) g(j) is separable and even, so
// IDFT(G . DFT(phi)) = K_n phi K_n with the symmetric circulant
// K_n[m] = sum_k g(k) cos(2 pi k m / n), computed on the host per box size with all n taps
// (the symbol is cut at Nyquist, so K_n has a slowly decaying tail and cannot be banded).
// Rows first, then columns.  Each lane produces a 4-wide run of outputs so that one LDS read
// of the input feeds four FMAs.  kk holds K_n twice (length 2n) so no modulo is needed.
// ------------------------------------------------------------------------------------------
template <class T, int S>
__device__ __forceinline__ void circ_run(const T* __restrict__ line, int stride, int n, int x0,
                                         const T* __restrict__ kk, T* acc) {
    // acc[s] = sum_j line[j] * K[(x0 + s - j) mod n],  kk[t] = K[t mod n] for t in [0, 2n)
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = T(0);
    for (int j = 0; j < n; ++j) {
        T v = line[j * stride];
        const T* kr = kk + (x0 - j + n);
#pragma unroll
        for (int s = 0; s < S; ++s) acc[s] += kr[s] * v;
    }
}

template <class T>
__device__ __forceinline__ void conv_one(int n, const T* __restrict__ s, T* __restrict__ d, T* kk, T* A, long long avail) {
    constexpr int S = 4;
    const long long nn = (long long)n * n;
    const int runs = (n + S - 1) / S;  // output runs per line
    if (2 * nn <= avail) {
        T* B = A + nn;
        for (long long p = threadIdx.x; p < nn; p += blockDim.x) A[p] = s[p];
        __syncthreads();
        for (int it = threadIdx.x; it < n * runs; it += blockDim.x) {
            int y = it / runs, x0 = (it - y * runs) * S;
            T acc[S];
            circ_run<T, S>(A + (long long)y * n, 1, n, x0, kk, acc);
#pragma unroll
            for (int q = 0; q < S; ++q)
                if (x0 + q < n) B[(long long)y * n + x0 + q] = acc[q];
        }
        __syncthreads();
        for (int it = threadIdx.x; it < n * runs; it += blockDim.x) {
            int x = it / runs, y0 = (it - x * runs) * S;
            T acc[S];
            circ_run<T, S>(B + x, n, n, y0, kk, acc);
#pragma unroll
            for (int q = 0; q < S; ++q)
                if (y0 + q < n) d[(long long)(y0 + q) * n + x] = acc[q];
        }
        return;
    }
    // strip mode: rows in strips of H rows, then columns in strips of H columns
    int H = (int)(avail / (2LL * n));
    if (H < 1) H = 1;  // the host guarantees room for two lines
    for (int y0 = 0; y0 < n; y0 += H) {
        int hh = min(H, n - y0);
        T* B = A + (long long)hh * n;
        for (long long p = threadIdx.x; p < (long long)hh * n; p += blockDim.x) A[p] = s[(long long)y0 * n + p];
        __syncthreads();
        for (int it = threadIdx.x; it < hh * runs; it += blockDim.x) {
            int y = it / runs, x0 = (it - y * runs) * S;
            T acc[S];
            circ_run<T, S>(A + (long long)y * n, 1, n, x0, kk, acc);
#pragma unroll
            for (int q = 0; q < S; ++q)
                if (x0 + q < n) B[(long long)y * n + x0 + q] = acc[q];
        }
        __syncthreads();
        for (long long p = threadIdx.x; p < (long long)hh * n; p += blockDim.x) d[(long long)y0 * n + p] = B[p];
        __syncthreads();
    }
    __threadfence();
    __syncthreads();
    for (int xs = 0; xs < n; xs += H) {
        int ww = min(H, n - xs);
        T* B = A + (long long)ww * n;
        for (long long p = threadIdx.x; p < (long long)ww * n; p += blockDim.x) {
            int y = (int)(p / ww), x = (int)(p - (long long)y * ww);
            A[(long long)x * n + y] = d[(long long)y * n + xs + x];
        }
        __syncthreads();
        for (int it = threadIdx.x; it < ww * runs; it += blockDim.x) {
            int x = it / runs, y0 = (it - x * runs) * S;
            T acc[S];
            circ_run<T, S>(A + (long long)x * n, 1, n, y0, kk, acc);
#pragma unroll
            for (int q = 0; q < S; ++q)
                if (y0 + q < n) B[(long long)x * n + y0 + q] = acc[q];
        }
        __syncthreads();
        for (long long p = threadIdx.x; p < (long long)ww * n; p += blockDim.x) {
            int y = (int)(p / ww), x = (int)(p - (long long)y * ww);
            d[(long long)y * n + xs + x] = B[(long long)x * n + y];
        }
        __syncthreads();
    }
}

// Persistent: every workgroup pulls grains of its bucket until the list is exhausted.
template <class T>
__global__ void __launch_bounds__(256) k_conv_circulant(const int* __restrict__ list, const int* __restrict__ count,
                                                        const Box* __restrict__ box,
                                                        const long long* __restrict__ off, const T* __restrict__ src,
                                                        T* __restrict__ dst, const long long* __restrict__ kern_off,
                                                        const T* __restrict__ kern, int nb, int lds_bytes) {
    constexpr int S = 4;
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    const int kkn = (2 * nb + S + 1) & ~1;  // kk region sized for the bucket's largest box
    T* kk = (T*)smem;
    T* A = kk + kkn;
    const long long avail = (long long)lds_bytes / (long long)sizeof(T) - kkn;
    const int total = *count;  // written by k_tally (or the host) before this kernel
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        __syncthreads();  // the previous box's LDS is free
        int g = list[item];
        int n = box[g].n;
        long long o = off[g];
        const T* kg = kern + kern_off[n];
        for (int t = threadIdx.x; t < 2 * n + S; t += blockDim.x) kk[t] = kg[kKPad + t % n];
        __syncthreads();
        conv_one<T>(n, src + o, dst + o, kk, A, avail);
    }
}

// ------------------------------------------------------------------------------------------
// The same circulant convolution, register-blocked for boxes whose two tiles fit in LDS.
// Row pass: lane = row y, each task a block of 8 outputs x0..x0+7 of the wave's rows,
//   B[y][x] = sum_j A[y][j] K[x - j];
// column pass: lane = column x, each task a block of 8 outputs y0..y0+7,
//   D[y][x] = sum_i B[i][x] K[y - i].
// The circulant coefficients of a block depend only on the task, so they are wave-uniform and
// come through the scalar cache into SGPRs; LDS only feeds the field values (one 8-byte read per
// 8 FMAs).  The tiles are zero-padded to n8 = 8 ceil(n/8) rows and columns and their pitch
// (n8 + 2 doubles, n8 + 4 floats) keeps the per-lane 16-byte row reads free of bank conflicts.
// ------------------------------------------------------------------------------------------
template <class T>
__host__ __device__ inline int dense_pitch(int n8) { return n8 + (sizeof(T) == 8 ? 2 : 4); }

template <class T>
__host__ __device__ inline long long dense_lds(int nb) {
    const int n8 = (nb + 7) & ~7;
    return 2LL * n8 * dense_pitch<T>(n8) * (long long)sizeof(T);
}

template <class T>
using ctab_ptr = const __attribute__((address_space(4))) T*;

template <class T>
__device__ __forceinline__ void load8(const T* p, T* a) {
    if constexpr (sizeof(T) == 8) {
        const double2* q = reinterpret_cast<const double2*>(p);
#pragma unroll
        for (int k = 0; k < 4; ++k) { double2 v = q[k]; a[2 * k] = v.x; a[2 * k + 1] = v.y; }
    } else {
        const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
        for (int k = 0; k < 2; ++k) { float4 v = q[k]; a[4 * k] = v.x; a[4 * k + 1] = v.y; a[4 * k + 2] = v.z; a[4 * k + 3] = v.w; }
    }
}

template <class T>
__device__ __forceinline__ void store8(T* p, const T* a) {
    if constexpr (sizeof(T) == 8) {
        double2* q = reinterpret_cast<double2*>(p);
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = make_double2(a[2 * k], a[2 * k + 1]);
    } else {
        float4* q = reinterpret_cast<float4*>(p);
#pragma unroll
        for (int k = 0; k < 2; ++k) q[k] = make_float4(a[4 * k], a[4 * k + 1], a[4 * k + 2], a[4 * k + 3]);
    }
}

// acc[q] += sum_u v[u] * W[q - u + 7], W = 15 consecutive (wave-uniform) table entries
template <class T>
__device__ __forceinline__ void block8(T* acc, const T* v, ctab_ptr<T> w) {
    T W[15];
#pragma unroll
    for (int t = 0; t < 15; ++t) W[t] = w[t];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[q] += v[u] * W[q - u + 7];
}

template <class T>
__global__ void __launch_bounds__(256) k_conv_dense(const int* __restrict__ list, const int* __restrict__ count,
                                                    const Box* __restrict__ box,
                                                    const long long* __restrict__ off, const T* __restrict__ src,
                                                    T* __restrict__ dst, const long long* __restrict__ kern_off,
                                                    const T* __restrict__ kern) {
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = (int)(blockDim.x >> 6);
    const int total = __builtin_amdgcn_readfirstlane(*count);  // written by k_tally (or the host)
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        __syncthreads();  // the previous box's LDS is free
        const int g = list[item];
        const int n = box[g].n;
        const long long o = off[g];
        const int n8 = (n + 7) & ~7;
        const int pa = dense_pitch<T>(n8);
        T* A = (T*)smem;
        T* B = A + (long long)n8 * pa;
        const ctab_ptr<T> kt = (ctab_ptr<T>)(kern + kern_off[n]);
        const T* s = src + o;
        // A = phi, zero-padded to n8 x n8
        for (int p = threadIdx.x; p < n8 * n8; p += blockDim.x) {
            const int y = p / n8, x = p - y * n8;
            A[y * pa + x] = (y < n && x < n) ? s[y * n + x] : T(0);
        }
        __syncthreads();
        // row pass
        const int xb = n8 >> 3, rg = (n8 + 63) >> 6;
        for (int task = wave; task < rg * xb; task += nwaves) {
            const int r64 = task / xb, bx = task - r64 * xb;
            const int y = r64 * 64 + lane, x0 = bx * 8;
            T acc[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[q] = T(0);
            const T* arow = A + (long long)y * pa;
            const bool on = y < n8;
            for (int j0 = 0; j0 < n8; j0 += 8) {
                T v[8];
                if (on) load8(arow + j0, v);
                else {
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = T(0);
                }
                block8(acc, v, kt + (x0 - j0 + n + kKPad - 7));
            }
            if (on) store8(B + (long long)y * pa + x0, acc);
        }
        __syncthreads();
        // column pass
        const int yb = n8 >> 3, cg = (n + 63) >> 6;
        T* d = dst + o;
        for (int task = wave; task < cg * yb; task += nwaves) {
            const int c64 = task / yb, by = task - c64 * yb;
            const int x = c64 * 64 + lane, y0 = by * 8;
            const bool on = x < n;
            T acc[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) acc[r] = T(0);
            for (int i0 = 0; i0 < n8; i0 += 8) {
                T v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = on ? B[(long long)(i0 + u) * pa + x] : T(0);
                block8(acc, v, kt + (y0 - i0 + n + kKPad - 7));
            }
            if (on) {
#pragma unroll
                for (int r = 0; r < 8; ++r)
                    if (y0 + r < n) d[(long long)(y0 + r) * n + x] = acc[r];
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------
// Contour, volume, motion check, new box and direct neighbours:
// LSbox::extractContour (box.cpp:1089-1153) with MarchingSquaresAlgorithm::generateContour
// (marchingSquares.cpp:28-188), isMotionRegular (box.cpp:1155-1190), clearContourGrainArea
// (1883-1904), then computeVolumeAndEnergy (1201-1228) -> buildDirectNeighbours
// (grainBoundary.cpp:85-199).  One workgroup per grain: the inside/outside test of the box is
// kept as a bitmask in LDS so lane 0's trace never waits on memory for its direction; the
// neighbour probes run on all lanes.
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
