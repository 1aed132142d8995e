// level.h -- the level-set phase of a step: comparison, contour and neighbours, redistancing, as
// four kernels with one work split each.
//
// Together they perform, for every grain, what the reference does in the phases comparison_box,
// level_set and redistancing (src/grainhdl.cpp:815-869):
//   k_compare  LSbox::executeComparison (box.cpp:890-943) + boundaryCondition (968-1025),
//              LSbox::executeSetComparison (838-879); one wave per 8 rows of a grain
//   k_contour  LSbox::extractContour (1089-1153): MarchingSquaresAlgorithm::generateContour
//              (marchingSquares.cpp:28-188), computeVolume, isMotionRegular (1155-1190),
//              clearContourGrainArea (1883-1904), bounds clamp + resizeToSquare, computePerimeter,
//              then LSbox::computeVolumeAndEnergy (1201-1228): buildDirectNeighbours
//              (grainBoundary.cpp:85-199); one wave per grain up to side 64, four above
//   k_alloc    room in the next field arena for every new box (one atomic per 256 grains)
//   k_redist   LSbox::executeRedistancing (1259-1399); one line per lane, the new field in LDS
// The kernels hand each other the compared field C (in an arena of its own at the step's offsets: a
// frame's copy may still be reading the input fields) and its signs as bit planes: per grain, rows and
// columns of the tests C >= 0 and C > 0.  The contour's topology and the sweeps' signs come from the
// bits; C itself is read at the zero crossings only.  On the 100k-grain lognormal network in FP64
// (1.61e8 box points) the four take 2.2, 1.8, 0.01 and 2.1 ms per step; one kernel that did all of
// it per grain, 256 lanes wide with C and the new field in LDS, took 11.8 ms: its serial phases
// left three of four waves idle and its LDS tiles held four or five grains per CU.
#pragma once
#include "aniso.h"
#include "kernels.h"

namespace ggx {

// Sign planes of the compared fields, 64-bit words in the grain's field slot (offset / 8 words,
// which n rows of ceil(n / 64) words always fit): per row and per column the bits C >= 0 and C > 0.
// Row bits beyond the box are zero; column bits beyond it are undefined.
enum { kRowGe = 0, kRowGt = 1, kColGe = 2, kColGt = 3, kPlanes = 4 };
__host__ __device__ inline long long plane_words(long long field_elems) { return field_elems / 8 + 8; }

// Slots of the gathered-pixel count (one cache line each): the waves of a launch spread over them.
constexpr int kCountSlots = 64, kCountStride = 16;

template <class T>
struct LevelArgs {
    Items it;
    const long long* contour_base;  // first contour slot of each bucket (k_tally); null: atomic bump
    const Box* box;
    const long long* off;
    const int* cmp_cnt;
    const int* cmp;
    const T* tilde;            // convolved fields (all grains)
    T* cfield;                 // takes the compared fields: an arena of their own (after a coarsening, the phi arena)
    unsigned long long* bits;  // sign planes, `plane` words each
    long long plane;
    const uint32_t* idl_old;
    uint32_t* idl_new;
    long long* off_prev;       // in: IDLocal layout of the previous step; out (k_contour): this step's
    int* n_prev;
    T* out_field;              // next phi arena
    T* rec_s;                  // non-null (a recorded step): per pixel the set-compared field ...
    int* rec_win;              // ... and the comparison's winner (grain id, 0 wall, -1 none, -2 cleared),
    int* rec_area;             // ... and per grain 1 where the step wrote a new area
    ContourOut O;
    GridConst G;
    const int* loop;           // loop index of the step (device counter, so a captured step replays)
    int analysis_timestep;
    unsigned long long* gather_part;   // kCountSlots running sums of neighbour pixels compared
    unsigned long long* out_total;     // running sum of the new boxes' areas
    int nb;                    // largest box side of the launch
    int cap;                   // largest contour capacity of the launch
    int blocks;                // k_compare: waves per grain; each loops over blocks of 8 rows x 64 columns
    int tile;                  // k_redist: largest new box side the LDS tile holds (0: no tile)
    AnisoConst K;              // anisotropic boundaries (K.on = 0: isotropic network)
    AnisoState AS;
};

// True where the grain's box reaches the domain wall's neighbourhood (boundaryCondition applies).
__device__ __forceinline__ bool at_wall(const Box& b, const GridConst& G) {
    const int lo = 2 * G.gb, hi = G.m - 2 * G.gb;
    return !(b.x0 > lo && b.x0 + b.n < hi && b.y0 > lo && b.y0 + b.n < hi);
}

// boundaryCondition (box.cpp:968-1025): the wall's value at pixel (i, j).
__device__ __forceinline__ double wall_distance(int i, int j, const GridConst& G) {
    const int gb = G.gb, m2 = G.m;
    const int dXMin = -(j - gb), dYMin = -(i - gb);
    const int dXMax = (j - (m2 - gb)), dYMax = (i - (m2 - gb));
    const int dX = (abs(dXMin) < abs(dXMax)) ? dXMin : dXMax;
    const int dY = (abs(dYMin) < abs(dYMax)) ? dYMin : dYMax;
    if (dX > 0 && dY > 0) return sqrt((double)dX * dX + dY * dY);
    if (dX < 0 && dY > 0) return dY;
    if (dX > 0 && dY < 0) return dX;
    if (dX < 0 && dY < 0) return max(dX, dY);
    if (dX == 0) return (dY > 0) ? (double)dY : 0.0;
    return (dX > 0) ? (double)dX : 0.0;
}

// Interpolated point of a recorded move (marchingSquares.cpp:204-265).
template <class T>
__device__ __forceinline__ double2 move_point(const T* C, int n, int cp, int x0, int y0, uint32_t mv) {
    int dir = (int)(mv & 3u);
    int left = (int)((mv >> 2) & 0x3fffu) + x0 - 1;
    int top = (int)((mv >> 16) & 0x3fffu) + y0 - 1;
    int right = left + 1, bottom = top + 1;
    auto val = [&](int row, int col) { return (double)C[(row - y0) * cp + (col - x0)]; };
    double2 r;
    double delta;
    switch (dir) {
        case D_LEFT:
            r.x = left;
            if (top < y0) r.y = bottom;
            else { delta = val(bottom, left) - val(top, left); r.y = bottom - val(bottom, left) / delta; }
            break;
        case D_RIGHT:
            r.x = right;
            if (bottom >= y0 + n) r.y = top;
            else { delta = val(top, right) - val(bottom, right); r.y = top + val(top, right) / delta; }
            break;
        case D_UP:
            r.y = top;
            if (right >= x0 + n) r.x = left;
            else { delta = val(top, left) - val(top, right); r.x = left + val(top, left) / delta; }
            break;
        default:  // D_DOWN
            r.y = bottom;
            if (left < x0) r.x = right;
            else { delta = val(bottom, right) - val(bottom, left); r.x = right - val(bottom, right) / delta; }
            break;
    }
    return r;
}

// The square walk of MarchingSquaresAlgorithm::generateContour (marchingSquares.cpp:44-176)
// from the first inside pixel (sx, sy): inside(row, col) is the inside test (value >= 0 within
// the box), emit(k, move) records the k-th point-generating move packed as direction (2 bits),
// left - x0 + 1 (14 bits) and top - y0 + 1 (16 bits); the two corners shared with the next
// square are reused.  Returns 0, kErrContourCap or kErrTrace; *nmoves gets the move count.
// visit(left, top, mask) is called at every square the walk passes, saddles included, in walk
// order (generateJunction's call site, marchingSquares.cpp:177).
template <class Inside, class Emit, class Visit>
__device__ __forceinline__ int walk_squares_v(int sx, int sy, int x0, int y0, int n, int ccap, Inside inside, Emit emit,
                                              Visit visit, int* nmoves) {
    int left = sx - 1, top = sy - 1;
    int next = D_NONE, prev = D_NONE;
    const long long itcap = 8LL * (n + 2) * (n + 2) + 16;
    long long it = 0;
    int nm = 0, st = 0;
    bool tl = inside(top, left), tr = inside(top, left + 1);
    bool bl = inside(top + 1, left), br = inside(top + 1, left + 1);
    do {
        const int mask = (tl ? MS_TL : 0) | (tr ? MS_TR : 0) | (bl ? MS_BL : 0) | (br ? MS_BR : 0);
        bool gen = true;
        switch (mask) {
            case MS_TL: next = D_UP; break;
            case MS_TR: next = D_RIGHT; break;
            case MS_TL | MS_TR: next = D_RIGHT; break;
            case MS_BL: next = D_LEFT; break;
            case MS_BL | MS_TL: next = D_UP; break;
            case MS_BL | MS_TR: next = (prev == D_UP) ? D_RIGHT : D_LEFT; gen = false; break;
            case MS_BL | MS_TR | MS_TL: next = D_RIGHT; break;
            case MS_BR: next = D_DOWN; break;
            case MS_BR | MS_TL: next = (prev == D_RIGHT) ? D_DOWN : D_UP; gen = false; break;
            case MS_BR | MS_TR: next = D_DOWN; break;
            case MS_BR | MS_TR | MS_TL: next = D_DOWN; break;
            case MS_BR | MS_BL: next = D_LEFT; break;
            case MS_BR | MS_BL | MS_TL: next = D_UP; break;
            case MS_BR | MS_BL | MS_TR: next = D_LEFT; break;
            default: gen = false; break;
        }
        if (gen) {
            if (nm >= ccap) { st = kErrContourCap; break; }
            emit(nm++, (uint32_t)next | ((uint32_t)(left - x0 + 1) << 2) | ((uint32_t)(top - y0 + 1) << 16));
        }
        visit(left, top, mask);
        switch (next) {
            case D_UP: top--; bl = tl; br = tr; tl = inside(top, left); tr = inside(top, left + 1); break;
            case D_DOWN: top++; tl = bl; tr = br; bl = inside(top + 1, left); br = inside(top + 1, left + 1); break;
            case D_LEFT: left--; tr = tl; br = bl; tl = inside(top, left); bl = inside(top + 1, left); break;
            case D_RIGHT: left++; tl = tr; bl = br; tr = inside(top, left + 1); br = inside(top + 1, left + 1); break;
            default: break;
        }
        prev = next;
        if (++it > itcap) { st = kErrTrace; break; }
    } while (left != sx - 1 || top + 1 != sy);
    *nmoves = nm;
    return st;
}

// Exclusive prefix count of a per-lane flag over the workgroup in lane order, and the total:
// one ballot per wave and one exchange of wave totals through LDS (s_wt, one int per wave).
__device__ __forceinline__ int block_flag_scan(bool f, int* s_wt, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const unsigned long long m = __ballot(f);
    const int pre = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) s_wt[wave] = __popcll(m);
    __syncthreads();
    int base = 0, tot = 0;
    for (int w = 0; w < nw; ++w) {
        const int c = s_wt[w];
        if (w < wave) base += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return base + pre;
}

// ------------------------------------------------------------------------------------------
// k_compare: one wave per block of 8 rows and 64 columns of a grain's box, lane = column.
//
// Bound by the rate of the neighbours' row loads (3.7 neighbour pixels per box pixel on the
// lognormal networks, in rows that fill about a quarter of the lanes): without the gathers it takes
// 1.2 of 2.6 ms, without the stores 2.1.  A row of a neighbour's overlap is one coalesced load off a
// wave-uniform address; two entries' rows (16 loads) are in flight at a time.  With the rows' cases
// in branches of their own the values met in copies, which waited for one entry's loads before the
// next entry's were issued.  The lanes hold the list's boxes (readlane hands them out), so the waves
// of a grain share nothing and meet no barrier.  Only the entries that meet the block are walked, in
// list order (strict >, first wins).  One launch takes all sides in spatial order, a contiguous part
// per die: 8 launches, one per side, fetched 8.9 GB in place of 4.7 from beyond the dies' caches.
// 100k-grain network in FP64 2.65 -> 2.2 ms per step, 30k in FP32 0.62 -> 0.51, 2000 grains 0.39 -> 0.23.
//
// COARSEN: the pass after a grid coarsening (grainhdl.cpp:1464-1476): the comparison of the grains
// that exist writes IDLocal (LSbox::recalculateIDLocal, box.cpp:1497-1505; `tilde` holds the
// regridded fields), no set comparison.
// ------------------------------------------------------------------------------------------
// f[i] of a wave-uniform field: its address stays in scalar registers and the lane adds 32 bits.
template <class T>
__device__ __forceinline__ T at_lane(const T* f, unsigned i) {
    return *(const T*)((const char*)f + (unsigned long long)(i * (unsigned)sizeof(T)));
}

constexpr int kRows = 8;   // rows of a wave's block (one byte of the column planes)
constexpr unsigned kDies = 8;

template <class T, bool COARSEN>
__global__ void __launch_bounds__(256) k_compare(LevelArgs<T> A) {
    const GridConst& G = A.G;
    const int lane = (int)(threadIdx.x & 63);
    const int total = items_total(A.it);
    // Workgroups go to the dies in turn; each die takes a contiguous part of the (spatially ordered)
    // list, so that its cache holds the fields its grains share.
    const unsigned dies = gridDim.x >= 8 * kDies ? kDies : 1, die = blockIdx.x % dies;
    const int last = (int)((long long)total * (die + 1) / dies);
    const unsigned wpb = blockDim.x >> 6;
    const unsigned w0 = (unsigned)__builtin_amdgcn_readfirstlane((int)((blockIdx.x / dies) * wpb + (threadIdx.x >> 6)));
    const unsigned step = (gridDim.x - die + dies - 1) / dies * wpb, blocks = (unsigned)A.blocks;
    int item = (int)((long long)total * die / dies) + (int)(w0 / blocks), blk = (int)(w0 % blocks);
    const int item_step = (int)(step / blocks), blk_step = (int)(step % blocks);
    unsigned long long hits = 0;
    for (; item < last; item += item_step, blk += blk_step) {
        if (blk >= A.blocks) {
            blk -= A.blocks;
            if (++item >= last) break;
        }
        int bucket, pos;
        const int g = item_grain(A.it, item, &bucket, &pos);
        const Box b = sload_box(A.box + g);
        const int n = b.n, W = (n + 63) >> 6, rb = (n + kRows - 1) / kRows;
        if (blk >= rb * W) continue;
        const long long o = sload(A.off + g);
        const bool cmp_on = COARSEN ? ((sload(A.O.flags + g) & kExists) != 0) : true;
        const int cnt = cmp_on ? sload(A.cmp_cnt + g) : 0;
        // lane e holds entry e0 + e of the comparison list
        int eid = 0, ex = 0, ey = 0, en = 0;
        long long eo = 0;
        auto entries = [&](int e0) {
            if (e0 + lane < cnt) {
                eid = A.cmp[(size_t)g * kCmpCap + e0 + lane];
                const Box q = A.box[eid];
                ex = q.x0 - b.x0;
                ey = q.y0 - b.y0;
                en = q.n;
                eo = A.off[eid];
            }
        };
        entries(0);
        for (int block = blk; block < rb * W; block += A.blocks) {
            const int xc = block / rb, rblk = block - xc * rb;
            const int r0 = rblk * kRows, rows = min(kRows, n - r0), x = xc * 64 + lane;
            const bool on = x < n;
            const int xl = min(x, n - 1);
            T mx[kRows];
            int id[kRows];
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                mx[r] = T(-1.0);
                id[r] = -1;
            }
            for (int e0 = 0; e0 < cnt; e0 += 64) {
                const bool have = e0 + lane < cnt;
                if (cnt > 64) entries(e0);
                if (block == 0) {  // pixels of the whole box that the entry covers (a statistic)
                    const int ox = min(n, ex + en) - max(0, ex), oy = min(n, ey + en) - max(0, ey);
                    if (have && ox > 0 && oy > 0) hits += (unsigned long long)ox * (unsigned long long)oy;
                }
                unsigned long long todo = __ballot(have && ey < r0 + rows && ey + en > r0 && ex < xc * 64 + 64 && ex + en > xc * 64);
                while (todo) {
                    // The loads of kK entries are in flight together: pixels an entry does not cover stay
                    // unset and are not compared, so no value has to be merged (and waited for) between the
                    // entries.  A missing last entry is the one before again (strict >: without effect).
                    constexpr int kK = 2;
                    T v[kK][kRows];
                    int sid[kK], y0[kK], nk[kK], k = 0;
                    bool in[kK];
#pragma unroll
                    for (int u = 0; u < kK; ++u) {
                        if (todo) k = (int)__builtin_ctzll(todo);
                        todo &= todo - 1ull;
                        sid[u] = __builtin_amdgcn_readlane(eid, k);
                        const int col = xl - __builtin_amdgcn_readlane(ex, k);
                        nk[u] = __builtin_amdgcn_readlane(en, k);
                        y0[u] = r0 - __builtin_amdgcn_readlane(ey, k);  // the block's first row in the entry's box
                        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)eo, k);
                        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)((unsigned long long)eo >> 32), k);
                        const T* src = A.tilde + (long long)(((unsigned long long)hi << 32) | lo);
                        in[u] = (unsigned)col < (unsigned)nk[u];
#pragma unroll
                        for (int r = 0; r < kRows; ++r)
                            if (in[u] && (unsigned)(y0[u] + r) < (unsigned)nk[u])
                                v[u][r] = at_lane(src, (unsigned)((y0[u] + r) * nk[u] + col));
                    }
#pragma unroll
                    for (int u = 0; u < kK; ++u)
#pragma unroll
                        for (int r = 0; r < kRows; ++r) {
                            const bool ok = (unsigned)(y0[u] + r) < (unsigned)nk[u] && in[u];
                            if (ok && v[u][r] > mx[r]) { mx[r] = v[u][r]; id[r] = sid[u]; }
                        }
                }
            }
            // per pixel: the wall as grain 0, IDLocal, the set comparison, the sign bits
            const bool bnd = at_wall(b, G) && cmp_on;
            const double band = 0.7 * G.delta;
            const int nprev = sload(A.n_prev + g);
            const int np = nprev * nprev;
            const long long op = sload(A.off_prev + g);
            if (bnd) {
#pragma unroll
                for (int r = 0; r < kRows; ++r) {
                    const double dist = wall_distance(b.y0 + r0 + r, b.x0 + x, G);
                    if ((T)(dist * G.h) > mx[r]) { mx[r] = (T)(dist * G.h); id[r] = 0; }
                }
            }
            // all rows' loads are in flight together: what is not needed loads a pixel that is there anyway
            const T* field = A.tilde + o;
            const uint32_t* old = A.idl_old + (np > 0 ? op : 0);
            const int p0 = r0 * n + x;
            T own[kRows];
            uint32_t stale[kRows];
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                own[r] = at_lane(field, (unsigned)(min(r0 + r, n - 1) * n + xl));
                const int p = (on && r < rows && id[r] < 0 && p0 + r * n < np) ? p0 + r * n : -1;
                stale[r] = at_lane(old, (unsigned)max(p, 0));
                if (p < 0) stale[r] = 0u;
            }
            unsigned long long row_ge = 0, row_gt = 0;  // of the block's row `lane`
            unsigned col_ge = 0, col_gt = 0;            // of the lane's column, bit = row
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                if (r < rows) {
                    const int p = p0 + r * n;
                    T c = T(-1.0);
                    if (on) {
                        const T tv = own[r];
                        c = COARSEN ? tv : ((fabs((double)tv) < band) ? (T)(0.5 * ((double)tv - (double)mx[r])) : tv);
                        A.cfield[o + p] = c;
                        A.idl_new[o + p] = (id[r] >= 0) ? (uint32_t)id[r] : stale[r];
                        if (A.rec_s) {
                            A.rec_s[o + p] = c;
                            A.rec_win[o + p] = id[r];
                        }
                    }
                    const unsigned long long mge = __ballot(on && c >= T(0)), mgt = __ballot(on && c > T(0));
                    if (lane == r) { row_ge = mge; row_gt = mgt; }
                    col_ge |= (on && c >= T(0)) ? 1u << r : 0u;
                    col_gt |= (on && c > T(0)) ? 1u << r : 0u;
                }
            }
            unsigned long long* bits = A.bits + (o >> 3);
            if (lane < rows) {
                bits[kRowGe * A.plane + (long long)(r0 + lane) * W + xc] = row_ge;
                bits[kRowGt * A.plane + (long long)(r0 + lane) * W + xc] = row_gt;
            }
            if (on) {
                ((unsigned char*)(bits + kColGe * A.plane + (long long)x * W))[rblk] = (unsigned char)col_ge;
                ((unsigned char*)(bits + kColGt * A.plane + (long long)x * W))[rblk] = (unsigned char)col_gt;
            }
        }
    }
    // one addition per wave that met a grain's first block, spread over the slots
    if (__ballot(hits != 0ull)) {
        double h = (double)hits;  // exact: far below 2^53
        for (int d = 32; d >= 1; d >>= 1) h += __shfl_xor(h, d);
        if (lane == 0) atomicAdd(A.gather_part + (size_t)(w0 % kCountSlots) * kCountStride, (unsigned long long)h);
    }
}

// ------------------------------------------------------------------------------------------
// k_contour: contour, motion check, new box and direct neighbours of one grain per workgroup.
//
// The marching-squares walk is a chain of dependent steps, about 100 per grain.  Without a saddle
// the walk is a cycle over the squares the contour crosses, each with one successor, so it is
// ranked instead of walked: the squares are numbered by a scan over the bit rows, every square
// finds its successor with one popcount, and log2(squares) rounds of pointer jumping give each
// square of the start's cycle its place.  Boxes with a saddle, or with more squares than the node
// arrays hold, are walked by wave 0 over the bit rows.  Both record the same moves.
// The ordered sums (area, perimeter, energy, lengths per neighbour) keep the contour's order: 64
// terms at a time go through LDS and one wave adds them, so every sum sees the reference's
// rounding; the terms are loaded eight ahead (a 100-grain network 49 -> 36 us per step, 30k grains in
// FP32 0.82 -> 0.74 ms: a load per addition waited for the LDS each time).  One wave per grain up to
// side 64 (no barrier), four above.  What is left is one grain's latency, phase after phase.
// ------------------------------------------------------------------------------------------
constexpr int kNodeEnd = 0xffff;

// use(k, load(k)) for k = 0 .. m - 1 in order, U loads ahead of their uses: an ordered sum over LDS
// then waits for the LDS once in U terms.
template <int U, class Load, class Use>
__device__ __forceinline__ void in_order(int m, Load load, Use use) {
    int k = 0;
    for (; k + U <= m; k += U) {
        decltype(load(0)) v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load(k + u);
#pragma unroll
        for (int u = 0; u < U; ++u) use(k + u, v[u]);
    }
    for (; k < m; ++k) use(k, load(k));
}

// nearest_vertex by a whole wave: the smallest squared distance below 1e6, the first vertex that
// has it; 1e9 where there is none.  pt(i) reads contour point i.
template <class Pt>
__device__ __forceinline__ double wave_nearest_vertex(Pt pt, int size, double px, double py) {
#pragma clang fp contract(off)
    double best = 1000000.0, at = 1e9;
    for (int k = (int)(threadIdx.x & 63); k < size - 1; k += 64) {
        const double2 v = pt(k);
        const double dx = px - v.x, dy = py - v.y;
        const double dist = dx * dx + dy * dy;
        if (dist < best) { at = (double)k; best = dist; }
    }
    for (int d = 32; d >= 1; d >>= 1) {
        const double ob = __shfl_xor(best, d), oa = __shfl_xor(at, d);
        if (ob < best || (ob == best && oa < at)) { best = ob; at = oa; }
    }
    return at;
}

// LDS of k_contour for boxes up to nb with contours up to cap points: bit rows, the squares' bit
// rows and node bases, a chunk's staging, the first points and segment lengths of the contour
// (the rest are read back from the contour arena), and the nodes / moves / neighbour slots.
struct ContourLayout {
    int W, Wq, nodes, pts;
    int o_act, o_base, o_stage, o_pts, o_len, o_node, total;
};

__host__ __device__ inline ContourLayout contour_layout(int nb, int cap, int nt) {
    ContourLayout L;
    L.W = (nb + 63) / 64;
    L.Wq = (nb + 64) / 64;
    L.nodes = min(cap, 4 * nb + 64);
    L.pts = min(3 * nb + 64, 1024);
    L.o_act = nb * L.W * 8;
    L.o_base = L.o_act + (nb + 1) * L.Wq * 8;
    L.o_stage = (L.o_base + (nb + 1) * L.Wq * 4 + 15) & ~15;
    L.o_pts = L.o_stage + (nt + 1) * 16;
    L.o_len = L.o_pts + L.pts * 16;
    L.o_node = L.o_len + L.pts * 8;
    L.total = (L.o_node + max(12 * L.nodes, 4 * cap) + 15) & ~15;
    return L;
}

// Direction the walk leaves an ordinary square in, by its case (marchingSquares.cpp:44-176): two
// bits per case; cases 0, 6, 9 and 15 (no boundary, the saddles) hold nothing.
constexpr unsigned kSquareDir =
    (D_UP << 2 * MS_TL) | ((unsigned)D_RIGHT << 2 * MS_TR) | ((unsigned)D_RIGHT << 2 * (MS_TL | MS_TR)) |
    ((unsigned)D_LEFT << 2 * MS_BL) | (D_UP << 2 * (MS_BL | MS_TL)) | ((unsigned)D_RIGHT << 2 * (MS_BL | MS_TR | MS_TL)) |
    ((unsigned)D_DOWN << 2 * MS_BR) | ((unsigned)D_DOWN << 2 * (MS_BR | MS_TR)) |
    ((unsigned)D_DOWN << 2 * (MS_BR | MS_TR | MS_TL)) | ((unsigned)D_LEFT << 2 * (MS_BR | MS_BL)) |
    (D_UP << 2 * (MS_BR | MS_BL | MS_TL)) | ((unsigned)D_LEFT << 2 * (MS_BR | MS_BL | MS_TR));

// Corner bits of the squares 64 w .. 64 w + 63 of square row r (corners at pixel rows r - 1 and r,
// the square's right corners at its own column): s_ge holds n rows of W words.
struct SquareBits {
    unsigned long long tl, tr, bl, br;
};

__device__ __forceinline__ SquareBits square_bits(const unsigned long long* s_ge, int n, int W, int r, int w) {
    auto right = [&](int row) -> unsigned long long {
        return (unsigned)row < (unsigned)n && w < W ? s_ge[row * W + w] : 0ull;
    };
    auto carry = [&](int row) -> unsigned long long {
        return (unsigned)row < (unsigned)n && w > 0 ? s_ge[row * W + w - 1] >> 63 : 0ull;
    };
    SquareBits q;
    q.tr = right(r - 1);
    q.br = right(r);
    q.tl = (q.tr << 1) | carry(r - 1);
    q.bl = (q.br << 1) | carry(r);
    return q;
}

template <class T, bool ANISO, bool COARSEN, int NT>
__global__ void __launch_bounds__(NT) k_contour(LevelArgs<T> A) {
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    const GridConst& G = A.G;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const ContourLayout LY = contour_layout(A.nb, A.cap, NT);
    unsigned long long* s_ge = (unsigned long long*)smem;
    unsigned long long* s_act = (unsigned long long*)(smem + LY.o_act);
    int* s_base = (int*)(smem + LY.o_base);
    double2* s_stage = (double2*)(smem + LY.o_stage);
    double2* s_pt = (double2*)(smem + LY.o_pts);
    double* s_len = (double*)(smem + LY.o_len);
    uint32_t* s_node = (uint32_t*)(smem + LY.o_node);
    uint32_t* s_hopA = s_node + LY.nodes;
    uint32_t* s_hopB = s_hopA + LY.nodes;
    int* s_cand = (int*)s_node;   // neighbour of each segment, later its slot in the neighbour list
    __shared__ int s_tmp[16];
    __shared__ int s_int[12];     // 0 saddles, 1 moves, 2 regular, 3 error, 4 flag kept, 5 xmin, 6 xmax, 7 ymin, 8 ymax, 9 stop, 10 junctions
    __shared__ double s_dbl[8];   // 0 volume sum, 1 minx, 2 maxx, 3 miny, 4 maxy, 5 perimeter
    __shared__ long long s_coff;
    __shared__ double s_nbe[ANISO ? kNbCap : 1];

    const int total = items_total(A.it);
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        __syncthreads();  // the previous grain's shared state is free
        int bucket, pos;
        const int g = item_grain(A.it, item, &bucket, &pos);
        const int ccap = A.it.cap[bucket];
        const Box b = sload_box(A.box + g);
        const int n = b.n, W = (n + 63) >> 6;
        const long long o = sload(A.off + g);
        const long long nn = (long long)n * n;
        unsigned long long* bits = A.bits + (o >> 3);
        T* C = A.cfield + o;
        const int old_len = A.O.clen[g];
        const double old_vol = A.O.volume[g];
        for (int k = tid; k < n * W; k += NT) s_ge[k] = bits[kRowGe * A.plane + k];
        if (tid == 0) {
            s_int[3] = 0;
            s_int[4] = 1;
            const unsigned long long co = A.contour_base
                                              ? (unsigned long long)(A.contour_base[bucket] + (long long)pos * ccap)
                                              : atomicAdd(&A.O.tops[1], (unsigned long long)ccap);
            s_coff = (long long)co;
            if (co + (unsigned long long)ccap > (unsigned long long)A.O.contour_cap) s_int[3] = kErrContourCap;
            const bool bnd = at_wall(b, G);
            const int f = A.O.flags[g];
            A.O.flags[g] = bnd ? (f | kBoundary) : (f & ~kBoundary);
            A.n_prev[g] = n;       // this step's IDLocal is the stale source of the next step
            A.off_prev[g] = o;
            if constexpr (ANISO) A.AS.idl_org[g] = make_int2(b.x0, b.y0);
        }
        __syncthreads();
        if (s_int[3]) {  // no contour space: the grain leaves the step (no slot of it is used again)
            if (tid == 0) {
                A.O.err[g] = s_int[3];
                A.O.flags[g] &= ~kExists;
            }
            continue;
        }
        double2* pts = A.O.pts + s_coff;
        // bounding box of C >= 0, before any clearing (box.cpp:856-868)
        if (tid < 64) {
            int x0 = n, x1 = -1, y0 = n, y1 = -1;
            for (int c = 0; c < W; ++c) {
                const int k = c * 64 + lane;
                bool row = false, col = false;
                if (k < n) {
                    for (int w = 0; w < W; ++w) {
                        const unsigned long long last = w == W - 1 && (n & 63) ? (1ull << (n & 63)) - 1ull : ~0ull;
                        row = row || s_ge[k * W + w] != 0ull;
                        col = col || (bits[kColGe * A.plane + (long long)k * W + w] & last) != 0ull;
                    }
                }
                const unsigned long long mr = __ballot(row), mc = __ballot(col);
                if (mr) { y0 = min(y0, c * 64 + (int)__builtin_ctzll(mr)); y1 = c * 64 + 63 - (int)__builtin_clzll(mr); }
                if (mc) { x0 = min(x0, c * 64 + (int)__builtin_ctzll(mc)); x1 = c * 64 + 63 - (int)__builtin_clzll(mc); }
            }
            if (tid == 0) { s_int[5] = x0; s_int[6] = x1; s_int[7] = y0; s_int[8] = y1; }
        }
        __syncthreads();
        // ---------------- contour with motion check and retries ----------------
        int retries = 0, nm = 0, len = 0, start_row = 0, start_col = 0;
        bool exists = true, ranked = false;
        const uint32_t* moves = s_node;
        const int bb_x0 = s_int[5], bb_x1 = s_int[6], bb_y0 = s_int[7], bb_y1 = s_int[8];
        auto pt = [&](int i) -> double2 { return i < LY.pts ? s_pt[i] : pts[i]; };
        while (true) {
            // start: the first inside pixel in row-major order (marchingSquares.cpp:32-42)
            int sr = -1, sc = 0;
            for (int r0 = retries ? 0 : bb_y0; r0 < n && sr < 0; r0 += 64) {
                bool any = false;
                if (r0 + lane < n)
                    for (int w = 0; w < W; ++w) any = any || s_ge[(r0 + lane) * W + w] != 0ull;
                const unsigned long long m = __ballot(any);
                if (m) sr = r0 + (int)__builtin_ctzll(m);
            }
            if (sr < 0) {  // no inside point: the grain vanished
                exists = false;
                len = 0;
                break;
            }
            for (int w = 0; w < W; ++w)
                if (s_ge[sr * W + w] != 0ull) { sc = w * 64 + (int)__builtin_ctzll(s_ge[sr * W + w]); break; }
            sr = __builtin_amdgcn_readfirstlane(sr);
            sc = __builtin_amdgcn_readfirstlane(sc);
            start_row = sr;
            start_col = sc;
            // number the squares the contours cross
            const int Wq = (n + 64) >> 6, Q = (n + 1) * Wq;
            if (tid == 0) s_int[0] = 0;
            __syncthreads();
            int M = 0;
            for (int q0 = 0; q0 < Q; q0 += NT) {
                const int q = q0 + tid;
                int c = 0;
                if (q < Q) {
                    const SquareBits s = square_bits(s_ge, n, W, q / Wq, q % Wq);
                    const unsigned long long act = (s.tl | s.tr | s.bl | s.br) & ~(s.tl & s.tr & s.bl & s.br);
                    const unsigned long long saddle = (s.tr & s.bl & ~s.tl & ~s.br) | (s.tl & s.br & ~s.tr & ~s.bl);
                    s_act[q] = act;
                    c = __popcll(act);
                    if (saddle) s_int[0] = 1;
                }
                int tot;
                const int base = M + block_scan(c, s_tmp, &tot);
                if (q < Q) s_base[q] = base;
                M += tot;
            }
            __syncthreads();
            ranked = !s_int[0] && M <= LY.nodes;
            nm = 0;
            if (ranked) {
                const int k0 = s_base[sr * Wq + (sc >> 6)] + __popcll(s_act[sr * Wq + (sc >> 6)] & ((1ull << (sc & 63)) - 1ull));
                for (int q = tid; q < Q; q += NT) {
                    const int r = q / Wq, w = q % Wq;
                    const SquareBits s = square_bits(s_ge, n, W, r, w);
                    unsigned long long act = s_act[q];
                    int k = s_base[q];
                    while (act) {
                        const int t = (int)__builtin_ctzll(act);
                        act &= act - 1ull;
                        const int code = (int)((s.tl >> t) & 1ull) * MS_TL + (int)((s.tr >> t) & 1ull) * MS_TR +
                                         (int)((s.bl >> t) & 1ull) * MS_BL + (int)((s.br >> t) & 1ull) * MS_BR;
                        const int d = (int)((kSquareDir >> (2 * code)) & 3u);
                        const int c = w * 64 + t;
                        const int r2 = r + (d == D_DOWN) - (d == D_UP), c2 = c + (d == D_RIGHT) - (d == D_LEFT);
                        const int q2 = r2 * Wq + (c2 >> 6);  // the move crosses an edge with an inside corner: a square of the table
                        int k2 = s_base[q2] + __popcll(s_act[q2] & ((1ull << (c2 & 63)) - 1ull));
                        if (k2 == k0) k2 = kNodeEnd;
                        s_node[k] = (uint32_t)d | ((uint32_t)c << 2) | ((uint32_t)r << 16);
                        s_hopA[k] = (uint32_t)k2 | (1u << 16);
                        ++k;
                    }
                }
                __syncthreads();
                uint32_t *a = s_hopA, *c = s_hopB;
                for (int span = 1; span < M; span <<= 1) {
                    for (int k = tid; k < M; k += NT) {
                        uint32_t h = a[k];
                        const int s = (int)(h & 0xffffu);
                        if (s != kNodeEnd) {
                            const uint32_t h2 = a[s];
                            h = (h2 & 0xffffu) | ((h & 0xffff0000u) + (h2 & 0xffff0000u));
                        }
                        c[k] = h;
                    }
                    __syncthreads();
                    uint32_t* t = a;
                    a = c;
                    c = t;
                }
                nm = __builtin_amdgcn_readfirstlane((int)(a[k0] >> 16));  // moves to the end of the start's cycle
                for (int k = tid; k < M; k += NT)
                    if ((a[k] & 0xffffu) == (uint32_t)kNodeEnd) c[nm - (int)(a[k] >> 16)] = s_node[k];
                moves = c;
                if (nm > ccap && tid == 0) s_int[3] = kErrContourCap;
                __syncthreads();
            } else {
                if (tid < 64) {
                    uint32_t* out = s_node;
                    auto inside = [&](int row, int col) -> bool {
                        const int r = row - b.y0, q = col - b.x0;
                        if ((unsigned)r >= (unsigned)n || (unsigned)q >= (unsigned)n) return false;
                        return ((s_ge[r * W + (q >> 6)] >> (q & 63)) & 1ull) != 0ull;
                    };
                    auto emit = [&](int k, uint32_t mv) { if (lane == 0) out[k] = mv; };
                    const int st = walk_squares_v(b.x0 + sc, b.y0 + sr, b.x0, b.y0, n, ccap, inside, emit, [](int, int, int) {}, &nm);
                    if (tid == 0) {
                        s_int[1] = nm;
                        if (st) s_int[3] = st;
                    }
                }
                moves = s_node;
                __syncthreads();
                nm = __builtin_amdgcn_readfirstlane(s_int[1]);
            }
            if (s_int[3]) { exists = false; break; }
            // all lanes: interpolate the moves, drop consecutive duplicates (insertPoint,
            // marchingSquares.cpp:197-203) and compact in order
            int kept = 0;
            for (int r0 = 0; r0 < nm; r0 += NT) {
                const int k = r0 + tid;
                double2 p = make_double2(0.0, 0.0);
                if (k < nm) {
                    p = move_point(C, n, n, b.x0, b.y0, moves[k]);
                    s_stage[tid + 1] = p;
                }
                __syncthreads();
                bool keep = false;
                if (k < nm) {
                    keep = true;
                    if (k > 0) {
                        const double2 q = s_stage[tid];
                        keep = (p.x != q.x || p.y != q.y);
                    }
                }
                int tot;
                const int at = kept + block_flag_scan(keep, s_tmp, &tot);
                if (keep && at < ccap) {
                    pts[at] = p;
                    if (at < LY.pts) s_pt[at] = p;
                }
                kept += tot;
                if (tid == NT - 1) s_stage[0] = p;  // the next chunk's predecessor
                __syncthreads();
            }
            // close the contour (marchingSquares.cpp:180-186)
            len = kept;
            if (len > ccap) { if (tid == 0) s_int[3] = kErrContourCap; }
            else if (len > 0) {
                const double2 f = pt(0), l = pt(len - 1);
                if (f.x != l.x || f.y != l.y) {
                    if (len < ccap && tid == 0) {
                        pts[len] = f;
                        if (len < LY.pts) s_pt[len] = f;
                    }
                    len++;
                }
                if (len > ccap && tid == 0) s_int[3] = kErrContourCap;
            }
            len = __builtin_amdgcn_readfirstlane(len);
            __syncthreads();
            if (s_int[3]) { exists = false; break; }
            // shoelace sum and perimeter (computePerimeter, grainBoundary.cpp:224-231), in contour order
            {
                const int L1 = len - 1;
                double vs = 0.0, per = 0.0;
                for (int c0 = 0; c0 < L1; c0 += NT) {
                    const int i = c0 + tid;
                    if (i < L1) {
                        const double2 a = pt(i), c2 = pt(i + 1);
                        const double dx = a.x - c2.x, dy = a.y - c2.y;
                        const double term = (a.y + c2.y) * (a.x - c2.x), ln = sqrt(dx * dx + dy * dy);
                        s_stage[tid] = make_double2(term, ln);
                        if (i < LY.pts) s_len[i] = ln;
                    }
                    __syncthreads();
                    if (tid < 64) {
                        const int m = min(NT, L1 - c0);
                        in_order<8>(m, [&](int k) { return s_stage[k]; }, [&](int, const double2& v) {
                            vs += v.x;
                            per = fma(v.y, G.h, per);
                        });
                    }
                    __syncthreads();
                }
                if (tid < 64) {  // computeVolume + isMotionRegular (box.cpp:1155-1190)
                    const double newVolume = fabs(vs) * G.h * G.h * 0.5;
                    const double mullins = (newVolume - old_vol) / G.dt * (3 / 3.14159265358979323846);
                    const double contourRatio = ((double)len) / old_len;
                    const double volumeRatio = newVolume / old_vol;
                    int regular, flag_off = 0;
                    if (mullins > -6.0) regular = 1;
                    else if (volumeRatio < 0.10) regular = 0;
                    else if (contourRatio < 0.35) regular = 0;
                    else if (contourRatio > 0.7) regular = 1;
                    else { flag_off = 1; regular = 1; }
                    if (tid == 0) {
                        s_dbl[0] = vs;
                        s_dbl[5] = per;
                        if (flag_off) s_int[4] = 0;
                        s_int[2] = regular;
                    }
                    if (!regular) {  // bounding box of the contour for clearContourGrainArea
                        const double2 f = pt(0);
                        double mnx = f.x, mxx = mnx, mny = f.y, mxy = mny;
                        for (int i = tid; i < len; i += 64) {
                            const double2 q = pt(i);
                            mnx = fmin(mnx, q.x); mxx = fmax(mxx, q.x);
                            mny = fmin(mny, q.y); mxy = fmax(mxy, q.y);
                        }
                        for (int d = 32; d >= 1; d >>= 1) {
                            mnx = fmin(mnx, __shfl_xor(mnx, d)); mxx = fmax(mxx, __shfl_xor(mxx, d));
                            mny = fmin(mny, __shfl_xor(mny, d)); mxy = fmax(mxy, __shfl_xor(mxy, d));
                        }
                        if (tid == 0) { s_dbl[1] = mnx; s_dbl[2] = mxx; s_dbl[3] = mny; s_dbl[4] = mxy; }
                    }
                }
            }
            __syncthreads();
            if (s_int[2]) break;
            if (++retries > 256) {
                if (tid == 0) s_int[3] = kErrTrace;
                exists = false;
                __syncthreads();
                break;
            }
            {  // clearContourGrainArea: i in [int(miny-1), maxy+1), j in [int(minx-1), maxx+1)
                const int i0 = (int)(s_dbl[3] - 1), j0 = (int)(s_dbl[1] - 1);
                const double maxy = s_dbl[4], maxx = s_dbl[2];
                int ih = 0, jw = 0;
                while (i0 + ih < maxy + 1) ih++;
                while (j0 + jw < maxx + 1) jw++;
                for (int p = tid; p < ih * jw; p += NT) {
                    const int ii = i0 + p / jw, jj = j0 + p % jw;
                    const long long k = flat_index(ii, jj, b.x0, b.y0, n, nn);
                    if (k < 0) { s_int[3] = kErrClearBounds; continue; }
                    const int kr = (int)(k / n), kc = (int)(k % n);
                    const unsigned bit = 1u << (kc & 31);
                    unsigned* word = (unsigned*)(s_ge + kr * W) + (kc >> 5);
                    if (*word & bit) {  // C >= 0: below zero from here on, in every plane
                        C[k] = (T)(-G.h);
                        if (A.rec_win) A.rec_win[o + k] = -2;
                        atomicAnd(word, ~bit);
                    }
                }
                __syncthreads();
                // the planes of the cleared field, written whole with plain stores (an atomic on memory
                // another die's L2 may hold a line of would leave that line stale for k_redist)
                for (int k = tid; k < n * W; k += NT) {
                    const unsigned long long ge = s_ge[k];
                    bits[kRowGe * A.plane + k] = ge;
                    bits[kRowGt * A.plane + k] &= ge;
                    const int col = k / W, w = k - col * W;
                    unsigned long long cge = 0;
                    for (int t = 0; t < 64 && w * 64 + t < n; ++t)
                        cge |= ((s_ge[(w * 64 + t) * W + (col >> 6)] >> (col & 63)) & 1ull) << t;
                    bits[kColGe * A.plane + k] = cge;
                    bits[kColGt * A.plane + k] &= cge;
                }
                __syncthreads();
                if (s_int[3]) { exists = false; break; }
            }
        }
        if (tid == 0) {
            int f = A.O.flags[g];
            f = s_int[4] ? (f | kRegular) : (f & ~kRegular);
            if (!exists) f &= ~kExists;
            if constexpr (COARSEN) {
                if (exists) f |= kExists;  // a contour on the new grid: the grain exists again
                A.O.off_next[g] = o;
            }
            A.O.flags[g] = f;
            if (s_int[3]) A.O.err[g] = s_int[3];
            A.O.box_next[g] = b;
            A.O.coff[g] = s_coff;
            A.O.ccap[g] = ccap;
            if (exists) A.O.clen[g] = len;
        }
        if (!exists) continue;
        if constexpr (ANISO) {
            // ---------------- junctions of the final contour ----------------
            // generateJunction (marchingSquares.cpp:266-301) at every square the walk passes whose
            // four corners lie in the box: three or more distinct grains among the corners (the
            // grain itself where inside, else IDLocal's) make a junction at the square's centre,
            // projected onto the contour afterwards (grainBoundary.cpp:50-61).  Recorded in walk
            // order, 64 squares at a time: a ranked walk's squares are its moves; a walked one is
            // walked again (its saddles are passed without a move).
            const uint32_t* idn = A.idl_new + o;
            Junc* jdst = A.AS.junc + (size_t)g * kJuncCap;
            auto record = [&](bool valid, uint32_t mv, int jn) -> int {  // one wave; the junctions so far
                int order = 0;
                uint32_t gr[4] = {0xFFFFFFu, 0xFFFFFFu, 0xFFFFFFu, 0xFFFFFFu};
                const int c = (int)((mv >> 2) & 0x3fffu), r = (int)(mv >> 16);
                if (valid && r >= 1 && r <= n - 1 && c >= 1 && c <= n - 1) {
                    auto in = [&](int row, int col) -> bool { return ((s_ge[row * W + (col >> 6)] >> (col & 63)) & 1ull) != 0ull; };
                    const bool tl = in(r - 1, c - 1), tr = in(r - 1, c), bl = in(r, c - 1), br = in(r, c);
                    if ((int)tl + (int)tr + (int)bl + (int)br < 3) {  // three inside corners leave at most two grains
                        auto ins = [&](uint32_t v) {
                            for (int k = 0; k < order; ++k)
                                if (gr[k] == v) return;
                            gr[order++] = v;
                        };
                        const uint32_t* q = idn + (long long)(r - 1) * n + (c - 1);
                        ins(bl ? (uint32_t)g : q[n]);
                        ins(tl ? (uint32_t)g : q[0]);
                        ins(br ? (uint32_t)g : q[n + 1]);
                        ins(tr ? (uint32_t)g : q[1]);
                    }
                }
                const unsigned long long m = __ballot(order > 2);
                if (order > 2) {
                    const int at = jn + __popcll(m & ((1ull << lane) - 1ull));
                    if (at < kJuncCap) {
                        Junc J;
                        J.x = (b.x0 + c - 1) + 0.5; J.y = (b.y0 + r - 1) + 0.5; J.lambda = 0.0; J.seg = -1; J.order = order;
                        for (int k = 0; k < 4; ++k) J.gr[k] = gr[k];
                        jdst[at] = J;
                    }
                }
                return jn + __popcll(m);
            };
            if (tid < 64) {
                int jn = 0;
                if (ranked) {
                    for (int c0 = 0; c0 < nm; c0 += 64) jn = record(c0 + lane < nm, c0 + lane < nm ? moves[c0 + lane] : 0u, jn);
                } else {
                    uint32_t* s_visit = (uint32_t*)s_stage;
                    int nv = 0, dummy = 0;
                    auto inside = [&](int row, int col) -> bool {
                        const int r = row - b.y0, q = col - b.x0;
                        if ((unsigned)r >= (unsigned)n || (unsigned)q >= (unsigned)n) return false;
                        return ((s_ge[r * W + (q >> 6)] >> (q & 63)) & 1ull) != 0ull;
                    };
                    auto visit = [&](int left, int top, int) {
                        if (lane == 0) s_visit[nv] = ((uint32_t)(left - b.x0 + 1) << 2) | ((uint32_t)(top - b.y0 + 1) << 16);
                        if (++nv == 64) {
                            wave_lds_sync();
                            jn = record(true, s_visit[lane], jn);
                            wave_lds_sync();
                            nv = 0;
                        }
                    };
                    (void)walk_squares_v(b.x0 + start_col, b.y0 + start_row, b.x0, b.y0, n, ccap, inside,
                                         [](int, uint32_t) {}, visit, &dummy);
                    wave_lds_sync();
                    jn = record(lane < nv, lane < nv ? s_visit[lane] : 0u, jn);
                }
                if (tid == 0) {
                    s_int[10] = jn;
                    A.AS.jcnt[g] = min(jn, kJuncCap);
                    if (jn > kJuncCap) A.O.err[g] = kErrJuncCap;
                }
            }
            __syncthreads();
            const int jn = min(s_int[10], kJuncCap);
            // a wave per junction: the nearest vertex (the first of the nearest in contour order), then
            // the segment part of the projection
            for (int k = tid >> 6; k < jn; k += NT / 64) {
                Junc J = jdst[k];
                const double nearest = wave_nearest_vertex(pt, len, J.x, J.y);
                double lambda = 0.0;
                const int seg = segment_at(pts, len, nearest < 1e8 ? (int)nearest : -1, J.x, J.y, &lambda);
                if (seg < 0) {
                    if (lane == 0) A.O.err[g] = kErrAniso;
                    continue;
                }
                const int nxt = (seg + 1 + (len - 1)) % (len - 1);  // PERIODIC (grainBoundary.cpp:27)
                J.x = lerp_nc(pts[seg].x, pts[nxt].x, lambda);
                J.y = lerp_nc(pts[seg].y, pts[nxt].y, lambda);
                J.seg = seg;
                J.lambda = lambda;
                if (lane == 0) jdst[k] = J;
            }
            __syncthreads();
        }
        // ---------------- new box (box.cpp:1118-1148); k_alloc gives it room ----------------
        if (!COARSEN && tid == 0) {
            const bool any = bb_x1 >= 0;
            const int ixmin = any ? b.x0 + bb_x0 : b.x0 + n, ixmax = any ? b.x0 + bb_x1 : b.x0;
            const int iymin = any ? b.y0 + bb_y0 : b.y0 + n, iymax = any ? b.y0 + bb_y1 : b.y0;
            int nXMin = ixmin - G.gb, nXMax = ixmax + G.gb, nYMin = iymin - G.gb, nYMax = iymax + G.gb;
            if (nXMin >= nXMax || nYMin >= nYMax) { nXMin = b.x0; nXMax = b.x0 + n; nYMin = b.y0; nYMax = b.y0 + n; }
            const int m = G.m;
            if (nXMin < 0) nXMin = 0;
            if (nYMin < 0) nYMin = 0;
            if (nXMax > m) nXMax = m;
            if (nYMax > m) nYMax = m;
            int xmin = nXMin, xmax = nXMax, ymin = nYMin, ymax = nYMax;
            const int grid_size = m - 1;
            const unsigned int height = (unsigned int)(ymax - ymin), width = (unsigned int)(xmax - xmin);
            if (width != height) {
                if (width > height) { int diff = (int)(width - height); ymin -= diff / 2; ymax += diff / 2 + diff % 2; }
                else { int diff = (int)(height - width); xmin -= diff / 2; xmax += diff / 2 + diff % 2; }
                if (xmin < 0) { int dl = -xmin; xmax += dl; xmin += dl; }
                else if (xmax > grid_size) { int dl = grid_size - xmax; xmax += dl; xmin += dl; }
                if (ymin < 0) { int dl = -ymin; ymax += dl; ymin += dl; }
                else if (ymax > grid_size) { int dl = grid_size - ymax; ymax += dl; ymin += dl; }
            }
            Box nbx;
            nbx.x0 = xmin; nbx.y0 = ymin; nbx.n = xmax - xmin; nbx.pad = ymax - ymin;
            A.O.box_next[g] = nbx;
        }
        const int L1 = len - 1;
        // ---------------- direct neighbours (only after a regular motion) ----------------
        const bool nbs = !COARSEN && s_int[4] != 0;
        if (tid == 0) s_int[9] = L1;  // first failed probe (none yet)
        __syncthreads();
        if (nbs) {  // one probe pixel per contour point (buildDirectNeighbours, grainBoundary.cpp:85-120)
            int fail = L1;
            for (int i = tid; i < L1; i += NT) {
                const double2 p = pt(i);
                int pxGrid = (int)p.x, pyGrid = (int)p.y;
                int cand = -1;
                bool ok = true;
                auto above = [&](long long k) -> bool {  // C > 0
                    const int kr = (int)(k / n), kc = (int)(k % n);
                    return ((bits[kRowGt * A.plane + (long long)kr * W + (kc >> 6)] >> (kc & 63)) & 1ull) != 0ull;
                };
                long long k = flat_index(pyGrid, pxGrid, b.x0, b.y0, n, nn);
                if (k < 0) ok = false;
                else if (above(k)) {
                    pxGrid = (int)(p.x + 1);
                    k = flat_index(pyGrid, pxGrid, b.x0, b.y0, n, nn);
                    if (k < 0) ok = false;
                    else if (above(k)) {
                        pyGrid = (int)(p.y + 1);
                        k = flat_index(pyGrid, pxGrid, b.x0, b.y0, n, nn);
                        if (k < 0) ok = false;
                        else if (above(k)) pxGrid = (int)p.x;
                    }
                }
                if (ok) {
                    if (pyGrid < 0 || pyGrid >= b.y0 + n || pxGrid < 0 || pxGrid >= b.x0 + n) ok = false;
                    else {
                        k = flat_index(pyGrid, pxGrid, b.x0, b.y0, n, nn);
                        if (k < 0) ok = false;
                        else {
                            const uint32_t nid = A.idl_new[o + k];
                            if (nid == 0u) cand = 0;
                            else if (nid < (uint32_t)G.nslots && (A.O.flags[nid] & kPresent)) cand = (int)nid;
                            else ok = false;
                        }
                    }
                }
                s_cand[i] = ok ? cand : -1;
                if (!ok) fail = min(fail, i);
            }
            if (fail < L1) atomicMin(&s_int[9], fail);
        }
        __syncthreads();
        if (tid < 64) {
            const int stop = __builtin_amdgcn_readfirstlane(nbs ? s_int[9] : L1);
            const double h = G.h;
            if (lane == 0) A.O.perimeter[g] = s_dbl[5];
            if (nbs) {
                // the neighbours in first-encounter order (lane e holds neighbour e), and each point's slot
                int my_id = -1, cnt2 = 0, over = 0;
                for (int c0 = 0; c0 < stop; c0 += 64) {
                    const int i = c0 + lane;
                    const int cv = i < stop ? s_cand[i] : -1;
                    int slot = -1;
                    unsigned long long left = __ballot(i < stop);
                    while (left) {
                        const int cd = __builtin_amdgcn_readlane(cv, (int)__builtin_ctzll(left));
                        const unsigned long long known = __ballot(my_id == cd);
                        int e = kNbCap;
                        if (known) e = (int)__builtin_ctzll(known);
                        else if (cnt2 < kNbCap) {
                            e = cnt2++;
                            if (lane == e) my_id = cd;
                        } else over = 1;
                        if (cv == cd) slot = e;
                        left &= ~__ballot(i < stop && cv == cd);
                    }
                    if (i < stop) s_cand[i] = slot;
                }
                double my_e = 0.0, my_m = 0.0;
                if constexpr (ANISO) {  // characteristics: energy density and mobility of the boundary
                    if (lane < cnt2) {
                        const double th = misorientation(A.AS.quat[g], A.AS.quat[my_id]);
                        my_e = gb_energy(A.K, th);
                        my_m = gb_mobility(A.K, th);
                    }
                    s_nbe[lane] = my_e;
                }
                wave_lds_sync();
                // the lengths per neighbour up to the first failed probe, and the energy (computeEnergy,
                // grainBoundary.cpp:215-222): the segments from that probe on keep the -1 of a fresh SPoint.
                // Without a failed probe the isotropic energy is the perimeter's sum, term by term.
                double my_len = 0.0, e = 0.0;
                const bool whole = !ANISO && stop == L1;
                for (int c0 = 0; c0 < L1; c0 += 64) {
                    const int i = c0 + lane;
                    double lv = 0.0, ev = -1.0;
                    if (i < L1) {
                        if (i < LY.pts) lv = s_len[i];
                        else {
                            const double2 a = pt(i), c2 = pt(i + 1);
                            const double dx = a.x - c2.x, dy = a.y - c2.y;
                            lv = sqrt(dx * dx + dy * dy);
                        }
                        if (i < stop) {
                            if constexpr (ANISO) {
                                const int sl = s_cand[i];
                                // a neighbour beyond the list's capacity has no slot (the grain reports it)
                                ev = s_nbe[sl < kNbCap ? sl : 0];
                            } else ev = 1.0;
                        }
                    }
                    s_stage[lane] = make_double2(lv, ANISO ? lv * ev : 0.0);
                    wave_lds_sync();
                    const int m = min(64, L1 - c0), ms = min(m, stop - c0);
                    struct Term { double2 v; int slot; };
                    in_order<8>(ms, [&](int k) { return Term{s_stage[k], s_cand[c0 + k]}; }, [&](int, const Term& q) {
                        const double longer = fma(q.v.x, h, my_len);
                        my_len = q.slot == lane ? longer : my_len;
                        if constexpr (ANISO) e = fma(q.v.y, h, e);
                    });
                    if constexpr (ANISO) {
                        const int from = max(ms, 0);
                        in_order<8>(m - from, [&](int k) { return s_stage[from + k].y; }, [&](int, double v) { e = fma(v, h, e); });
                    } else if (!whole) {
                        in_order<8>(m, [&](int k) { return s_stage[k].x; },
                                    [&](int k, double v) { e = fma(c0 + k >= stop ? -v : v, h, e); });
                    }
                    wave_lds_sync();
                }
                if (whole) e = s_dbl[5];
                if (lane < cnt2) {
                    A.O.nb_id[(size_t)g * kNbCap + lane] = my_id;
                    A.O.nb_len[(size_t)g * kNbCap + lane] = my_len;
                    if constexpr (ANISO) {
                        A.AS.nb_e[(size_t)g * kNbCap + lane] = my_e;
                        A.AS.nb_m[(size_t)g * kNbCap + lane] = my_m;
                    }
                }
                if (lane == 0) {
                    A.O.energy[g] = e;
                    A.O.nb_cnt[g] = cnt2;
                    if (over) A.O.err[g] = kErrNbCap;
                    if (stop < L1) A.O.flags[g] &= ~kRegular;  // markAsInvalidMotion
                    double newVolume = fabs(fabs(s_dbl[0]) * G.h * G.h * 0.5);
                    double dA = newVolume - old_vol;
                    dA = dA / G.dt;
                    dA = dA * (3 / 3.14159265358979323846);
                    A.O.volume[g] = newVolume;
                    if (A.rec_area) A.rec_area[g] = 1;
                    unsigned int lp = (unsigned int)*A.loop;
                    unsigned long at = A.analysis_timestep > 0 ? (unsigned long)A.analysis_timestep : 1ul;
                    double md = A.O.meanda[g];
                    if ((unsigned long)(lp - 1u) % at == 0 || lp == 0) md = 0;
                    A.O.meanda[g] = md + dA;
                }
            }
        }
    }
}

// Room in the next field arena for the new box of every grain that exists after the contour: one
// scan and one atomic per 256 grains (a same-address atomic per grain would serialise across the
// chip).  A grain that finds no room leaves the step.
__global__ void __launch_bounds__(256) k_alloc(const int* __restrict__ list, const int* __restrict__ count, ContourOut O,
                                               unsigned long long* __restrict__ out_total) {
    __shared__ int s_tmp[4];
    __shared__ unsigned long long s_first;
    const int total = *count;
    for (int i0 = (int)blockIdx.x * 256; i0 < total; i0 += (int)gridDim.x * 256) {
        const int i = i0 + (int)threadIdx.x;
        int g = 0, n = 0;
        if (i < total) {
            g = list[i];
            if (O.flags[g] & kExists) n = O.box_next[g].n;
        }
        const int need = (int)(((long long)n * n + kAlign - 1) / kAlign);  // in units of kAlign
        int sum, area;
        const int at = block_scan(need, s_tmp, &sum);
        (void)block_scan(n * n, s_tmp, &area);
        if (threadIdx.x == 0) {
            s_first = atomicAdd(&O.tops[0], (unsigned long long)sum * kAlign);
            if (area) atomicAdd(out_total, (unsigned long long)area);
        }
        __syncthreads();
        if (n > 0) {
            const unsigned long long fo = s_first + (unsigned long long)at * kAlign;
            if ((long long)(fo + (unsigned long long)need * kAlign) > O.field_cap) {  // no field space
                O.err[g] = kErrArena;
                O.flags[g] &= ~kExists;
            }
            O.off_next[g] = (long long)fo;
        }
        __syncthreads();
    }
}

// One redistancing sweep along a line of cells t = 0..L in sweep order (box.cpp:1291-1388):
// step t carries cur (cell t) into nxt (cell t + 1); while t < tIn both cells lie in the old box
// and the candidate takes the sign of the compared field at cell t + 1, else the sign of nxt.
// Forward sweeps (CROSS) first move cur onto an interface crossing between cells t and t + 1.
// oload / ostore / cload address the line's output and compared field.  The line is processed
// in chunks of kCh steps whose inputs are loaded together; the divisions of the crossings of a
// chunk run in wave-wide rounds (one per crossing of the busiest lane), not at every step a lane
// crosses.  Every lane of the wave calls this with the same L and tIn.
template <class T, bool CROSS, class OL, class OS, class CL>
__device__ __forceinline__ void sweep_line(OL oload, OS ostore, CL cload, int L, int tIn, bool active, bool cvalid,
                                           double h) {
    constexpr int kCh = 4;
    if (L <= 0) return;
    const int tI = cvalid ? tIn : 0;
    T cur = active ? oload(0) : T(0);
    double cprev = (CROSS && active && tI > 0) ? (double)cload(0) : 0.0;
    for (int tb = 0; tb < L; tb += kCh) {
        T ov[kCh];
        double cv[kCh];
#pragma unroll
        for (int q = 0; q < kCh; ++q) {
            const int t1 = tb + 1 + q;
            ov[q] = (active && t1 <= L) ? oload(t1) : T(0);
            cv[q] = (active && t1 <= tI) ? (double)cload(t1) : 0.0;
        }
        double dd[kCh], ss[kCh];
        if constexpr (CROSS) {
            unsigned cm = 0u;
#pragma unroll
            for (int q = 0; q < kCh; ++q) {
                const int t = tb + q;
                const double a = q == 0 ? cprev : cv[q - 1];
                if (active && t < L && t < tI && a * cv[q] <= 0.0) cm |= 1u << q;
                dd[q] = 0.0;
                ss[q] = 0.0;
            }
            while (__ballot(cm != 0u) != 0ull) {
                if (cm != 0u) {
                    const int q = __builtin_ctz(cm);
                    double a = cprev, a1 = cv[0];
#pragma unroll
                    for (int r = 1; r < kCh; ++r)
                        if (r == q) { a = cv[r - 1]; a1 = cv[r]; }
                    const double slope = (a1 - a) / h;
                    const double d0 = -a / slope;
                    const double sg = (double)sgn_of(slope);
#pragma unroll
                    for (int r = 0; r < kCh; ++r)
                        if (r == q) { dd[r] = d0; ss[r] = sg; }
                    cm &= cm - 1u;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kCh; ++q) {
            const int t = tb + q;
            if (active && t < L) {
                T nxt = ov[q];
                double cand;
                if (t < tI) {
                    if constexpr (CROSS) {
                        const double a = q == 0 ? cprev : cv[q - 1];
                        if (a * cv[q] <= 0.0) {
                            if (fabs((double)cur) > fabs(dd[q])) { cur = (T)(-dd[q] * ss[q]); ostore(t, cur); }
                        }
                    }
                    cand = (double)cur + (sgn_of(cv[q]) * h);
                } else {
                    cand = (double)cur + (sgn_of(nxt) * h);
                }
                if (fabs(cand) < fabs((double)nxt)) { nxt = (T)cand; ostore(t + 1, nxt); }
                cur = nxt;
            }
        }
        if constexpr (CROSS) cprev = cv[kCh - 1];
    }
}

// LSbox::executeRedistancing (box.cpp:1259-1399) of one grain in place in the output arena, for what
// does not fit k_redist's tile: Ob is the grain's slot (row pitch `pitch`), C the compared field on the
// old box b (row pitch cp), bo the new box.  Lanes own columns (y sweeps) or rows (x sweeps); the value carried
// along a sweep stays in a register and the next line's inputs are loaded one step ahead (a
// sweep step only writes its own two lines, so the early loads see final values).
template <class T>
__device__ __forceinline__ void redistance(T* Ob, int pitch, const T* C, int cp, Box b, Box bo, const GridConst& G,
                                           T* gout) {
    const int n = b.n, no = bo.n;
    const double h = G.h;
    const int oxmin = bo.x0, oxmax = bo.x0 + no, oymin = bo.y0, oymax = bo.y0 + no;
    const int ixmn = b.x0, ixmx = b.x0 + n, iymn = b.y0, iymx = b.y0 + n;
    const int ixmin = ixmn < oxmin ? oxmin : ixmn;
    const int iymin = iymn < oymin ? oymin : iymn;
    const int ixmax = ixmx < oxmax ? ixmx : oxmax;
    const int iymax = iymx < oymax ? iymx : oymax;
#define OV(i, j) Ob[((i) - oymin) * pitch + ((j) - oxmin)]
#define CI(i, j) C[((i) - iymn) * cp + ((j) - ixmn)]
    for (int p = threadIdx.x; p < no * no; p += blockDim.x) {
        int yy = p / no, xx = p - yy * no;
        Ob[yy * pitch + xx] = T(-1.0);
    }
    __syncthreads();
    // y forward (box.cpp:1291-1319), y backward (1321-1338): lanes own columns
    for (int j0 = ixmin; j0 < oxmax; j0 += blockDim.x) {
        if (j0 + (int)(threadIdx.x & ~63u) >= oxmax) continue;  // a wave without a line skips the sweep
        const int j = j0 + (int)threadIdx.x;
        const bool act = j < oxmax, colin = j < ixmax;
        sweep_line<T, true>([&](int t) { return OV(iymin + t, j); }, [&](int t, T v) { OV(iymin + t, j) = v; },
                            [&](int t) { return CI(iymin + t, j); }, oymax - 1 - iymin, iymax - 1 - iymin, act, colin, h);
    }
    __syncthreads();
    for (int j0 = ixmin; j0 < oxmax; j0 += blockDim.x) {
        if (j0 + (int)(threadIdx.x & ~63u) >= oxmax) continue;
        const int j = j0 + (int)threadIdx.x;
        const bool act = j < oxmax, colin = j < ixmax;
        sweep_line<T, false>([&](int t) { return OV(iymax - 1 - t, j); }, [&](int t, T v) { OV(iymax - 1 - t, j) = v; },
                             [&](int t) { return CI(iymax - 1 - t, j); }, iymax - 1 - oymin, iymax - 1 - iymin, act, colin, h);
    }
    __syncthreads();
    // x forward (1339-1367), x backward (1369-1388): lanes own rows
    for (int i0 = iymin; i0 < oymax; i0 += blockDim.x) {
        if (i0 + (int)(threadIdx.x & ~63u) >= oymax) continue;
        const int i = i0 + (int)threadIdx.x;
        const bool act = i < oymax, rowin = i < iymax;
        sweep_line<T, true>([&](int t) { return OV(i, ixmin + t); }, [&](int t, T v) { OV(i, ixmin + t) = v; },
                            [&](int t) { return CI(i, ixmin + t); }, oxmax - 1 - ixmin, ixmax - 1 - ixmin, act, rowin, h);
    }
    __syncthreads();
    for (int i0 = iymin; i0 < oymax; i0 += blockDim.x) {
        if (i0 + (int)(threadIdx.x & ~63u) >= oymax) continue;
        const int i = i0 + (int)threadIdx.x;
        const bool act = i < oymax, rowin = i < iymax;
        sweep_line<T, false>([&](int t) { return OV(i, ixmax - 1 - t); }, [&](int t, T v) { OV(i, ixmax - 1 - t) = v; },
                             [&](int t) { return CI(i, ixmax - 1 - t); }, ixmax - 1 - oxmin, ixmax - 1 - ixmin, act, rowin, h);
    }
    __syncthreads();
#undef OV
#undef CI
    // clampValues (dimensionalBufferReal.h:43-56)
    const T lo = (T)(-G.delta), hi = (T)G.delta;
    for (int p = threadIdx.x; p < no * no; p += blockDim.x) {
        int yy = p / no, xx = p - yy * no;
        T v = Ob[yy * pitch + xx];
        if (v < lo) v = lo;
        else if (v > hi) v = hi;
        gout[p] = v;
    }
}

// ------------------------------------------------------------------------------------------
// k_redist: LSbox::executeRedistancing of one grain per workgroup, one line per lane, the new
// field in an LDS tile (odd pitch, so that columns and rows are both free of bank conflicts).
//
// The four sweeps are chains of dependent steps, so a step is kept short: the sign of the compared
// field comes from the line's bit words (one shift and one merge into the sign of h), and the
// interface distances -- two FP64 divisions each -- are computed before a sweep for all crossings
// of all lines at once, 64 to an instruction, into a list each line reads in order.  Every cell
// is read and written once per sweep.  Boxes above the tile, and fields with more crossings than
// the list holds, take `redistance`, which sweeps in place in the output arena.
// ------------------------------------------------------------------------------------------
constexpr int kTileMargin = 3;  // the tile holds new boxes up to the launch's largest side plus this

__host__ __device__ inline int redist_crossings(int tile) { return 4 * tile + 64; }

template <class T>
__host__ __device__ inline long long redist_lds(int tile) {
    if (tile <= 0) return 0;
    return (long long)redist_crossings(tile) * 8 + (((long long)tile * (tile | 1) * (long long)sizeof(T) + 15) & ~15LL);
}

// 32 bits of a line from bit 32 w on (`words` 32-bit words per line; zero outside).
__device__ __forceinline__ uint32_t line_word(const uint32_t* line, int w, int words) {
    return (unsigned)w < (unsigned)words ? line[w] : 0u;
}

// Crossings of a line between its cells c and c + 1 for the 32 cells of word w: the product of the
// two values is not positive (signs from the bits; a product of two values of one sign would have
// to underflow to differ, and the fields are sums of terms of the order of delta).
__device__ __forceinline__ uint32_t line_crossings(const uint32_t* ge, const uint32_t* gt, int w, int words, int lo, int hi) {
    const uint32_t g0 = line_word(ge, w, words), p0 = line_word(gt, w, words);
    const uint32_t g1 = (g0 >> 1) | (line_word(ge, w + 1, words) << 31), p1 = (p0 >> 1) | (line_word(gt, w + 1, words) << 31);
    uint32_t x = ~((p0 & p1) | (~g0 & ~g1));
    const int a = lo - 32 * w, e = hi - 32 * w;  // cells [lo, hi)
    if (a > 0) x = a < 32 ? x & (~0u << a) : 0u;
    if (e < 32) x = e > 0 ? x & ((1u << e) - 1u) : 0u;
    return x;
}

// One sweep of a line: cells t = 0 .. L from `cell` on, `stride` elements apart; steps t < tI take
// the sign of the compared field at cell t + 1, whose index along the line is idx0 + dir (t + 1),
// the others the sign of the cell itself (box.cpp:1291-1388).  FRESH: every cell still holds the
// initial -1.  CROSS (dir = 1): cur first moves onto the crossing between cells t and t + 1, the
// next of the line's list.  `in`: the line lies in the old box (else the cell's own sign counts
// everywhere).  All lanes of the wave have the same L, tI and idx0; lanes without a line (act =
// false) address a line of their own that they leave alone.
template <class T, int DIR, bool CROSS, bool FRESH>
__device__ __forceinline__ void bit_sweep(T* cell, int stride, int L, int tI, int idx0, bool act, bool in,
                                          const uint32_t* ge, const uint32_t* gt, int words, const double* next, double h) {
    if (L < 0 || (L == 0 && !FRESH) || __ballot(act) == 0ull) return;
    const bool own_sign = !FRESH && __ballot(act && !in) != 0ull;  // some line of the wave lies outside the old box
    if (tI < 0) tI = 0;
    if (tI > L) tI = L;
    T cur = FRESH ? T(-1.0) : (act ? cell[0] : T(-1.0));
    double cross = 0.0;
    if (CROSS && act && in) cross = *next;  // the list has a spare entry behind the last line's
    int t = 0;
    const long long hb = __double_as_longlong(h);
    while (t < tI) {
        // the steps whose cell lies in one 32-bit word of the line
        const int c0 = idx0 + DIR * t, w = c0 >> 5;
        const int tend = min(tI, DIR > 0 ? t + 32 - (c0 & 31) : t + (c0 & 31) + 1);
        uint32_t neg = ~0u, zero = 0u, x = 0u;  // bit k: cell t + 1 of the step whose cell t is index 32 w + k
        if (act && in) {
            const uint32_t g0 = line_word(ge, w, words), p0 = line_word(gt, w, words);
            uint32_t g1, p1;
            if (DIR > 0) {
                g1 = (g0 >> 1) | (line_word(ge, w + 1, words) << 31);
                p1 = (p0 >> 1) | (line_word(gt, w + 1, words) << 31);
            } else {
                g1 = (g0 << 1) | (line_word(ge, w - 1, words) >> 31);
                p1 = (p0 << 1) | (line_word(gt, w - 1, words) >> 31);
            }
            neg = ~g1;
            zero = g1 & ~p1;
            if (CROSS) x = ~((p0 & p1) | (~g0 & ~g1));
        }
        const bool any_zero = __ballot(zero != 0u) != 0ull;
        while (t < tend) {
            constexpr int kU = 4;
            T nx[kU];
#pragma unroll
            for (int q = 0; q < kU; ++q)
                nx[q] = (!FRESH && act && t + q < tend) ? cell[(long long)(t + q + 1) * stride] : T(-1.0);
#pragma unroll
            for (int q = 0; q < kU; ++q) {
                if (t + q < tend) {
                    const int k = (idx0 + DIR * (t + q)) & 31;
                    if (CROSS) {
                        const bool hit = ((x >> k) & 1u) != 0u;
                        if (__ballot(hit)) {
                            if (hit) {
                                if (fabs((double)cur) > fabs(cross)) cur = (T)cross;
                                cross = *++next;
                            }
                        }
                    }
                    if ((CROSS || FRESH) && act) cell[(long long)(t + q) * stride] = cur;
                    double hs = __longlong_as_double(hb | (long long)((unsigned long long)((neg >> k) & 1u) << 63));
                    if (any_zero && ((zero >> k) & 1u)) hs = 0.0;
                    if (own_sign && !in) hs = sgn_of(nx[q]) * h;
                    const double cand = (double)cur + hs;
                    T nxt = nx[q];
                    if (fabs(cand) < fabs((double)nxt)) nxt = (T)cand;
                    cur = nxt;
                    if (!(CROSS || FRESH) && act) cell[(long long)(t + q + 1) * stride] = cur;
                }
            }
            t = min(t + kU, tend);
        }
    }
    for (; t < L; ++t) {
        const T nx = (!FRESH && act) ? cell[(long long)(t + 1) * stride] : T(-1.0);
        if ((CROSS || FRESH) && act) cell[(long long)t * stride] = cur;
        const double cand = (double)cur + (sgn_of(nx) * h);
        T nxt = nx;
        if (fabs(cand) < fabs((double)nxt)) nxt = (T)cand;
        cur = nxt;
        if (!(CROSS || FRESH) && act) cell[(long long)(t + 1) * stride] = cur;
    }
    if ((CROSS || FRESH) && act) cell[(long long)L * stride] = cur;
}

// The crossings of every lane's line (cells lo .. hi of the line's bits, where `in`) into list, line
// after line: first their places, then for all of them at once the value -(-a / slope) sgn(slope)
// the sweep puts on the cell before the crossing (box.cpp:1300-1309).  value(line, c) reads C at
// cell c of the line.  Returns the lane's first entry, or null when the list is too short.
template <class V>
__device__ __forceinline__ const double* list_crossings(double* list, int room, int line, bool in, const uint32_t* ge,
                                                        const uint32_t* gt, int words, int lo, int hi, double h, int* s_tmp,
                                                        V value) {
    int c = 0;
    if (in)
        for (int w = lo >> 5; w * 32 < hi; ++w) c += __popc(line_crossings(ge, gt, w, words, lo, hi));
    int total;
    const int first = block_scan(c, s_tmp, &total);
    if (total >= room) return nullptr;
    long long* places = (long long*)list;
    if (in) {
        int k = first;
        for (int w = lo >> 5; w * 32 < hi; ++w) {
            uint32_t x = line_crossings(ge, gt, w, words, lo, hi);
            while (x) {
                places[k++] = ((long long)line << 32) | (long long)(w * 32 + __builtin_ctz(x));
                x &= x - 1u;
            }
        }
    }
    __syncthreads();
    for (int k = (int)threadIdx.x; k < total; k += (int)blockDim.x) {
        const long long pl = places[k];
        const int ln = (int)(pl >> 32), cell = (int)(pl & 0xffffffffLL);
        const double a = value(ln, cell), a1 = value(ln, cell + 1);
        const double slope = (a1 - a) / h;
        const double d0 = -a / slope;
        list[k] = -d0 * (double)sgn_of(slope);
    }
    if (threadIdx.x == 0) list[total] = 0.0;  // read ahead behind the last crossing
    __syncthreads();
    return list + first;
}

template <class T, int NT>
__global__ void __launch_bounds__(NT) k_redist(LevelArgs<T> A) {
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    __shared__ int s_tmp[4];
    const GridConst& G = A.G;
    const double h = G.h;
    const int tid = (int)threadIdx.x;
    double* list = (double*)smem;
    const int room = redist_crossings(A.tile);
    T* tile = (T*)(list + room);
    const int total = items_total(A.it);
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        __syncthreads();  // the previous grain's tile is free
        int bucket, pos;
        const int g = item_grain(A.it, item, &bucket, &pos);
        if (!(sload(A.O.flags + g) & kExists)) continue;  // vanished, or no room for its field
        const Box b = sload_box(A.box + g), bo = sload_box(A.O.box_next + g);
        const int n = b.n, no = bo.n, W = (n + 63) >> 6, words = 2 * W;
        const long long o = sload(A.off + g);
        const T* C = A.cfield + o;
        T* gout = A.out_field + sload(A.O.off_next + g);
        const unsigned long long* bits = A.bits + (o >> 3);
        const int ixmin = max(b.x0, bo.x0), ixmax = min(b.x0 + n, bo.x0 + no);
        const int iymin = max(b.y0, bo.y0), iymax = min(b.y0 + n, bo.y0 + no);
        const int oxmax = bo.x0 + no, oymax = bo.y0 + no;
        bool done = false;
        if (no <= A.tile && no <= NT) {
            const int pitch = no | 1;
            if (ixmin > bo.x0 || iymin > bo.y0 || ixmin >= oxmax || iymin >= oymax)  // cells no forward y sweep passes
                for (int p = tid; p < no * pitch; p += NT) tile[p] = T(-1.0);
            // columns: y forward (box.cpp:1291-1319), y backward (1321-1338)
            {
                const int j = bo.x0 + tid;
                const bool act = tid < no && j >= ixmin, in = act && j < ixmax;
                const int col = in ? j - b.x0 : 0;
                const uint32_t* ge = (const uint32_t*)(bits + kColGe * A.plane + (long long)col * W);
                const uint32_t* gt = (const uint32_t*)(bits + kColGt * A.plane + (long long)col * W);
                const int lo = iymin - b.y0, hi = iymax - 1 - b.y0;
                const double* next = list_crossings(list, room, col, in && hi > lo, ge, gt, words, lo, hi, h, s_tmp,
                                                    [&](int ln, int c) { return (double)C[(long long)c * n + ln]; });
                if (next) {
                    done = true;
                    T* cell = tile + (long long)(iymin - bo.y0) * pitch + (act ? tid : 0);
                    bit_sweep<T, 1, true, true>(cell, pitch, oymax - 1 - iymin, iymax - 1 - iymin, lo, act, in, ge, gt, words, next, h);
                    __syncthreads();
                    cell = tile + (long long)(iymax - 1 - bo.y0) * pitch + (act ? tid : 0);
                    bit_sweep<T, -1, false, false>(cell, -pitch, iymax - 1 - bo.y0, iymax - 1 - iymin, hi, act, in, ge, gt, words, nullptr, h);
                }
            }
            __syncthreads();
            // rows: x forward (1339-1367), x backward (1369-1388)
            if (done) {
                const int i = bo.y0 + tid;
                const bool act = tid < no && i >= iymin, in = act && i < iymax;
                const int row = in ? i - b.y0 : 0;
                const uint32_t* ge = (const uint32_t*)(bits + kRowGe * A.plane + (long long)row * W);
                const uint32_t* gt = (const uint32_t*)(bits + kRowGt * A.plane + (long long)row * W);
                const int lo = ixmin - b.x0, hi = ixmax - 1 - b.x0;
                const double* next = list_crossings(list, room, row, in && hi > lo, ge, gt, words, lo, hi, h, s_tmp,
                                                    [&](int ln, int c) { return (double)C[(long long)ln * n + c]; });
                done = next != nullptr;
                if (done) {
                    T* line = tile + (long long)(act ? tid : 0) * pitch;
                    bit_sweep<T, 1, true, false>(line + (ixmin - bo.x0), 1, oxmax - 1 - ixmin, ixmax - 1 - ixmin, lo, act, in, ge, gt, words, next, h);
                    bit_sweep<T, -1, false, false>(line + (ixmax - 1 - bo.x0), -1, ixmax - 1 - bo.x0, ixmax - 1 - ixmin, hi, act, in, ge, gt, words, nullptr, h);
                }
            }
            __syncthreads();
            if (done) {  // clampValues (dimensionalBufferReal.h:43-56)
                const T vlo = (T)(-G.delta), vhi = (T)G.delta;
                const int wave = tid >> 6, lane = tid & 63;
                for (int r = wave; r < no; r += NT / 64)
                    for (int c = lane; c < no; c += 64) {
                        T v = tile[r * pitch + c];
                        if (v < vlo) v = vlo;
                        else if (v > vhi) v = vhi;
                        gout[(long long)r * no + c] = v;
                    }
            }
        }
        if (!done) redistance<T>(gout, no, C, n, b, bo, G, gout);
    }
}

}  // namespace ggx
