// fft.h -- 2-D convolution of square boxes by transforms (gfx950): in FP64, a step's and the standalone
// batch's, by products with the real transform matrix on the matrix cores; a step's in FP32 by
// mixed-radix FFT, and in FP64 too where the LDS allowed to a context is too small for the strips.
//
// LSbox::convolutionGeneratorFFTW (box.cpp:622-695): phi~ = IDFT2( G . DFT2(phi) ) with the
// real, even symbol G of ConvolutionMode 0 (Laplace, box.cpp:648-659), 1 (Laplace with the
// Richardson extrapolation, 660-673) or 2 (Gaussian, 674-688).  G carries the 1/n^2 of the
// unnormalised c2r transform and uses the global grid size R in nsq (636-637).
//
// The FFT (k_conv_fft): one 256-lane workgroup per box, exact n (no padding to a friendly size),
// three phases separated by workgroup barriers:
//   1. rows     each wave takes a pair of rows (2p, 2p+1), transforms z = row_2p + i row_2p+1
//               as one complex line and splits the result into the two half spectra
//               X[k] = (Z[k] + conj Z[n-k]) / 2, Y[k] = (Z[k] - conj Z[n-k]) / 2i, k <= n/2;
//   2. columns  each wave takes one column k of the n x (n/2+1) half spectrum, transforms it,
//               multiplies it by G(j, k) and transforms it back, without leaving the wave;
//   3. rows     each wave rebuilds the full spectra of a row pair from Hermitian symmetry,
//               inverse-transforms X + iY as one line and writes the real part to row 2p and
//               the imaginary part to row 2p+1.
// The half spectrum lives in LDS for boxes up to kFftLdsMax, above that in a per-workgroup
// slot of a global workspace.  A line transform runs inside its wave as a self-sorting
// (Stockham) sequence of stages, one per prime factor p of n: output t of a stage is the
// p-term sum  X'[t] = sum_r X[j + r n/p] w^(r s),  (j, s) fixed by t and the stage, with every
// twiddle a power of w = exp(-2 pi i / n) read from the per-n table.  The two ping-pong line
// buffers are private to the wave, so a stage needs a wave barrier only.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace ggx {

constexpr int kFftLdsMax = 128;     // largest box side whose half spectrum stays in LDS
constexpr int kFftMaxFactors = 10;  // prime factors of a side <= 1023
constexpr int kFftWaves = 4;        // waves per workgroup

// Start of side n's twiddle table (n entries) in the packed table of all sides 1..nmax.
constexpr __host__ __device__ inline long long tw_offset(int n) { return (long long)n * (n - 1) / 2; }

template <class T> struct Cplx;
template <> struct Cplx<double> { using type = double2; };
template <> struct Cplx<float> { using type = float2; };

struct FftSymbol {
    int mode;     // ConvolutionMode: 0 Laplace, 1 Laplace-Richardson, 2 Gaussian
    double dt;
    double nsq;   // R^2 of the global grid
};

// LDS bytes of one workgroup for boxes up to side nb: twiddles, the four waves' line buffers
// and, on the LDS path, the half spectrum.
template <class T>
__host__ __device__ inline long long fft_lds(int nb, bool spectrum_in_lds) {
    const long long c = (long long)sizeof(typename Cplx<T>::type);
    long long e = nb + 2LL * kFftWaves * nb;
    if (spectrum_in_lds) e += (long long)nb * (nb / 2 + 1);
    return e * c;
}

// Elements of one workgroup's global half-spectrum slot (boxes above kFftLdsMax).
constexpr __host__ __device__ inline long long fft_slot(int nb) { return (long long)nb * (nb / 2 + 1); }

// (cos 2 pi t / n, sin 2 pi t / n) for t < n, every side n of [nmin, nmax]; one workgroup per n.
__global__ void __launch_bounds__(256) k_fft_twiddles(double2* __restrict__ tw, int nmin, int nmax) {
    const int n = nmin + (int)blockIdx.x;
    if (n > nmax) return;
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        double s, c;
        sincospi(2.0 * (double)t / (double)n, &s, &c);
        tw[tw_offset(n) + t] = make_double2(c, s);
    }
}

// Prime factors of n in ascending order (n = 1: none).
__device__ __forceinline__ int fft_factors(int n, int* f) {
    int c = 0, m = n;
    for (int p = 2; m > 1; ++p) {
        if (p * p > m) { f[c++] = m; break; }
        while (m % p == 0) { f[c++] = p; m /= p; }
    }
    return c;
}

// Forward (INV = false, w = exp(-2 pi i/n)) or inverse (unnormalised, w = exp(+2 pi i/n)) DFT of
// the line in a, by one wave; b is the other buffer.  Returns the buffer holding the result.
template <class T, bool INV>
__device__ __forceinline__ typename Cplx<T>::type* line_fft(typename Cplx<T>::type* a, typename Cplx<T>::type* b,
                                                          int n, const int* fac, int nfac,
                                                          const typename Cplx<T>::type* W, int lane) {
    using C = typename Cplx<T>::type;
    int Ns = 1;
    for (int s = 0; s < nfac; ++s) {
        const int p = fac[s], np = n / p, Nsp = Ns * p, tstep = n / Nsp;
        for (int t = lane; t < n; t += 64) {
            const int u = t / Nsp, rem = t - u * Nsp;
            const int q = rem / Ns, k = rem - q * Ns;
            const int j = u * Ns + k;
            const int step = tstep * (k + q * Ns);  // < n
            T re = T(0), im = T(0);
            int e = 0;
            for (int r = 0; r < p; ++r) {
                const C x = a[j + r * np];
                const C w = W[e];
                const T wi = INV ? w.y : -w.y;
                re += x.x * w.x - x.y * wi;
                im += x.x * wi + x.y * w.x;
                e += step;
                if (e >= n) e -= n;
            }
            C o;
            o.x = re;
            o.y = im;
            b[t] = o;
        }
        wave_lds_sync();
        C* tmp = a;
        a = b;
        b = tmp;
        Ns = Nsp;
    }
    return a;
}

// G(j, i): row (y) frequency j, column (x) frequency i <= n/2 (box.cpp:646-691).
__device__ __forceinline__ double fft_symbol(int j, int i, int n, const FftSymbol& sy) {
    const double kPi = 3.14159265358979323846;
    const double n_nsq = (double)(n * n);
    if (sy.mode == 2) {
        const int i2 = min(i, n - i), j2 = min(j, n - j);
        return exp(-sqrt(2 / kPi) * (double)(i2 * i2 + j2 * j2) * 4.0 * sy.dt * sy.nsq / n_nsq * kPi * kPi) / n_nsq;
    }
    const double g = 2.0 * (2.0 - cospi(2.0 * (double)i / (double)n) - cospi(2.0 * (double)j / (double)n)) * sy.nsq;
    if (sy.mode == 0) return 1.0 / (1.0 + (sy.dt * g)) / n_nsq;
    return (4.0 / pow(1 + 1.5 * sy.dt / 40 * g, 40) - 1.0 / pow(1 + 3.0 * sy.dt / 40 * g, 40)) / 3.0 / n_nsq;
}

// The convolution of one box of side n (src -> dst, row-major n x n), by the whole workgroup.
// W: LDS for the n twiddles; L: the four waves' line buffers (2 nb each); H: the half spectrum.
template <class T>
__device__ void fft_conv_box(int n, int nb, const T* __restrict__ src, T* __restrict__ dst,
                             const double2* __restrict__ twn, const FftSymbol& sy, typename Cplx<T>::type* W,
                             typename Cplx<T>::type* L, typename Cplx<T>::type* H) {
    using C = typename Cplx<T>::type;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int nw = (int)(blockDim.x >> 6);
    const int n2 = n / 2 + 1;
    int fac[kFftMaxFactors];
    const int nfac = fft_factors(n, fac);
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        const double2 w = twn[t];
        C c;
        c.x = (T)w.x;
        c.y = (T)w.y;
        W[t] = c;
    }
    __syncthreads();
    C* a0 = L + (size_t)wave * 2 * nb;
    C* b0 = a0 + nb;

    // 1. forward row transforms, two real rows per complex line
    for (int p = wave; 2 * p < n; p += nw) {
        const int r0 = 2 * p;
        const bool two = r0 + 1 < n;
        for (int c = lane; c < n; c += 64) {
            C z;
            z.x = src[(size_t)r0 * n + c];
            z.y = two ? src[(size_t)(r0 + 1) * n + c] : T(0);
            a0[c] = z;
        }
        wave_lds_sync();
        const C* Z = line_fft<T, false>(a0, b0, n, fac, nfac, W, lane);
        for (int k = lane; k < n2; k += 64) {
            const C z = Z[k], zc = Z[k == 0 ? 0 : n - k];
            C x, y;
            x.x = (z.x + zc.x) * T(0.5);
            x.y = (z.y - zc.y) * T(0.5);
            y.x = (z.y + zc.y) * T(0.5);
            y.y = (zc.x - z.x) * T(0.5);
            H[(size_t)r0 * n2 + k] = x;
            if (two) H[(size_t)(r0 + 1) * n2 + k] = y;
        }
        wave_lds_sync();
    }
    __syncthreads();

    // 2. column transform, symbol, inverse column transform
    for (int k = wave; k < n2; k += nw) {
        for (int j = lane; j < n; j += 64) a0[j] = H[(size_t)j * n2 + k];
        wave_lds_sync();
        C* F = line_fft<T, false>(a0, b0, n, fac, nfac, W, lane);
        C* other = (F == a0) ? b0 : a0;
        for (int j = lane; j < n; j += 64) {
            const T g = (T)fft_symbol(j, k, n, sy);
            C v = F[j];
            v.x *= g;
            v.y *= g;
            F[j] = v;
        }
        wave_lds_sync();
        const C* B = line_fft<T, true>(F, other, n, fac, nfac, W, lane);
        for (int j = lane; j < n; j += 64) H[(size_t)j * n2 + k] = B[j];
        wave_lds_sync();
    }
    __syncthreads();

    // 3. inverse row transforms, two real rows per complex line
    for (int p = wave; 2 * p < n; p += nw) {
        const int r0 = 2 * p;
        const bool two = r0 + 1 < n;
        for (int k = lane; k < n; k += 64) {
            C x, y;
            if (k < n2) {
                x = H[(size_t)r0 * n2 + k];
                if (two) y = H[(size_t)(r0 + 1) * n2 + k];
                else { y.x = T(0); y.y = T(0); }
            } else {
                x = H[(size_t)r0 * n2 + (n - k)];
                x.y = -x.y;
                if (two) { y = H[(size_t)(r0 + 1) * n2 + (n - k)]; y.y = -y.y; }
                else { y.x = T(0); y.y = T(0); }
            }
            C z;
            z.x = x.x - y.y;
            z.y = x.y + y.x;
            a0[k] = z;
        }
        wave_lds_sync();
        const C* z = line_fft<T, true>(a0, b0, n, fac, nfac, W, lane);
        for (int c = lane; c < n; c += 64) {
            const C v = z[c];
            dst[(size_t)r0 * n + c] = v.x;
            if (two) dst[(size_t)(r0 + 1) * n + c] = v.y;
        }
        wave_lds_sync();
    }
    __syncthreads();
}

// The step's launch: the grains of one bucket (boxes up to nb), workgroup i taking items i, i + grid, ...
template <class T, bool LDS>
__global__ void __launch_bounds__(256) k_conv_fft(const int* __restrict__ list, const int* __restrict__ count,
                                                  const Box* __restrict__ box,
                                                  const long long* __restrict__ off, const T* __restrict__ src,
                                                  T* __restrict__ dst, const double2* __restrict__ tw, FftSymbol sy,
                                                  int nb, typename Cplx<T>::type* __restrict__ work) {
    using C = typename Cplx<T>::type;
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    C* W = (C*)smem;
    C* L = W + nb;
    C* H = LDS ? L + 2 * kFftWaves * nb : work + (size_t)blockIdx.x * (size_t)fft_slot(nb);
    const int total = *count;  // written by k_tally (or the host) before this kernel
    for (int item = (int)blockIdx.x; item < total; item += (int)gridDim.x) {
        __syncthreads();  // the previous box's LDS is free
        const int g = list[item];
        const int n = box[g].n;
        const long long o = off[g];
        fft_conv_box<T>(n, nb, src + o, dst + o, tw + tw_offset(n), sy, W, L, H);
    }
}

// ------------------------------------------------------------------------------------------
// The standalone batch (ggx_convolve_boxes): box b has side ns[b] and starts at offs[b] in src and
// dst.  The symbol is real and even in both directions, so the real transform with H[j][k] =
// cas(2 pi j k / n) = cos + sin diagonalises the convolution as the complex one does (H symmetric,
// H H = n I; Hartley, Proc. IRE 30, 1942):  phi~ = H ( G . (H phi H) ) H.  Four products with H per box, on the matrix cores
// in FP64 and without complex arithmetic, half spectra or a workspace:
//   k_box_rows     dst = src H   one workgroup per 16 rows
//   k_box_columns  dst = H (G . (H dst))   one workgroup per 16 columns
//   k_box_rows     dst = dst H
// each in place on its strip, which lies in LDS.  H is not stored: its elements are read from the n
// values cas(2 pi t / n) in LDS, the index j k mod n of a lane's next element by one addition.  An
// FP64 product of 16 x 16 x 4 keeps a SIMD's matrix core for 64 cycles, in which the LDS has room
// for far more than the two reads it needs.  6000 boxes of side 16 to 128 take 0.36, 0.74 and 0.37 ms
// (products with the sides rounded up to 16: 0.12 ms each; the rest is each strip's chain of load,
// table, product and store at 16 waves per CU), 96 of side 130 to 256 take 0.33 ms.  The FFT with a
// workgroup per box took 8.6 ms, bound by its p-term sums, and 25 ms, bound by its eight half-spectrum
// slots.  The Richardson symbol's two 40th powers are a third of k_box_columns with pow().
// In a step (k_box_rows and k_box_columns of FP64 networks with the FFT engine's symbols) the boxes
// are the grains of a launch's work items.  There the FFT took 1.2 of 2.0 ms per step of a 5000-grain
// Laplace network, up to 0.4 ms of it for the few widest boxes, one after the other's long sums in
// one workgroup; the strips take 0.42 ms, 0.06 of it in launches for sides that the network has few of.
// ------------------------------------------------------------------------------------------
struct BoxBatch {
    int count, strips;   // boxes; strips of 16 lines of the largest side allowed
    const int* ns;
    const int64_t* offs;
    int nmax;            // a box whose side is outside [1, nmax] is left alone and sets *bad
    int* bad;
};

struct StepBoxes {       // the same for a step's work items
    Items it;
    int strips, nmax;
    const Box* box;
    const long long* off;
};

constexpr int kStripPitch = 17;   // doubles per line of a strip: 16 and one against bank conflicts

constexpr __host__ __device__ inline int strip_lines(int n) { return (n + 3) & ~3; }
constexpr __host__ __device__ inline long long box_rows_lds(int n) { return 8LL * (strip_lines(n) * kStripPitch + n); }
constexpr __host__ __device__ inline long long box_columns_lds(int n) { return 8LL * (2 * strip_lines(n) * kStripPitch + 2 * n); }

// K tiles of a strip product, tiles t0, t0 + 4, ...: H times the strip (ROWS: the strip, whose lines
// are H's rows, times H).  s_in: strip_lines(n) lines of 16 values, zero beyond n.
template <bool ROWS, int K, class Out>
__device__ __forceinline__ void strip_tiles(int n, const double* s_cas, const double* s_in, int t0, Out out) {
    using V = typename Mma<double>::V;
    const int lane = (int)(threadIdx.x & 63), l = lane & 15, q = lane >> 4;
    V sum[K];
    int at[K], step[K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int i = ((t0 + 4 * u) * 16 + l) % n;
        sum[u] = V{0.0, 0.0, 0.0, 0.0};
        at[u] = i * q % n;
        step[u] = 4 * i % n;
    }
    const double* line = s_in + q * kStripPitch + l;
    auto products = [&](V* acc, int k) {  // lines k .. k + 3
        const double x = line[k * kStripPitch];
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const double h = s_cas[at[u]];
            acc[u] = ROWS ? Mma<double>::run(x, h, acc[u]) : Mma<double>::run(h, x, acc[u]);
            at[u] += step[u];
            if (at[u] >= n) at[u] -= n;
        }
    };
    // eight lines' products are summed by themselves before they join the total: rounding errors grow
    // with the longer of the two chains (0.7 to 0.95 of the FFT's error; one chain: up to 2.7 times it)
    int k = 0;
    for (; k + 8 <= n; k += 8) {
        V acc[K];
#pragma unroll
        for (int u = 0; u < K; ++u) acc[u] = V{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < 8; d += 4) products(acc, k + d);
#pragma unroll
        for (int u = 0; u < K; ++u) sum[u] += acc[u];
    }
    for (; k < n; k += 4) products(sum, k);
#pragma unroll
    for (int u = 0; u < K; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = Mma<double>::row(q, r);
            if (ROWS) out(row, (t0 + 4 * u) * 16 + l, sum[u][r]);
            else out((t0 + 4 * u) * 16 + row, l, sum[u][r]);
        }
}

// All tiles of a strip product over the workgroup's four waves; out(row, column, value) of each.
// `turn` moves the tiles on by a wave per strip: a box of five tiles gives one wave two of them.
template <bool ROWS, class Out>
__device__ __forceinline__ void strip_product(int n, const double* s_cas, const double* s_in, int turn, Out out) {
    const int tiles = (n + 15) >> 4;
    int t0 = __builtin_amdgcn_readfirstlane((int)((threadIdx.x >> 6) + (unsigned)turn) & 3);
    while (t0 < tiles) {
        const int left = (tiles - t0 + 3) >> 2;
        if (left >= 4) strip_tiles<ROWS, 4>(n, s_cas, s_in, t0, out);
        else if (left == 3) strip_tiles<ROWS, 3>(n, s_cas, s_in, t0, out);
        else if (left == 2) strip_tiles<ROWS, 2>(n, s_cas, s_in, t0, out);
        else strip_tiles<ROWS, 1>(n, s_cas, s_in, t0, out);
        t0 += 16;
    }
}

__device__ __forceinline__ int box_count(const BoxBatch& B) { return B.count; }
__device__ __forceinline__ int box_count(const StepBoxes& B) { return items_total(B.it); }

__device__ __forceinline__ void box_place(const BoxBatch& B, int b, int* n, int64_t* o) {
    *n = sload(B.ns + b);
    *o = sload(B.offs + b);
}
__device__ __forceinline__ void box_place(const StepBoxes& B, int b, int* n, int64_t* o) {
    int bucket, pos;
    const int g = item_grain(B.it, b, &bucket, &pos);
    *n = sload(&B.box[g].n);
    *o = sload(B.off + g);
}

__device__ __forceinline__ void clear_bad(const BoxBatch& B) { *B.bad = 0; }
__device__ __forceinline__ void clear_bad(const StepBoxes&) {}
__device__ __forceinline__ void set_bad(const BoxBatch& B) { *B.bad = 1; }
__device__ __forceinline__ void set_bad(const StepBoxes&) {}

// The box and strip of a work item; false: no such strip.  Box b's items take its strips from strip b on,
// wrapping at the last: workgroup i runs on die i mod 8, so with strip = item mod strips the strips of one
// place in a box, and the empty ones beyond it where max_n is far above the sides, all fell to the same
// dies.  6000 boxes of side 16 to 32 called with max_n 512: 5.2 -> 1.04 ms (two of eight dies had the work;
// the rest is one workgroup of 147 KB per CU); 96 of side 130 to 256 0.355 -> 0.331.
template <class Boxes>
__device__ __forceinline__ bool box_strip(const Boxes& B, long long item, int* n, int64_t* o, int* line0) {
    const int b = (int)(item / B.strips);
    *line0 = (int)(((unsigned)(item - (long long)b * B.strips) + (unsigned)b) % (unsigned)B.strips) * 16;
    box_place(B, b, n, o);
    return *n >= 1 && *n <= B.nmax && *line0 < *n;
}

// x^40 by squarings with their rounding errors carried along (l: what h lacks).
__device__ __forceinline__ double power40(double x) {
    double h = x, l = 0.0, h8 = 0.0, l8 = 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const double s = h * h;
        l = fma(h, h, -s) + 2.0 * h * l;
        h = s;
        if (k == 2) { h8 = h; l8 = l; }
    }
    const double p = h * h8;
    return p < 1e300 ? fma(h, h8, fma(h, l8, l * h8)) : p;  // not past an overflow
}

// fft_symbol with cos(2 pi t / n) from s_cos[t].
__device__ __forceinline__ double box_symbol(int j, int i, int n, const double* s_cos, const FftSymbol& sy) {
    const double kPi = 3.14159265358979323846;
    const double n_nsq = (double)(n * n);
    if (sy.mode == 2) {
        const int i2 = min(i, n - i), j2 = min(j, n - j);
        return exp(-sqrt(2 / kPi) * (double)(i2 * i2 + j2 * j2) * 4.0 * sy.dt * sy.nsq / n_nsq * kPi * kPi) / n_nsq;
    }
    const double g = 2.0 * (2.0 - s_cos[i] - s_cos[j]) * sy.nsq;
    if (sy.mode == 0) return 1.0 / (1.0 + (sy.dt * g)) / n_nsq;
    return (4.0 / power40(1 + 1.5 * sy.dt / 40 * g) - 1.0 / power40(1 + 3.0 * sy.dt / 40 * g)) / 3.0 / n_nsq;
}

// dst = src H by strips of 16 rows (src may be dst).  first: clears *bad.
template <class Boxes>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_box_rows(Boxes B, const double* src, double* dst, int first) {
    HIP_DYNAMIC_SHARED(double, s_box)
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (first && blockIdx.x == 0 && tid == 0) clear_bad(B);
    const long long items = (long long)box_count(B) * B.strips;
    for (long long item = blockIdx.x; item < items; item += gridDim.x) {
        int n, r0;
        int64_t o;
        if (!box_strip(B, item, &n, &o, &r0)) continue;
        double* s_in = s_box;
        double* s_cas = s_box + strip_lines(n) * kStripPitch;
        for (int t = tid; t < n; t += 256) {
            double s, c;
            sincospi(2.0 * (double)t / (double)n, &s, &c);
            s_cas[t] = c + s;
        }
        for (int r = wave; r < 16; r += 4)
            for (int k = lane; k < strip_lines(n); k += 64)
                s_in[k * kStripPitch + r] = (r0 + r < n && k < n) ? src[o + (int64_t)(r0 + r) * n + k] : 0.0;
        __syncthreads();
        strip_product<true>(n, s_cas, s_in, (int)item, [&](int row, int col, double v) {
            if (r0 + row < n && col < n) dst[o + (int64_t)(r0 + row) * n + col] = v;
        });
        __syncthreads();  // the strip is free
    }
}

// dst = H (G . (H dst)) by strips of 16 columns.
template <class Boxes>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_box_columns(Boxes B, double* dst, FftSymbol sy) {
    HIP_DYNAMIC_SHARED(double, s_box)
    const int tid = (int)threadIdx.x;
    const long long items = (long long)box_count(B) * B.strips;
    for (long long item = blockIdx.x; item < items; item += gridDim.x) {
        int n, c0;
        int64_t o;
        if (!box_strip(B, item, &n, &o, &c0)) {
            if (tid == 0 && (n < 1 || n > B.nmax)) set_bad(B);
            continue;
        }
        const int lines = strip_lines(n);
        double* s_in = s_box;
        double* s_mid = s_in + lines * kStripPitch;
        double* s_cas = s_mid + lines * kStripPitch;
        double* s_cos = s_cas + n;
        for (int t = tid; t < n; t += 256) {
            double s, c;
            sincospi(2.0 * (double)t / (double)n, &s, &c);
            s_cas[t] = c + s;
            s_cos[t] = c;
        }
        const int lc = tid & 15, c = min(c0 + lc, n - 1);
        for (int k = tid >> 4; k < lines; k += 16)
            s_in[k * kStripPitch + lc] = (k < n && c0 + lc < n) ? dst[o + (int64_t)k * n + c0 + lc] : 0.0;
        __syncthreads();
        for (int j = tid >> 4; 2 * j <= n; j += 16) {  // the symbol, even in j
            const double g = box_symbol(j, c, n, s_cos, sy);
            s_mid[j * kStripPitch + lc] = g;
            if (j > 0) s_mid[(n - j) * kStripPitch + lc] = g;
        }
        __syncthreads();
        strip_product<false>(n, s_cas, s_in, (int)item, [&](int j, int col, double v) {
            if (j < lines) s_mid[j * kStripPitch + col] = j < n ? v * s_mid[j * kStripPitch + col] : 0.0;
        });
        __syncthreads();
        strip_product<false>(n, s_cas, s_mid, (int)item + 2, [&](int row, int col, double v) {
            if (row < n && c0 + col < n) dst[o + (int64_t)row * n + c0 + col] = v;
        });
        __syncthreads();
    }
}

}  // namespace ggx
