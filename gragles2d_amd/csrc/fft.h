// fft.h -- batched 2-D convolution of square boxes by mixed-radix FFT (gfx950).
//
// LSbox::convolutionGeneratorFFTW (box.cpp:622-695): phi~ = IDFT2( G . DFT2(phi) ) with the
// real, even symbol G of ConvolutionMode 0 (Laplace, box.cpp:648-659), 1 (Laplace with the
// Richardson extrapolation, 660-673) or 2 (Gaussian, 674-688).  G carries the 1/n^2 of the
// unnormalised c2r transform and uses the global grid size R in nsq (636-637).
//
// One 256-lane workgroup per box, exact n (no padding to a friendly size), three phases
// separated by workgroup barriers:
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
// Workgroup 0 also clears *bad when given (the error flag of a batch call).
__global__ void __launch_bounds__(256) k_fft_twiddles(double2* __restrict__ tw, int nmin, int nmax,
                                                      int* __restrict__ bad) {
    if (bad && blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
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

// The standalone batch (ggx_convolve_boxes): box b has side ns[b] and starts at offs[b] in
// src and dst.  Workgroup i takes boxes i, i + grid, ...; this launch handles the boxes of
// side in (nlo, nhi].
// A box whose side is outside [1, nmax] is left alone and sets *bad (the host reports it).
template <bool LDS>
__global__ void __launch_bounds__(256) k_conv_fft_batch(int count, const int* __restrict__ ns,
                                                        const int64_t* __restrict__ offs,
                                                        const double* __restrict__ src, double* __restrict__ dst,
                                                        const double2* __restrict__ tw, FftSymbol sy, int nb, int nlo,
                                                        int nhi, int nmax, double2* __restrict__ work,
                                                        int* __restrict__ bad) {
    HIP_DYNAMIC_SHARED(unsigned char, smem)
    double2* W = (double2*)smem;
    double2* L = W + nb;
    double2* H = LDS ? L + 2 * kFftWaves * nb : work + (size_t)blockIdx.x * (size_t)fft_slot(nb);
    for (int b = (int)blockIdx.x; b < count; b += (int)gridDim.x) {
        const int n = ns[b];
        if (n < 1 || n > nmax) {
            if (threadIdx.x == 0) atomicOr(bad, 1);
            continue;
        }
        if (n <= nlo || n > nhi) continue;
        const int64_t o = offs[b];
        fft_conv_box<double>(n, nb, src + o, dst + o, tw + tw_offset(n), sy, W, L, H);
    }
}

}  // namespace ggx
