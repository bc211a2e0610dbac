/*
 * phx_fft_mixed.h -- host side of the mixed-radix transforms (phx_fft_mixed.hip): which
 * lengths they take, in which radices, and the tables they read.
 *
 * A length whose prime factors are at most 13 is split into passes of radix 2 .. 16; any
 * other length N goes through Bluestein's chirp convolution of a length M = 2^a 3^b 5^c,
 * M >= 2 N - 1 (L. I. Bluestein, "A linear filtering approach to the computation of discrete
 * Fourier transform", 1970).
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <complex>
#include <vector>

#include "phx_kernels.h"

namespace phx {

constexpr int kFftMaxPasses = 5; /* enough for every length below 8192 that the radices divide */

/* One length as a sequence of Stockham passes.  Pass i takes butterflies of radix[i] over
   nb = L / radix[i] inputs apart and writes them s[i] apart (s[i]: product of the earlier
   radices).  m_nb, m_s: ceil(2^32 / d) of the divisors nb and s (exact quotients while
   dividend * divisor < 2^32). */
struct FftPlan {
    int len = 0, passes = 0;
    int radix[kFftMaxPasses] = {}, s[kFftMaxPasses] = {};
    uint32_t m_nb[kFftMaxPasses] = {}, m_s[kFftMaxPasses] = {};
};

/* One axis of a 2D transform: the length, its plan in both directions (the inverse runs the
   radices in reverse order) and its table in device memory: e^{-2 pi i k / N} for k < N and, for a
   Bluestein length, e^{-2 pi i k / M} for k < M, the chirp e^{-i pi j^2 / N} for j < N and the
   transform of its conjugate over M, divided by M. */
struct FftAxis {
    int N = 0;
    int M = 0; /* Bluestein length; 0: N itself is split */
    FftPlan fwd, inv;
    void* table = nullptr;
};

/* lengths the mixed-radix kernels take in a given precision: two LDS buffers of one sequence */
bool fft_mixed_supported(int N, size_t real_size);
/* plan of an axis (no device work) and the table it needs, in double precision */
FftAxis fft_axis(int N);
std::vector<std::complex<double>> fft_axis_table(const FftAxis& a, size_t real_size);
/* What a transform forth and back along an axis multiplies amplitudes by, because the constants of its passes are
   rounded (0.4 units of the roundoff a transform and more, always the same): 1 for lengths whose table makes up for it
   (Bluestein's) and for powers of two, which other kernels take.  Rows run the radices in one order, columns turn them
   round for the way back. */
double fft_axis_gain(const FftAxis& a, bool columns, size_t real_size);

enum { kFftFilter = 0, kFftPropagate = 1, kFftForward = 2 };

/* rows: the transform of every row in place (inverse: unnormalised, sign +) */
template <typename real>
hipError_t launch_mixed_rows(typename Vec2<real>::type* data, const FftAxis& c, int Nr, bool inverse, hipStream_t s);
/* columns: forward transform, k-space factor, inverse transform (mode kFftForward: forward only) */
template <typename real>
hipError_t launch_mixed_cols(typename Vec2<real>::type* data, const FftAxis& r, int Nc, int mode, const real* mask, const void* rowf,
                             const void* colf, typename Vec2<real>::type* spec, hipStream_t s);

} // namespace phx
