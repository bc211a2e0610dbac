/*
 * phx_fft_mixed.hip -- transforms of lengths that are not powers of two (and of powers of two next
 * to them) for the k-space filter and the split-step iterator: mixed-radix Stockham passes in LDS,
 * Bluestein's convolution for lengths with a prime factor above 13.
 *
 * A pass of radix R over a sequence of L points (textbook Stockham autosort, Van Loan,
 * "Computational Frameworks for the FFT", 1992): butterfly b (b < L / R) with p = b / s, q = b - p s
 * reads elements b + j L / R, transforms them in registers, multiplies output j by
 * e^{-2 pi i j p s / L} and writes it to q + s (R p + j); s is the product of the earlier radices.
 * Only the forward direction exists: an inverse transform swaps real and imaginary parts on the
 * way in and out.
 *
 * The first pass reads its inputs from where they are (global memory: consecutive butterflies read
 * consecutive elements) and the last one writes its outputs there, so a transform of P passes goes
 * through LDS P - 1 times.  In a convolution (forward, factor, inverse: the column pass, and
 * Bluestein's) the inverse runs the radices in reverse: its first pass then takes exactly the
 * elements that the last forward pass left in the same thread, so the factor is applied in
 * registers and the turn costs no LDS trip.  Two LDS buffers take turns, one barrier a pass.
 * Column groups keep their CB columns adjacent in LDS and in the lanes.
 */
#include <algorithm>
#include <cmath>

#include "phx_fft_engine.h"

namespace phx {

namespace {

/* k-space factor of the column pass at column c, row k of the spectrum (k = 0 first) */
template <typename real>
struct ColFactor {
    using v2 = typename Vec2<real>::type;
    int mode;
    const real* mask;
    const Cx<real>*rowf, *colf;
    v2* spec;
    int Nc, Nr;
    real ntot;
    __device__ __forceinline__ Cx<real> operator()(int c, int k, Cx<real> f) const {
        if (mode == kFftPropagate) return cmul(cmul(f, colf[c]), rowf[k]);
        /* mask of the quadrant-swapped grid (fft_shift_2D, kernel_fft.cuh:15-32) */
        int rs = k + (Nr >> 1), cs = c + (Nc >> 1);
        if (rs >= Nr) rs -= Nr;
        if (cs >= Nc) cs -= Nc;
        const real m = mask[(size_t)rs * Nc + cs];
        f.r = f.r / ntot * m;
        f.i = f.i / ntot * m;
        if (spec) {
            v2 o;
            o.x = f.r;
            o.y = f.i;
            spec[(size_t)k * Nc + c] = o;
        }
        return f;
    }
};

} // namespace

/* ------------------------------------------------------------------------------- kernels */

/* rows per workgroup: rpb; `swap` runs the inverse transform */
template <typename real, bool BLUE, int FAM>
__global__ __launch_bounds__(kMixThreads) void mixed_rows(typename Vec2<real>::type* data, FftPlan fwd, FftPlan inv, int N, int Nr,
                                                          int rpb, int swap, const Cx<real>* __restrict__ table) {
    const int row0 = blockIdx.x * rpb, count = min(rpb, Nr - row0);
    int A = 0, B = rpb * fwd.len;
    typename Vec2<real>::type* rows = data + (size_t)row0 * N;
    auto load = [&](int seq, int i) {
        const auto v = rows[(size_t)seq * N + i];
        return swap ? Cx<real>{v.y, v.x} : Cx<real>{v.x, v.y};
    };
    auto store = [&](int seq, int i, Cx<real> f) {
        typename Vec2<real>::type o;
        o.x = swap ? f.i : f.r;
        o.y = swap ? f.r : f.i;
        rows[(size_t)seq * N + i] = o;
    };
    if constexpr (BLUE) {
        const Cx<real>*tw = table + N, *chirp = tw + fwd.len, *hat = chirp + N;
        convolve<real, 0, FAM>(
            fwd, inv, count, A, B, tw,
            [&](int seq, int i) { return i < N ? cmul(load(seq, i), chirp[i]) : Cx<real>{real(0), real(0)}; },
            [&](int, int bb, int nb, auto& x) {
                constexpr int R = sizeof(x) / sizeof(x[0]);
#pragma unroll
                for (int j = 0; j < R; j++) x[j] = cmul(x[j], hat[bb + j * nb]);
            },
            [&](int seq, int i, Cx<real> f) {
                if (i < N) store(seq, i, cmul(swapped(f), chirp[i]));
            });
    } else {
        transform<real, 0, FAM>(fwd, count, A, B, table, load, store);
    }
}

/* CB adjacent columns per workgroup: forward, factor, inverse; FWD: forward only.  Columns past the
   grid read column Nc - 1 and are not written. */
template <typename real, int CB, bool BLUE, int FAM, bool FWD>
__global__ __launch_bounds__(kMixThreads) void mixed_cols(typename Vec2<real>::type* data, FftPlan fwd, FftPlan inv, ColFactor<real> fac,
                                                          const Cx<real>* __restrict__ table) {
    const int Nc = fac.Nc, N = fac.Nr;
    const int c0 = fft_xcd_group(blockIdx.x, gridDim.x) * CB;
    int A = 0, B = CB * fwd.len;
    auto load = [&](int seq, int i) {
        const auto v = data[(size_t)i * Nc + min(c0 + seq, Nc - 1)];
        return Cx<real>{v.x, v.y};
    };
    auto store = [&](int seq, int i, Cx<real> f) {
        typename Vec2<real>::type o;
        o.x = f.r;
        o.y = f.i;
        if (c0 + seq < Nc) data[(size_t)i * Nc + c0 + seq] = o;
    };
    auto factor = [&](int seq, int k, Cx<real> f) { return c0 + seq < Nc ? fac(c0 + seq, k, f) : f; };
    if constexpr (!BLUE) {
        if constexpr (FWD)
            transform<real, CB, FAM>(fwd, CB, A, B, table, load, store);
        else
            convolve<real, CB, FAM>(
                fwd, inv, CB, A, B, table, load,
                [&](int seq, int bb, int nb, auto& x) {
                    constexpr int R = sizeof(x) / sizeof(x[0]);
#pragma unroll
                    for (int j = 0; j < R; j++) x[j] = factor(seq, bb + j * nb, x[j]);
                },
                [&](int seq, int i, Cx<real> f) { store(seq, i, swapped(f)); });
    } else {
        const Cx<real>*tw = table + N, *chirp = tw + fwd.len, *hat = chirp + N;
        auto by_hat = [&](int, int bb, int nb, auto& x) {
            constexpr int R = sizeof(x) / sizeof(x[0]);
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = cmul(x[j], hat[bb + j * nb]);
        };
        auto chirped = [&](int seq, int i) { return i < N ? cmul(load(seq, i), chirp[i]) : Cx<real>{real(0), real(0)}; };
        if constexpr (FWD) {
            convolve<real, CB, FAM>(fwd, inv, CB, A, B, tw, chirped, by_hat, [&](int seq, int i, Cx<real> f) {
                if (i < N) store(seq, i, cmul(swapped(f), chirp[i]));
            });
        } else {
            /* the filtered spectrum (parts swapped for the inverse) goes to the LDS buffer that the
               last pass of the first convolution does not read */
            convolve<real, CB, FAM>(fwd, inv, CB, A, B, tw, chirped, by_hat, [&](int seq, int i, Cx<real> f) {
                if (i < N) lds<real>()[B + i * CB + seq] = swapped(factor(seq, i, cmul(swapped(f), chirp[i])));
            });
            __syncthreads();
            const Cx<real>* in = lds<real>() + B;
            int A2 = B, B2 = A;
            convolve<real, CB, FAM>(
                fwd, inv, CB, A2, B2, tw,
                [&](int seq, int i) { return i < N ? cmul(in[i * CB + seq], chirp[i]) : Cx<real>{real(0), real(0)}; }, by_hat,
                [&](int seq, int i, Cx<real> f) {
                    if (i < N) store(seq, i, swapped(cmul(swapped(f), chirp[i])));
                });
        }
    }
}

/* ------------------------------------------------------------------------------- host side */
namespace {

constexpr int kRadices[] = {2, 3, 4, 5, 7, 8, 9, 10, 11, 13, 16};

/* fewest passes, then the smallest largest radix, then the smallest sum; `n` = kFftMaxPasses + 1: none */
void split_radices(int len, int depth, int* cur, int& n, int* best) {
    if (len == 1) {
        auto cost = [](const int* r, int k) {
            int mx = 0, sum = 0;
            for (int i = 0; i < k; i++) mx = std::max(mx, r[i]), sum += r[i];
            return mx * 1000 + sum;
        };
        if (depth < n || (depth == n && cost(cur, depth) < cost(best, n))) {
            for (int i = 0; i < depth; i++) best[i] = cur[i];
            n = depth;
        }
        return;
    }
    if (depth >= n || depth >= kFftMaxPasses) return;
    for (int r : kRadices)
        if (len % r == 0 && (depth == 0 || r <= cur[depth - 1])) {
            cur[depth] = r;
            split_radices(len / r, depth + 1, cur, n, best);
        }
}
int split_radices(int len, int* best) {
    int cur[kFftMaxPasses], n = kFftMaxPasses + 1;
    split_radices(len, 0, cur, n, best);
    return n;
}

FftPlan make_plan(int len, const int* radix, int passes) {
    FftPlan p;
    p.len = len;
    p.passes = passes;
    int s = 1;
    for (int i = 0; i < passes; i++) {
        p.radix[i] = radix[i];
        p.s[i] = s;
        const uint32_t nb = (uint32_t)(len / radix[i]);
        p.m_nb[i] = nb > 1 ? 0xFFFFFFFFu / nb + 1u : 0u;
        p.m_s[i] = s > 1 ? 0xFFFFFFFFu / (uint32_t)s + 1u : 0u;
        s *= radix[i];
    }
    return p;
}

/* ---- tables, and the transforms on the host, in arithmetic of type T: double for FP32, long double (64-bit mantissa
   on x86) for FP64, so that rounding to the kernels' precision is the only error that counts */
template <class T>
struct Hc {
    T r, i;
};
template <class T>
inline Hc<T> operator*(Hc<T> a, Hc<T> b) { return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; } /* (std::complex looks for NaN) */
template <class T>
inline Hc<T> conj(Hc<T> a) { return {a.r, -a.i}; }
template <class T>
using Hcs = std::vector<Hc<T>>;

/* e^{-2 pi i k / n}, k reduced exactly */
template <class T>
Hc<T> root(long long k, long long n) {
    const std::complex<T> z = std::polar((T)1, (T)-2 * (T)3.14159265358979323846264338327950288L * (T)(k % n) / (T)n);
    return {z.real(), z.imag()};
}
template <class T>
Hc<T> rounded(Hc<T> z, size_t real_size) { /* to the kernels' precision */
    if (real_size == sizeof(float)) return {(T)(float)z.r, (T)(float)z.i};
    return {(T)(double)z.r, (T)(double)z.i};
}
template <class T>
Hcs<T> rounded(Hcs<T> v, size_t real_size) {
    for (Hc<T>& z : v) z = rounded(z, real_size);
    return v;
}

/* the constants of the butterflies: exact (real_size 0) or as the kernels have them */
template <class T>
struct HostConstants {
    Hc<T> w[17][16]; /* e^{-2 pi i k / R} */
    explicit HostConstants(size_t real_size) {
        for (int R : kRadices)
            for (int k = 0; k < R; k++) {
                const Turn t = turn(k, R);
                w[R][k] = real_size ? rounded(Hc<T>{(T)t.c, (T)-t.s}, real_size) : root<T>(k, R);
            }
    }
};

/* dft() of phx_fft_engine.h: R values `step` apart, in place */
template <class T>
void host_dft(const HostConstants<T>& h, int R, Hc<T>* x, int step) {
    const int R1 = R == 4 ? R : first_factor(R), R2 = R / R1;
    Hc<T> y[16];
    if (R1 == R) {
        for (int j = 0; j < R; j++) {
            Hc<T> t{0, 0};
            for (int k = 0; k < R; k++) {
                const Hc<T> z = x[k * step] * h.w[R][j * k % R];
                t = {t.r + z.r, t.i + z.i};
            }
            y[j] = t;
        }
        for (int j = 0; j < R; j++) x[j * step] = y[j];
        return;
    }
    for (int n2 = 0; n2 < R2; n2++) { /* the values R2 n1 + n2, then their transform k1 there */
        host_dft(h, R1, x + n2 * step, R2 * step);
        for (int k1 = 1; k1 < R1; k1++) x[(R2 * k1 + n2) * step] = x[(R2 * k1 + n2) * step] * h.w[R][n2 * k1 % R];
    }
    for (int k1 = 0; k1 < R1; k1++) {
        host_dft(h, R2, x + R2 * k1 * step, step);
        for (int k2 = 0; k2 < R2; k2++) y[k1 + R1 * k2] = x[(R2 * k1 + k2) * step];
    }
    for (int k = 0; k < R; k++) x[k * step] = y[k];
}
/* transform(); w: the roots of len points */
template <class T>
Hcs<T> host_transform(const HostConstants<T>& h, const FftPlan& p, Hcs<T> x, const Hcs<T>& w) {
    Hcs<T> y(p.len);
    for (int i = 0; i < p.passes; i++) {
        const int R = p.radix[i], s = p.s[i], nb = p.len / R;
        const bool last = i == p.passes - 1;
        for (int b = 0; b < nb; b++) {
            const int pp = b / s, q = b - pp * s;
            Hc<T> t[16];
            for (int j = 0; j < R; j++) t[j] = x[b + j * nb];
            host_dft(h, R, t, 1);
            for (int j = 0; j < R; j++) y[q + s * (R * pp + j)] = last ? t[j] : t[j] * w[j * pp * s];
        }
        std::swap(x, y);
    }
    return x;
}
/* Bluestein's transform of N values from its tables; the sign of the second transform is turned by conjugation */
template <class T>
Hcs<T> host_bluestein(const HostConstants<T>& h, const FftAxis& a, const Hcs<T>& x, const Hcs<T>& w, const Hcs<T>& chirp, const Hcs<T>& hat) {
    Hcs<T> y(a.M, Hc<T>{0, 0});
    for (int j = 0; j < a.N; j++) y[j] = x[j] * chirp[j];
    y = host_transform(h, a.fwd, y, w);
    for (int k = 0; k < a.M; k++) y[k] = conj(y[k] * hat[k]);
    y = host_transform(h, a.inv, y, w);
    y.resize(a.N);
    for (int j = 0; j < a.N; j++) y[j] = conj(y[j]) * chirp[j];
    return y;
}
/* mean gain of `kernel` against `exact`, two linear maps of n values, over 512 or more fixed pseudo-random ones: known
   to a few hundredths of what the rounding of one constant does */
template <class T, class F, class G>
T mean_gain(int n, F kernel, G exact) {
    uint32_t state = 12345;
    auto next = [&] {
        state = state * 1664525u + 1013904223u;
        return (T)(int32_t)state / (T)2147483648.0;
    };
    T num = 0, den = 0;
    for (int done = 0; done < 512; done += n) {
        Hcs<T> x(n);
        for (Hc<T>& z : x) {
            z.r = next();
            z.i = next();
        }
        const Hcs<T> r = kernel(x), e = exact(x);
        for (int k = 0; k < n; k++) num += e[k].r * r[k].r + e[k].i * r[k].i, den += e[k].r * e[k].r + e[k].i * e[k].i;
    }
    return num / den;
}

/* the next power of two from 2 N - 1, or the length 2^a 3^b 5^c below it with the least cost where that
   is at most 0.6 of the power of two's; cost: passes x (points + 256), the 256 for what a pass takes
   whatever its length (a filter of 138 x 158 FP64: 34 us with 288 and 320 points, 27 with 512; a filter of 1030 x 1030 FP64: 201 us with 2304 = 16 16 9
   points, 302 with 4096; of 646 x 646: 108 with 1296 = 16 9 9, 100 with 2048) */
int bluestein_length(int N) {
    int pow2 = 1;
    while (pow2 < 2 * N - 1) pow2 <<= 1;
    int best = pow2, radix[kFftMaxPasses], cost = (pow2 + 256) * split_radices(pow2, radix) * 6 / 10;
    for (int M = 2 * N - 1; M < pow2; M++) {
        if (largest_prime(M) > 5) continue;
        const int n = split_radices(M, radix);
        if (n <= kFftMaxPasses && (M + 256) * n < cost) best = M, cost = (M + 256) * n;
    }
    return best;
}

} // namespace

bool fft_mixed_supported(int N, size_t real_size) { return N >= 2 && N % 2 == 0 && (size_t)N * 4 * real_size <= 65536; }

FftAxis fft_axis(int N) {
    FftAxis a;
    a.N = N;
    a.M = largest_prime(N) > 13 ? bluestein_length(N) : 0;
    const int len = a.M ? a.M : N;
    int best[kFftMaxPasses];
    const int n = split_radices(len, best);
    if (n > kFftMaxPasses) return a; /* passes = 0: refused by the launchers */
    /* odd radices first: the first pass writes its outputs R elements apart */
    std::stable_sort(best, best + n, [](int x, int y) { return (x & 1) > (y & 1); });
    a.fwd = make_plan(len, best, n);
    std::reverse(best, best + n);
    a.inv = make_plan(len, best, n);
    return a;
}

/* Bluestein's tables are rounded once: the chirp's transform in double was off by several units, as much as the FP64
   transform itself (a filter of 138 x 158, relative L2 in units of 2^-53: 12.0 with tables from double, 5.9 so, 4.3
   with hat made up for the gain below and the butterflies' constants rounded once; direct sums 11.2) */
template <class T>
static std::vector<std::complex<double>> axis_table(const FftAxis& a, size_t real_size) {
    std::vector<std::complex<double>> t;
    auto put = [&](auto z) { t.emplace_back((double)z.r, (double)z.i); };
    for (int k = 0; k < a.N; k++) put(root<double>(k, a.N));
    if (!a.M || !a.fwd.passes) return t;
    const HostConstants<T> exact(0), kernel(real_size);
    Hcs<T> w(a.M), chirp(a.N), b(a.M, Hc<T>{0, 0});
    for (int k = 0; k < a.M; k++) w[k] = root<T>(k, a.M);
    for (long long j = 0; j < a.N; j++) {
        chirp[j] = root<T>(j * j % (2 * a.N), 2 * a.N);
        b[j] = conj(chirp[j]);
        if (j) b[a.M - j] = b[j];
    }
    Hcs<T> hat = host_transform(exact, a.fwd, b, w);
    for (Hc<T>& z : hat) z = {z.r / a.M, z.i / a.M};
    /* the rounded constants of the two transforms shrink or stretch what passes through by 0.4 to 1 units, the same way
       every time: hat makes up for it (a split-step run of 106 x 106 FP32 lost 2.5 units of amplitude a step, 76 x 76
       3.2, direct sums less than 0.5; now 0.03 and -0.7) */
    const Hcs<T> wr = rounded(w, real_size), cr = rounded(chirp, real_size), hr = rounded(hat, real_size);
    const T gain = mean_gain<T>(
        a.N, [&](const Hcs<T>& x) { return host_bluestein(kernel, a, x, wr, cr, hr); },
        [&](const Hcs<T>& x) { return host_bluestein(exact, a, x, w, chirp, hat); });
    for (const auto& z : w) put(z);
    for (const auto& z : chirp) put(z);
    for (const auto& z : hat) put(Hc<T>{z.r / gain, z.i / gain});
    return t;
}

std::vector<std::complex<double>> fft_axis_table(const FftAxis& a, size_t real_size) {
    return real_size == sizeof(float) ? axis_table<double>(a, real_size) : axis_table<long double>(a, real_size);
}

template <class T>
static double plan_gain(const FftPlan& p, size_t real_size) {
    const HostConstants<T> exact(0), kernel(real_size);
    Hcs<T> w, wr;
    for (int k = 0; k < p.len; k++) {
        const Hc<double> z = root<double>(k, p.len); /* as the table holds it */
        w.push_back(root<T>(k, p.len));
        wr.push_back(rounded(Hc<T>{(T)z.r, (T)z.i}, real_size));
    }
    return (double)mean_gain<T>(
        p.len, [&](const Hcs<T>& x) { return host_transform(kernel, p, x, wr); }, [&](const Hcs<T>& x) { return host_transform(exact, p, x, w); });
}

double fft_axis_gain(const FftAxis& a, bool columns, size_t real_size) {
    if (a.M || !a.fwd.passes || largest_prime(a.N) <= 2) return 1.0;
    auto gain = [&](const FftPlan& p) { return real_size == sizeof(float) ? plan_gain<double>(p, real_size) : plan_gain<long double>(p, real_size); };
    const double g = gain(a.fwd);
    return g * (columns ? gain(a.inv) : g);
}

template <typename real>
hipError_t launch_mixed_rows(typename Vec2<real>::type* data, const FftAxis& c, int Nr, bool inverse, hipStream_t s) {
    const int len = c.fwd.len;
    const size_t per = 2 * (size_t)len * sizeof(Cx<real>);
    if (!c.fwd.passes || per > kMixLdsMax) return hipErrorInvalidValue;
    const int wide = widest_pass(c.fwd), rpb = rows_per_block(c.fwd);
    const dim3 grid((Nr + rpb - 1) / rpb), blk(mixed_threads(wide * rpb));
    const auto* t = (const Cx<real>*)c.table;
    auto go = [&](auto kernel) {
        const hipError_t e = allow_lds(kernel, per * rpb);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, blk, per * rpb, s, data, c.fwd, c.inv, c.N, Nr, rpb, (int)inverse, t);
        return hipGetLastError();
    };
    if (c.M) return radix_family(len) == 0 ? go(&mixed_rows<real, true, 0>) : go(&mixed_rows<real, true, 1>);
    return radix_family(len) < 2 ? go(&mixed_rows<real, false, 1>) : go(&mixed_rows<real, false, 2>);
}

template <typename real, int CB, bool BLUE, int FAM>
static hipError_t cols_cb(typename Vec2<real>::type* data, const FftAxis& r, const ColFactor<real>& f, hipStream_t s) {
    const size_t lds = 2 * (size_t)CB * r.fwd.len * sizeof(Cx<real>);
    const dim3 grid((f.Nc + CB - 1) / CB), blk(mixed_threads(CB * widest_pass(r.fwd)));
    auto go = [&](auto kernel) {
        const hipError_t e = allow_lds(kernel, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, blk, lds, s, data, r.fwd, r.inv, f, (const Cx<real>*)r.table);
        return hipGetLastError();
    };
    return f.mode == kFftForward ? go(&mixed_cols<real, CB, BLUE, FAM, true>) : go(&mixed_cols<real, CB, BLUE, FAM, false>);
}

template <typename real>
hipError_t launch_mixed_cols(typename Vec2<real>::type* data, const FftAxis& r, int Nc, int mode, const real* mask, const void* rowf,
                             const void* colf, typename Vec2<real>::type* spec, hipStream_t s) {
    const ColFactor<real> f{mode, mask, (const Cx<real>*)rowf, (const Cx<real>*)colf, spec, Nc, r.N, (real)((double)Nc * (double)r.N)};
    const size_t per = 2 * (size_t)r.fwd.len * sizeof(Cx<real>);
    if (!r.fwd.passes || per > kMixLdsMax) return hipErrorInvalidValue;
    /* two columns per workgroup while two workgroups still fit a CU's LDS: one column reads 8 or 16 bytes of
       each 128-byte line (600 x 600 FP64: 39.5 us a filter with one, 32.9 with two, 36.5 with four; 1500 x
       1500 FP64, 96 KiB for two, 104 / 120).  Bluestein's lengths take one: their buffers are twice to four
       times as long (1030 x 1030 FP32: 185 / 223) */
    const int fam = radix_family(r.fwd.len);
    if (r.M) return fam == 0 ? cols_cb<real, 1, true, 0>(data, r, f, s) : cols_cb<real, 1, true, 1>(data, r, f, s);
    if (2 * per <= 65536 && Nc > 1)
        return fam < 2 ? cols_cb<real, 2, false, 1>(data, r, f, s) : cols_cb<real, 2, false, 2>(data, r, f, s);
    return fam < 2 ? cols_cb<real, 1, false, 1>(data, r, f, s) : cols_cb<real, 1, false, 2>(data, r, f, s);
}

template hipError_t launch_mixed_rows<float>(float2*, const FftAxis&, int, bool, hipStream_t);
template hipError_t launch_mixed_rows<double>(double2*, const FftAxis&, int, bool, hipStream_t);
template hipError_t launch_mixed_cols<float>(float2*, const FftAxis&, int, int, const float*, const void*, const void*, float2*, hipStream_t);
template hipError_t launch_mixed_cols<double>(double2*, const FftAxis&, int, int, const double*, const void*, const void*, double2*, hipStream_t);

} // namespace phx
