/*
 * phx_fft_engine.h -- device side of the mixed-radix transforms: Stockham passes over LDS with their
 * ends in the caller's hands (phx_fft_mixed.hip: rows, columns; phx_ssfm_rows.hip: the split-step rows).
 */
#pragma once
#include <type_traits>

#include "phx_fft_cx.h"
#include "phx_fft_mixed.h"

namespace phx {

/* ------------------------------------------------------------------ transforms in registers */
/* cos and sin of 2 pi k / R to more digits than a double holds, k / R in lowest terms below one half; the compiler
   rounds them once (a Taylor series in double was off by up to 1.6 units: the rotations by an eighth of a turn shrank
   what they turned by 0.8 units of 2^-53, and with it a split-step run) */
inline constexpr struct {
    int k, R;
    double c, s;
} kTurns[] = {
    {1, 3, -0.500000000000000000000, 0.866025403784438646764},  {1, 5, 0.309016994374947424102, 0.951056516295153572116},
    {2, 5, -0.809016994374947424102, 0.587785252292473129169},  {1, 7, 0.623489801858733530525, 0.781831482468029808708},
    {2, 7, -0.222520933956314404289, 0.974927912181823607018},  {3, 7, -0.900968867902419126236, 0.433883739117558120476},
    {1, 8, 0.707106781186547524401, 0.707106781186547524401},   {3, 8, -0.707106781186547524401, 0.707106781186547524401},
    {1, 9, 0.766044443118978035202, 0.642787609686539326323},   {2, 9, 0.173648177666930348852, 0.984807753012208059367},
    {4, 9, -0.939692620785908384054, 0.342020143325668733044},  {1, 10, 0.809016994374947424102, 0.587785252292473129169},
    {3, 10, -0.309016994374947424102, 0.951056516295153572116}, {1, 11, 0.841253532831181168862, 0.540640817455597582108},
    {2, 11, 0.415415013001886425529, 0.909631995354518371412},  {3, 11, -0.142314838273285140444, 0.989821441880932732376},
    {4, 11, -0.654860733945285064057, 0.755749574354258283774}, {5, 11, -0.959492973614497389890, 0.281732556841429697711},
    {1, 13, 0.885456025653209895900, 0.464723172043768545656},  {2, 13, 0.568064746731155802512, 0.822983865893656394580},
    {3, 13, 0.120536680255323053349, 0.992708874098053992801},  {4, 13, -0.354604887042535625970, 0.935016242685414823440},
    {5, 13, -0.748510748171101098635, 0.663122658240795202377}, {6, 13, -0.970941817426052027157, 0.239315664287557767149},
    {1, 16, 0.923879532511286756128, 0.382683432365089771728},  {3, 16, 0.382683432365089771728, 0.923879532511286756128},
    {5, 16, -0.382683432365089771728, 0.923879532511286756128}, {7, 16, -0.923879532511286756128, 0.382683432365089771728},
};
struct Turn {
    double c, s;
};
/* of k Rths of a turn, R one of the radices */
constexpr Turn turn(int k, int R) {
    k %= R;
    if (k == 0) return {1.0, 0.0};
    if (2 * k == R) return {-1.0, 0.0};
    if (2 * k > R) {
        const Turn t = turn(R - k, R);
        return {t.c, -t.s};
    }
    if (4 * k == R) return {0.0, 1.0};
    for (const auto& t : kTurns)
        if (k * t.R == t.k * R) return {t.c, t.s};
    return {0.0, 0.0}; /* not reached */
}

template <int R>
struct Roots {
    double c[R] = {}, s[R] = {};
    constexpr Roots() {
        for (int k = 0; k < R; k++) {
            c[k] = turn(k, R).c;
            s[k] = turn(k, R).s;
        }
    }
};
template <int R>
struct RootTable {
    static constexpr Roots<R> v{};
};

/* factor of a composite radix that is transformed first */
constexpr int first_factor(int R) { return R % 4 == 0 && R > 4 ? 4 : R % 2 == 0 ? 2 : R % 3 == 0 ? 3 : R; }

/* forward DFT of R values in registers */
template <typename real, int R>
__device__ __forceinline__ void dft(Cx<real> (&x)[R]) {
    if constexpr (R == 2) {
        const Cx<real> a = x[0], b = x[1];
        x[0] = {a.r + b.r, a.i + b.i};
        x[1] = {a.r - b.r, a.i - b.i};
    } else if constexpr (R == 4) {
        const Cx<real> s02 = {x[0].r + x[2].r, x[0].i + x[2].i}, d02 = {x[0].r - x[2].r, x[0].i - x[2].i};
        const Cx<real> s13 = {x[1].r + x[3].r, x[1].i + x[3].i}, d13 = {x[1].r - x[3].r, x[1].i - x[3].i};
        x[0] = {s02.r + s13.r, s02.i + s13.i};
        x[1] = {d02.r + d13.i, d02.i - d13.r};
        x[2] = {s02.r - s13.r, s02.i - s13.i};
        x[3] = {d02.r - d13.i, d02.i + d13.r};
    } else if constexpr (first_factor(R) != R) {
        /* R = R1 R2: n = R2 n1 + n2, k = k1 + R1 k2 */
        constexpr int R1 = first_factor(R), R2 = R / R1;
        Cx<real> y[R2][R1];
#pragma unroll
        for (int n2 = 0; n2 < R2; n2++) {
            Cx<real> t[R1];
#pragma unroll
            for (int n1 = 0; n1 < R1; n1++) t[n1] = x[R2 * n1 + n2];
            dft<real, R1>(t);
#pragma unroll
            for (int k1 = 0; k1 < R1; k1++) {
                const int m = (n2 * k1) % R;
                y[n2][k1] = m == 0 ? t[k1] : cmul(t[k1], Cx<real>{(real)RootTable<R>::v.c[m], (real)-RootTable<R>::v.s[m]});
            }
        }
#pragma unroll
        for (int k1 = 0; k1 < R1; k1++) {
            Cx<real> t[R2];
#pragma unroll
            for (int n2 = 0; n2 < R2; n2++) t[n2] = y[n2][k1];
            dft<real, R2>(t);
#pragma unroll
            for (int k2 = 0; k2 < R2; k2++) x[k1 + R1 * k2] = t[k2];
        }
    } else {
        /* odd prime: sums and differences of the pairs k, R - k */
        constexpr int P = (R - 1) / 2;
        Cx<real> t[P], u[P];
        Cx<real> z = x[0];
#pragma unroll
        for (int k = 0; k < P; k++) {
            t[k] = {x[k + 1].r + x[R - 1 - k].r, x[k + 1].i + x[R - 1 - k].i};
            u[k] = {x[k + 1].r - x[R - 1 - k].r, x[k + 1].i - x[R - 1 - k].i};
            z.r += t[k].r;
            z.i += t[k].i;
        }
        const Cx<real> x0 = x[0];
        x[0] = z;
#pragma unroll
        for (int j = 1; j <= P; j++) {
            Cx<real> a = x0, b = {real(0), real(0)};
#pragma unroll
            for (int k = 0; k < P; k++) {
                const int m = (j * (k + 1)) % R;
                const real c = (real)RootTable<R>::v.c[m], s = (real)RootTable<R>::v.s[m];
                a.r = phx_fma(c, t[k].r, a.r);
                a.i = phx_fma(c, t[k].i, a.i);
                b.r = phx_fma(s, u[k].r, b.r);
                b.i = phx_fma(s, u[k].i, b.i);
            }
            x[j] = {a.r + b.i, a.i - b.r};
            x[R - j] = {a.r - b.i, a.i + b.r};
        }
    }
}

template <typename real>
__device__ __forceinline__ Cx<real> swapped(Cx<real> v) {
    return {v.i, v.r};
}

/* ------------------------------------------------------------------------------ the passes */

/* Butterfly b of a group of sequences -> (sequence, butterfly of the sequence), and the LDS slot of
   an element.  Rows: one sequence after the other; columns: the CB columns adjacent. */
template <int CB>
struct Lay {
    static __device__ __forceinline__ void split(int b, int nb, uint32_t m_nb, int& seq, int& bb) {
        if constexpr (CB > 0) {
            seq = b % CB;
            bb = b / CB;
        } else {
            seq = nb == 1 ? b : (int)__umulhi((uint32_t)b, m_nb);
            bb = b - seq * nb;
        }
    }
    static __device__ __forceinline__ int slot(int seq, int idx, int len) {
        if constexpr (CB > 0)
            return idx * CB + seq;
        else
            return seq * len + idx;
    }
};

/* the workgroup's LDS; the two buffers are kept as offsets into it, not as pointers (a pointer that is
   exchanged in a loop loses its address space, and every access becomes a flat one) */
template <typename real>
__device__ __forceinline__ Cx<real>* lds() {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    return reinterpret_cast<Cx<real>*>(lds_raw);
}

/* entry i of a plan array by selects: the plan is a kernel argument, and an indexed read of it would be a
   scalar load in the middle of the kernel instead of one of those at its start */
template <typename T>
__device__ __forceinline__ T pick(const T (&v)[kFftMaxPasses], int i) {
    T r = v[0];
#pragma unroll
    for (int k = 1; k < kFftMaxPasses; k++) r = i == k ? v[k] : r;
    return r;
}

/* One pass of radix R.  Inputs come from rd(seq, idx) when `first`, else from A; outputs go to
   wr(seq, idx, value) when `last`, else to B (element offsets in LDS). */
template <typename real, int R, int CB, class RD, class WR>
__device__ __forceinline__ void one_pass(const FftPlan& pl, int i, int count, bool first, bool last, int A, int B,
                                         const Cx<real>* __restrict__ tw, RD rd, WR wr) {
    const int nb = pl.len / R, s = pick(pl.s, i), total = nb * count;
    const uint32_t m_nb = pick(pl.m_nb, i), m_s = pick(pl.m_s, i);
    Cx<real>* const L = lds<real>();
    for (int b = threadIdx.x; b < total; b += blockDim.x) {
        int seq, bb;
        Lay<CB>::split(b, nb, m_nb, seq, bb);
        const int p = s == 1 ? bb : (int)__umulhi((uint32_t)bb, m_s), ps = p * s, q = bb - ps;
        Cx<real> x[R], w[R];
#pragma unroll
        for (int j = 1; j < R; j++) w[j] = tw[last ? 0 : j * ps];
        if (first) {
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = rd(seq, bb + j * nb);
        } else {
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = L[A + Lay<CB>::slot(seq, bb + j * nb, pl.len)];
        }
        dft<real, R>(x);
        if (last) {
#pragma unroll
            for (int j = 0; j < R; j++) wr(seq, bb + j * s, x[j]);
        } else {
            const int o = q + R * ps;
            L[B + Lay<CB>::slot(seq, o, pl.len)] = x[0];
#pragma unroll
            for (int j = 1; j < R; j++) L[B + Lay<CB>::slot(seq, o + s * j, pl.len)] = cmul(x[j], w[j]);
        }
    }
}

/* The turn of a convolution: the last forward pass, the factor, and the first pass of the inverse
   (radices reversed, real and imaginary parts swapped), which takes the same elements. */
template <typename real, int R, int CB, class RD, class FA, class WR>
__device__ __forceinline__ void turn_pass(const FftPlan& pl, int i, int count, bool first, int A, int B,
                                          const Cx<real>* __restrict__ tw, RD rd, FA factor, WR wr) {
    const int nb = pl.len / R, total = nb * count;
    const uint32_t m_nb = pick(pl.m_nb, i);
    Cx<real>* const L = lds<real>();
    for (int b = threadIdx.x; b < total; b += blockDim.x) {
        int seq, bb;
        Lay<CB>::split(b, nb, m_nb, seq, bb);
        Cx<real> x[R], w[R];
#pragma unroll
        for (int j = 1; j < R; j++) w[j] = tw[j * bb];
        if (first) {
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = rd(seq, bb + j * nb);
        } else {
#pragma unroll
            for (int j = 0; j < R; j++) x[j] = L[A + Lay<CB>::slot(seq, bb + j * nb, pl.len)];
        }
        dft<real, R>(x);
        factor(seq, bb, nb, x);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = swapped(x[j]);
        dft<real, R>(x);
        if (first) { /* a single pass: the whole transform */
#pragma unroll
            for (int j = 0; j < R; j++) wr(seq, bb + j, x[j]);
        } else {
            L[B + Lay<CB>::slot(seq, R * bb, pl.len)] = x[0];
#pragma unroll
            for (int j = 1; j < R; j++) L[B + Lay<CB>::slot(seq, R * bb + j, pl.len)] = cmul(x[j], w[j]);
        }
    }
}

/* run `f` with the radix as a compile-time constant, out of a family of radices: 0 the powers of two,
   1 with 3, 5, 9 and 10, 2 with 7, 11 and 13 too.  Every pass of a kernel holds the code of its whole
   family, and the instruction cache is 64 KiB for two CUs: a filter of 646 x 646 (Bluestein, 2048
   points) takes 100 us FP64 / 60 us FP32 with family 0 and 122 / 77 with family 1. */
template <int FAM, class F>
__device__ __forceinline__ void with_radix(int r, F f) {
    switch (r) {
        case 2: f(std::integral_constant<int, 2>{}); return;
        case 4: f(std::integral_constant<int, 4>{}); return;
        case 8: f(std::integral_constant<int, 8>{}); return;
        case 16: f(std::integral_constant<int, 16>{}); return;
        default: break;
    }
    if constexpr (FAM >= 1) {
        switch (r) {
            case 3: f(std::integral_constant<int, 3>{}); return;
            case 5: f(std::integral_constant<int, 5>{}); return;
            case 9: f(std::integral_constant<int, 9>{}); return;
            case 10: f(std::integral_constant<int, 10>{}); return;
            default: break;
        }
    }
    if constexpr (FAM >= 2) {
        switch (r) {
            case 7: f(std::integral_constant<int, 7>{}); return;
            case 11: f(std::integral_constant<int, 11>{}); return;
            case 13: f(std::integral_constant<int, 13>{}); return;
            default: break;
        }
    }
}

/* forward transform of `count` sequences: rd -> wr.  The last pass reads the buffer that A names on return:
   B is free for wr. */
template <typename real, int CB, int FAM, class RD, class WR>
__device__ __forceinline__ void transform(const FftPlan& pl, int count, int& A, int& B, const Cx<real>* __restrict__ tw, RD rd, WR wr) {
    for (int i = 0; i < pl.passes; i++) {
        const bool last = i == pl.passes - 1;
        with_radix<FAM>(pick(pl.radix, i), [&](auto R) { one_pass<real, decltype(R)::value, CB>(pl, i, count, i == 0, last, A, B, tw, rd, wr); });
        if (last) break;
        __syncthreads();
        const int t = A;
        A = B;
        B = t;
    }
}

/* forward, factor, inverse (its real and imaginary parts still swapped when they reach wr).  The
   last pass reads the buffer that is returned as the second one: the first is free for wr. */
template <typename real, int CB, int FAM, class RD, class FA, class WR>
__device__ __forceinline__ void convolve(const FftPlan& fwd, const FftPlan& inv, int count, int& A, int& B,
                                         const Cx<real>* __restrict__ tw, RD rd, FA factor, WR wr) {
    const int last_fwd = fwd.passes - 1;
    auto flip = [&] {
        const int t = A;
        A = B;
        B = t;
    };
    for (int i = 0; i < last_fwd; i++) {
        with_radix<FAM>(pick(fwd.radix, i), [&](auto R) { one_pass<real, decltype(R)::value, CB>(fwd, i, count, i == 0, false, A, B, tw, rd, wr); });
        __syncthreads();
        flip();
    }
    with_radix<FAM>(pick(fwd.radix, last_fwd),
                     [&](auto R) { turn_pass<real, decltype(R)::value, CB>(fwd, last_fwd, count, last_fwd == 0, A, B, tw, rd, factor, wr); });
    for (int i = 1; i <= last_fwd; i++) {
        __syncthreads();
        flip();
        const bool last = i == last_fwd;
        with_radix<FAM>(pick(inv.radix, i), [&](auto R) { one_pass<real, decltype(R)::value, CB>(inv, i, count, false, last, A, B, tw, rd, wr); });
    }
}

/* threads of the row and column kernels, and the LDS that the two buffers of a workgroup may take of the
   160 KiB a gfx950 workgroup may hold */
constexpr int kMixThreads = 256;
constexpr size_t kMixLdsMax = 128 * 1024;

/* host helpers of the launchers */
inline int largest_prime(int n) {
    int big = 1;
    for (int p = 2; p * p <= n; p++)
        while (n % p == 0) big = p, n /= p;
    return n > big ? n : big;
}
/* family of radices (with_radix) that splits a length */
inline int radix_family(int len) {
    const int p = largest_prime(len);
    return p <= 2 ? 0 : p <= 5 ? 1 : 2;
}
/* butterflies of one sequence in the widest pass */
inline int widest_pass(const FftPlan& p) {
    int r = p.radix[0];
    for (int i = 1; i < p.passes; i++) r = p.radix[i] < r ? p.radix[i] : r;
    return p.len / r;
}
/* threads of a workgroup with `work` butterflies in its widest pass */
inline int mixed_threads(int work) {
    const int t = (work + 63) / 64 * 64;
    return t < kMixThreads ? t : kMixThreads;
}
/* as few rows per workgroup as fill its waves: the transforms wait on LDS and L2, and more, smaller
   workgroups spread the waits (400 x 400 FP64: 1 row 23.2 us a filter, 3 rows 23.3; 1500 x 1500 FP32
   67.0 / 69.4; 138 x 158 FP64, Bluestein, 27.3 / 30.9 for 1 and 4 rows) */
inline int rows_per_block(const FftPlan& p) {
    const int w = widest_pass(p);
    return w < 64 ? 64 / w : 1;
}
template <typename K>
inline hipError_t allow_lds(K kernel, size_t lds) {
    return lds > 65536 ? hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMixLdsMax) : hipSuccess;
}

} // namespace phx
