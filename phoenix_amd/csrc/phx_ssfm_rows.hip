/*
 * phx_ssfm_rows.hip -- the row pass between two linear half steps of the split-step iterator: inverse row
 * transform, the pointwise step in real space, forward row transform, one kernel over LDS.
 *
 * Scalar model with a real reservoir.  Between the column passes of two propagations the reference's
 * sequence (split_step_fourier_method.cu:25-71) is inverse rows, gp_scalar_nonlinear, forward rows: three
 * kernels that each read and write psi.  Here a row stays in LDS from the inverse transform's last pass to
 * the forward one's first, and what the cells need from memory (n, V, P) is requested before the inverse
 * transform starts.  Bound by the latency of the passes (LDS round trips and their barriers), as the other
 * transforms of these lengths: 1024 x 512 FP32 17.1 us instead of 20.0 for the
 * three kernels.
 */
#include "phx_fft_engine.h"
#include "phx_kernels.h"
#include "phx_noise.h"
#include "phx_ssfm_cell.h"

namespace phx {

namespace {

/* gp_scalar_nonlinear (kernel_gp_compute.cuh:264-382) of one cell, as ssfm_nonlinear */
template <typename real>
struct CellNonlinear {
    SsfmArgs<real> a;
    struct Pre {
        real n, vr, vi, p;
    };
    __device__ __forceinline__ Pre load(size_t i) const {
        Pre q{a.n_cur[0] ? a.n_cur[0][i] : real(0), real(0), real(0), real(0)};
        for (int g = 0; g < a.npot; g++) {
            const real v = a.pot[0][g][i];
            q.vr += v * a.vamp[g].x;
            q.vi += v * a.vamp[g].y;
        }
        if (a.n_nxt[0])
            for (int g = 0; g < a.npump; g++) q.p += a.pump[0][g][i] * a.pamp[g];
        return q;
    }
    __device__ __forceinline__ void apply(const Pre& q, size_t i, Cx<real>& z) const {
        const PhxPhys<real>& ph = a.ph;
        const real nrm = phx_fma(z.r, z.r, z.i * z.i);
        real A = ph.g_c * nrm;
        A += q.vr;
        A += ph.g_r * q.n;
        if (a.stochastic) A -= ph.g_c / ph.dV;
        const real er = phx_fma(a.dt * ph.one_over_h_bar_s, q.vi, a.dt * (real(0.5) * (ph.R * q.n - ph.gamma_c)));
        real sn, cs;
        phx_sincos_dev(-(A * ph.one_over_h_bar_s * a.dt), sn, cs);
        const real m = phx_exp_dev(er);
        z = cmul(z, Cx<real>{m * cs, m * sn});
        if (a.n_nxt[0]) {
            real rn = -(ph.gamma_r * q.n);
            rn -= ph.R * nrm * q.n;
            rn += q.p;
            if (a.stochastic) rn += ph.R * q.n / ph.dV;
            a.n_nxt[0][i] = phx_fma(rn, a.dt, q.n);
        }
    }
};

/* the pulse of gp_scalar_independent (kernel_gp_compute.cuh:392-396): psi += (dt / hbar) sum_g F_g a_g */
template <typename real>
struct CellPulse {
    SsfmArgs<real> a;
    struct Pre {
        real r, i;
    };
    __device__ __forceinline__ Pre load(size_t i) const {
        Pre q{real(0), real(0)};
        const real f = a.dt * a.ph.one_over_h_bar_s;
        for (int g = 0; g < a.npulse; g++) {
            const auto F = a.pulse[0][g][i];
            const auto am = a.lamp[g];
            q.r += f * phx_fma(F.x, am.x, -(F.y * am.y));
            q.i += f * phx_fma(F.x, am.y, F.y * am.x);
        }
        return q;
    }
    __device__ __forceinline__ void apply(const Pre& q, size_t, Cx<real>& z) const {
        z.r += q.r;
        z.i += q.i;
    }
};

} // namespace

template <typename real, bool BLUE, int FAM, class OP>
__global__ __launch_bounds__(kMixThreads) void rows_cell_rows(typename Vec2<real>::type* data, FftPlan fwd, FftPlan inv, int N, int Nr,
                                                              int rpb, const Cx<real>* __restrict__ table, OP op) {
    const int row0 = blockIdx.x * rpb, count = min(rpb, Nr - row0), cells = count * N, len = fwd.len;
    const size_t cell0 = (size_t)row0 * N;
    constexpr int U = 4; /* cells of a thread whose inputs are in flight together */
    typename OP::Pre pre[U];
#pragma unroll
    for (int u = 0; u < U; u++) pre[u] = op.load(cell0 + min((int)(threadIdx.x + u * blockDim.x), cells - 1));

    int A = 0, B = rpb * len;
    typename Vec2<real>::type* rows = data + cell0;
    auto load_swapped = [&](int seq, int i) {
        const auto v = rows[(size_t)seq * N + i];
        return Cx<real>{v.y, v.x};
    };
    auto store = [&](int seq, int i, Cx<real> f) {
        typename Vec2<real>::type o;
        o.x = f.r;
        o.y = f.i;
        rows[(size_t)seq * N + i] = o;
    };
    const Cx<real>*tw = BLUE ? table + N : table, *chirp = tw + len, *hat = chirp + N;
    auto by_hat = [&](int, int bb, int nb, auto& x) {
        constexpr int R = sizeof(x) / sizeof(x[0]);
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = cmul(x[j], hat[bb + j * nb]);
    };
    /* inverse transform (parts swapped on the way in and out) into the LDS buffer its last pass leaves free */
    if constexpr (BLUE)
        convolve<real, 0, FAM>(
            fwd, inv, count, A, B, tw,
            [&](int seq, int i) { return i < N ? cmul(load_swapped(seq, i), chirp[i]) : Cx<real>{real(0), real(0)}; }, by_hat,
            [&](int seq, int i, Cx<real> f) {
                if (i < N) lds<real>()[B + seq * len + i] = swapped(cmul(swapped(f), chirp[i]));
            });
    else
        transform<real, 0, FAM>(fwd, count, A, B, tw, load_swapped,
                                [&](int seq, int i, Cx<real> f) { lds<real>()[B + seq * len + i] = swapped(f); });
    __syncthreads();
    Cx<real>* const z = lds<real>() + B;
    for (int base = threadIdx.x; base < cells; base += U * blockDim.x) {
        if (base != (int)threadIdx.x) {
#pragma unroll
            for (int u = 0; u < U; u++) pre[u] = op.load(cell0 + min((int)(base + u * blockDim.x), cells - 1));
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = base + u * blockDim.x;
            if (i < cells) {
                const int k = BLUE && rpb > 1 ? i / N * len + i % N : i;
                op.apply(pre[u], cell0 + i, z[k]);
            }
        }
    }
    __syncthreads();
    int A2 = B, B2 = A;
    if constexpr (BLUE)
        convolve<real, 0, FAM>(
            fwd, inv, count, A2, B2, tw,
            [&](int seq, int i) { return i < N ? cmul(z[seq * len + i], chirp[i]) : Cx<real>{real(0), real(0)}; }, by_hat,
            [&](int seq, int i, Cx<real> f) {
                if (i < N) store(seq, i, cmul(swapped(f), chirp[i]));
            });
    else
        transform<real, 0, FAM>(fwd, count, A2, B2, tw, [&](int seq, int i) { return z[seq * len + i]; }, store);
}

template <typename real, class OP>
static hipError_t launch_rows_cell(const FftAxis& c, int Nr, const OP& op, hipStream_t s) {
    const int len = c.fwd.len, rpb = rows_per_block(c.fwd);
    const size_t lds = 2 * (size_t)len * rpb * sizeof(Cx<real>);
    if (!c.fwd.passes || lds > kMixLdsMax) return hipErrorInvalidValue;
    const dim3 grid((Nr + rpb - 1) / rpb), blk(mixed_threads(widest_pass(c.fwd) * rpb));
    auto go = [&](auto kernel) {
        const hipError_t e = allow_lds(kernel, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, blk, lds, s, op.a.psi[0], c.fwd, c.inv, c.N, Nr, rpb, (const Cx<real>*)c.table, op);
        return hipGetLastError();
    };
    const int fam = radix_family(len);
    if (c.M) return fam == 0 ? go(&rows_cell_rows<real, true, 0, OP>) : go(&rows_cell_rows<real, true, 1, OP>);
    return fam == 0   ? go(&rows_cell_rows<real, false, 0, OP>)
           : fam == 1 ? go(&rows_cell_rows<real, false, 1, OP>)
                      : go(&rows_cell_rows<real, false, 2, OP>);
}

template <typename real>
hipError_t launch_ssfm_rows(const SsfmArgs<real>& a, const FftAxis& c, int Nr, bool pulse, hipStream_t s) {
    if (a.tetm || a.cres) return hipErrorInvalidValue;
    return pulse ? launch_rows_cell<real>(c, Nr, CellPulse<real>{a}, s) : launch_rows_cell<real>(c, Nr, CellNonlinear<real>{a}, s);
}

template hipError_t launch_ssfm_rows<float>(const SsfmArgs<float>&, const FftAxis&, int, bool, hipStream_t);
template hipError_t launch_ssfm_rows<double>(const SsfmArgs<double>&, const FftAxis&, int, bool, hipStream_t);

} // namespace phx
