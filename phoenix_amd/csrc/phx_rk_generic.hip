/*
 * phx_rk_generic.hip -- instantiations of the fused Runge-Kutta kernel
 * (phx_rk_generic.h) for RK4 (with noise or TE-TM; the plain scalar RK4 has its own
 * hand-tuned kernel in phx_rk4.h) and Dormand-Prince 5(4) fixed and adaptive, the
 * deterministic reduction of the adaptive error partials, the per-step noise field, the
 * imaginary-time normalisation, and the dispatch over all tableaux (the other groups are instantiated in phx_rk_tab3.hip,
 * phx_rk_tab4.hip, phx_rk_tab6.hip and phx_rk_tab6f.hip).
 */
#include <algorithm>
#include <cstdlib>

#include "phx_rk_generic.h"

namespace phx {

/* deterministic reduction of the per-wave partials: one workgroup, fixed order */
constexpr int kReduceThreads = 1024;
__global__ __launch_bounds__(kReduceThreads) void reduce_partials(const double* __restrict__ partials, int nwaves, double* __restrict__ out) {
    __shared__ double se[kReduceThreads], sn[kReduceThreads];
    double e = 0, n = 0;
    for (int i = threadIdx.x; i < nwaves; i += kReduceThreads) {
        e += partials[2 * i];
        n += partials[2 * i + 1];
    }
    se[threadIdx.x] = e;
    sn[threadIdx.x] = n;
    __syncthreads();
    for (int w = kReduceThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            se[threadIdx.x] += se[threadIdx.x + w];
            sn[threadIdx.x] += sn[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = se[0];
        out[1] = sn[0];
    }
}

hipError_t launch_reduce_partials(const double* partials, int nwaves, double* sums, hipStream_t s) {
    hipLaunchKernelGGL(reduce_partials, dim3(1), dim3(kReduceThreads), 0, s, partials, nwaves, sums);
    return hipGetLastError();
}

/* per-256-cell FP64 sums of |psi+|^2 and |psi-|^2, fixed order inside the block */
template <typename real>
__global__ __launch_bounds__(256) void sumsq_blocks(const typename Vec2<real>::type* __restrict__ a,
                                                    const typename Vec2<real>::type* __restrict__ b, size_t cells,
                                                    double* __restrict__ partials) {
    __shared__ double sa[256], sb[256];
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    double x = 0.0, y = 0.0;
    if (i < cells) {
        const auto u = a[i];
        x = (double)u.x * (double)u.x + (double)u.y * (double)u.y;
        if (b) {
            const auto v = b[i];
            y = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
        }
    }
    sa[threadIdx.x] = x;
    sb[threadIdx.x] = y;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            sa[threadIdx.x] += sa[threadIdx.x + w];
            sb[threadIdx.x] += sb[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = sa[0];
        partials[2 * blockIdx.x + 1] = sb[0];
    }
}

/* psi_k *= sqrt(amp / (S_k dV)), S_k < 1e-10 -> 1 (solver_normalize_imag_time.cu:13-45) */
template <typename real>
__global__ __launch_bounds__(256) void imag_scale(typename Vec2<real>::type* __restrict__ a, typename Vec2<real>::type* __restrict__ b,
                                                  size_t cells, const double* __restrict__ sums, double amp, double dV) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= cells) return;
    const double s0 = sums[0] < 1e-10 ? 1.0 : sums[0];
    const real f0 = (real)sqrt(amp / (s0 * dV));
    auto u = a[i];
    u.x *= f0;
    u.y *= f0;
    a[i] = u;
    if (b) {
        const double s1 = sums[1] < 1e-10 ? 1.0 : sums[1];
        const real f1 = (real)sqrt(amp / (s1 * dV));
        auto v = b[i];
        v.x *= f1;
        v.y *= f1;
        b[i] = v;
    }
}

template <typename real>
hipError_t launch_imag_normalize(typename Vec2<real>::type* psi_plus, typename Vec2<real>::type* psi_minus, size_t cells,
                                 double amp, double dV, double* partials, double* sums, hipStream_t s) {
    const size_t nb = imag_norm_blocks(cells);
    hipLaunchKernelGGL(sumsq_blocks<real>, dim3((unsigned)nb), dim3(256), 0, s, psi_plus, psi_minus, cells, partials);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((e = launch_reduce_partials(partials, (int)nb, sums, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(imag_scale<real>, dim3((unsigned)nb), dim3(256), 0, s, psi_plus, psi_minus, cells, sums, amp, dV);
    return hipGetLastError();
}

template hipError_t launch_imag_normalize<float>(float2*, float2*, size_t, double, double, double*, double*, hipStream_t);
template hipError_t launch_imag_normalize<double>(double2*, double2*, size_t, double, double, double*, double*, hipStream_t);

/* one complex normal pair per cell, scaled by amp (own Philox stream, see phx_noise.h) */
template <typename real>
__global__ __launch_bounds__(256) void noise_field(typename Vec2<real>::type* __restrict__ xi, uint32_t cells, uint64_t seed,
                                                   uint64_t step, real amp) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= cells) return;
    real zr, zi;
    phx_noise_normal2<real>(seed, step, i, 0, zr, zi);
    typename Vec2<real>::type z;
    z.x = zr * amp;
    z.y = zi * amp;
    xi[i] = z;
}

template <typename real>
hipError_t launch_noise_field(typename Vec2<real>::type* xi, int Nc, int Nr, uint64_t seed, uint64_t step, real amp,
                              hipStream_t s) {
    const size_t cells = (size_t)Nc * (size_t)Nr;
    if (cells * sizeof(typename Vec2<real>::type) > kMaxArrayBytes) return hipErrorInvalidValue;
    hipLaunchKernelGGL(noise_field<real>, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, s, xi, (uint32_t)cells, seed,
                       step, amp);
    return hipGetLastError();
}

template hipError_t launch_noise_field<float>(float2*, int, int, uint64_t, uint64_t, float, hipStream_t);
template hipError_t launch_noise_field<double>(double2*, int, int, uint64_t, uint64_t, double, hipStream_t);

int rk4_simds() {
    static const int simds = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            cus = 256;
        return 4 * std::max(cus, 1);
    }();
    return simds;
}

Rk4Tune rk4_default_tune(int Nc, int Nr, size_t real_size) {
    /* The rows of a tile are a serial chain: a grid that fits the SIMDs in one round takes the shortest tile
       that does.  Up to two rounds FP32 runs best at 10 rows (two waves a SIMD cover each other's waits);
       FP64, whose waves issue twice the work a row, at one round of 20; larger grids are within 5 % of their
       best at 16.  us per launch at 16 rows and by this rule: 200 x 150 FP32 7.3 and 3.7, FP64 8.7 and 4.4;
       400^2 7.7 / 4.5, 9.2 / 5.4; 512^2 7.7 / 5.5, 9.4 / 6.8; 768^2 8.4 / 7.1, 10.4 / 8.8; 1024^2 11.2 / 9.2,
       16.0 / 13.5; 1500^2 16.0, 25.0. */
    Rk4Tune t;
    for (int ty : {2, 4, 8, 12})
        if (rk4_tiles(Nc, Nr, ty) <= rk4_simds()) {
            t.ty = ty;
            return t;
        }
    if (real_size == 4 && rk4_tiles(Nc, Nr, 10) <= 2 * rk4_simds()) t.ty = 10;
    if (real_size == 8 && rk4_tiles(Nc, Nr, 20) <= rk4_simds()) t.ty = 20;
    return t;
}

int rk4_generic_tile_rows(int Nc, int Nr) {
    if (const char* e = std::getenv("PHX_RK4G_TY")) return std::atoi(e); /* 4, 8 or 16 */
    /* The model of dp45_adaptive_tile_rows for four stages: rounds of tiles over the SIMDs x row evaluations
       of a tile.  A tile's rows are a serial chain, so a grid that does not fill the chip wants short tiles,
       and a large one tall tiles, which recompute fewer halo rows.  TE-TM, us per step alone / with two other
       grids in flight, 4, 8 and 16 rows (the rule's choice in brackets): 200^2 FP64 [12.5 / 4.4] 16 / 5.6
       26 / 8.9; 480 x 640 FP64 24 / 16.7 [19 / 13.6] 29 / 13.5; 1200^2 FP64 75 / 85 64 / 66 [60 / 57];
       one-component chain kernel at 512 x 384 FP32 [8.4 / 3.4] 8.8 / 3.5 12.1 / 4.7. */
    constexpr int S = 4;
    int best = 16;
    long best_cost = -1;
    for (int ty : {16, 8, 4}) {
        const long waves = (long)((Nc + 55) / 56) * ((Nr + ty - 1) / ty);
        const long cost = ((waves + rk4_simds() - 1) / rk4_simds()) * (long)(S * (ty + 2 * S) - S * (S + 1));
        if (best_cost < 0 || cost < best_cost) best = ty, best_cost = cost;
    }
    return best;
}

int dp45_adaptive_tile_rows(bool tetm, bool fp32, int Nc, int Nr) {
    const bool tall = tetm && fp32; /* the tall tiles exist for the FP32 spinor kernel */
    const char* e = std::getenv("PHX_GEN_TY"); /* read at every launch: tests switch it within a process */
    const int env_ty = e ? std::atoi(e) : 0;
    if (env_ty == 8 || env_ty == 16 || (tall && (env_ty == 28 || env_ty == 32 || env_ty == 42))) return env_ty;
    /* One wave per SIMD at the kernel's register count (over 256 VGPRs + AGPRs at every height),
       and about the same VALU work per row evaluation at every height (135-148 instructions): a
       grid's time is its blocks in rounds over the CUs (rounded up) times the row evaluations of one
       tile, S (TY + 2 S) - S (S + 1) for S = 7.  us per attempt, FP32 TE-TM, 8 / 16 / 28 / 32 / 42 rows
       (the rule's choice in brackets): 2048^2 with noise 365 / 318 / 242 / 266 / [229], without 303 / 265 /
       202 / 221 / [190]; 1536 x 1200 148 / 141 / 137 / 150 / [103]; 1024^2 95 / 99 / [78] / 85 / 101; 600^2
       [43] / 56 / 72 / 79 / 95; FP64 1024^2 [488] / 482, 300^2 [126] / 171. */
    constexpr int S = 7;
    int best = kRkGenTileRows;
    long best_cost = -1;
    for (int ty : {16, 8, 28, 32, 42}) {
        if (ty > kRkGenTileRows && !tall) continue;
        /* the 42-row tiles address ten rows further past the grid's end than the 32-row ones (launch_gen): a
           grid of nearly 2 GiB a field stays with those */
        if (ty > 32 && (size_t)Nc * (size_t)(Nr + ty + S) * sizeof(float2) > kMaxArrayBytes) continue;
        const long blocks = tile_blocks((Nc + 63 - 2 * S) / (64 - 2 * S), (Nr + ty - 1) / ty), cus = rk4_simds() / 4;
        const long cost = ((blocks + cus - 1) / cus) * (long)(S * (ty + 2 * S) - S * (S + 1));
        if (best_cost < 0 || cost < best_cost) best = ty, best_cost = cost;
    }
    return best;
}

template <typename real>
hipError_t launch_rk_generic(const RkGenArgs<real>& a, RkTableau tab, hipStream_t s) {
    switch (tab) {
        case RkTableau::RK4: return launch_rk4_generic<real>(a, s);
        case RkTableau::DP45_FIXED: return launch_tab<real, TabDP45Fixed>(a, s);
        case RkTableau::DP45_ADAPTIVE: {
            const int ty = dp45_adaptive_tile_rows(a.tetm, sizeof(real) == 4, a.Nc, a.Nr);
            if constexpr (sizeof(real) == 4)
                if (ty > kRkGenTileRows && a.tetm) return launch_dp45_tetm_tall(a, ty, s);
            return launch_dp45_adaptive<real>(a, ty, s);
        }
        case RkTableau::NEWTON:
        case RkTableau::MP:
        case RkTableau::HEUN2:
        case RkTableau::RALSTON:
        case RkTableau::HEUN3:
        case RkTableau::RALSTON3:
        case RkTableau::RK3:
        case RkTableau::SSPRK3:
        case RkTableau::HW: return launch_rk_tab3<real>(a, tab, s);
        case RkTableau::FEHLBERG2:
        case RkTableau::FEHLBERG2_ADAPTIVE:
        case RkTableau::RALSTON4:
        case RkTableau::RULE38:
        case RkTableau::BOSHA:
        case RkTableau::BOSHA_ADAPTIVE: return launch_rk_tab4<real>(a, tab, s);
        case RkTableau::NYSTROEM:
        case RkTableau::CASHKARP:
        case RkTableau::CASHKARP_ADAPTIVE: return launch_rk_tab6<real>(a, tab, s);
        case RkTableau::FEHLBERG5:
        case RkTableau::FEHLBERG5_ADAPTIVE: return launch_rk_tab6f<real>(a, tab, s);
        /* more stages than the fused kernel keeps in registers: staged path (launch_staged) */
        case RkTableau::NSRK78:
        case RkTableau::NSRK78_ADAPTIVE:
        case RkTableau::DP85:
        case RkTableau::DP85_ADAPTIVE: return hipErrorInvalidValue;
    }
    return hipErrorInvalidValue;
}

template hipError_t launch_rk_generic<float>(const RkGenArgs<float>&, RkTableau, hipStream_t);
template hipError_t launch_rk_generic<double>(const RkGenArgs<double>&, RkTableau, hipStream_t);

} // namespace phx
