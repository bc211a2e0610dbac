/*
 * phx_rk_chain.hip -- RK4 under source chains (pulses, pumps and potentials of several temporal groups,
 * complex temporal amplitudes) in one launch per step: the fused kernel of phx_rk_generic.h with one
 * register window per source group.
 *
 * The staged path (phx_staged.hip) takes any tableau and up to eight groups of each source, with one
 * launch per stage and sum and every K in HBM: at 512 x 384 FP32 with a pump, a potential and a pulse
 * eight launches of 4-5 us a step, 30 us a step with other work in between.  RK4 is the default
 * iterator and sources rarely have more than two groups (a continuous and a timed one), so that case
 * keeps its K's in registers: 8.9 us a step alone (39 staged), 3.7 us with other work in between.  Bound
 * by the chain of a tile's rows at that size (960 waves of 12 rows), by VALU issue on large grids.
 */
#include "phx_rk_generic.h"

namespace phx {

template <typename real, int TY, bool TETM, bool RES, bool STOCH, int NG>
__global__ __launch_bounds__(256) void rk_chain_fused(RkGenArgs<real> a, RkChainArgs<real> ch) {
    rk_generic_tile<real, TabRK4, TY, TETM, RES, STOCH, true, NG>(a, ch);
}

bool rk_chain_supported(int Nc, int Nr, int groups, size_t real_size) {
    /* 32-bit offsets reach every group of a source and the dropped stores past the grid end */
    return groups <= kChainGroups && (size_t)Nc * ((size_t)std::max(groups, 1) * Nr + 16 + kChainStages) * 2 * real_size <= kMaxArrayBytes;
}

template <typename real, int TY, bool TETM, bool RES, bool STOCH>
static hipError_t launch_chain_ng(const RkGenArgs<real>& a0, const RkChainArgs<real>& ch, hipStream_t s) {
    RkGenArgs<real> a = a0;
    constexpr int outw = kWave - 2 * TabRK4::S;
    a.nstrips = (a.Nc + outw - 1) / outw;
    a.nbands = (a.Nr + TY - 1) / TY;
    const dim3 grid(tile_blocks(a.nstrips, a.nbands)), blk(kWave * kWavesPerBlock);
    if (std::max(std::max(ch.npump, ch.npot), ch.npulse) <= 1)
        hipLaunchKernelGGL((rk_chain_fused<real, TY, TETM, RES, STOCH, 1>), grid, blk, 0, s, a, ch);
    else
        hipLaunchKernelGGL((rk_chain_fused<real, TY, TETM, RES, STOCH, 2>), grid, blk, 0, s, a, ch);
    return hipGetLastError();
}

template <typename real, int TY>
static hipError_t launch_chain_ty(const RkGenArgs<real>& a, const RkChainArgs<real>& ch, hipStream_t s) {
    const bool res = a.n_in[0] != nullptr;
    if (a.tetm) {
        if (res) return a.stochastic ? launch_chain_ng<real, TY, true, true, true>(a, ch, s) : launch_chain_ng<real, TY, true, true, false>(a, ch, s);
        return a.stochastic ? launch_chain_ng<real, TY, true, false, true>(a, ch, s) : launch_chain_ng<real, TY, true, false, false>(a, ch, s);
    }
    if (res) return a.stochastic ? launch_chain_ng<real, TY, false, true, true>(a, ch, s) : launch_chain_ng<real, TY, false, true, false>(a, ch, s);
    return a.stochastic ? launch_chain_ng<real, TY, false, false, true>(a, ch, s) : launch_chain_ng<real, TY, false, false, false>(a, ch, s);
}

template <typename real>
hipError_t launch_rk_chain(const RkGenArgs<real>& a, const RkChainArgs<real>& ch, hipStream_t s) {
    if (!rk_chain_supported(a.Nc, a.Nr, std::max(std::max(ch.npump, ch.npot), ch.npulse), sizeof(real))) return hipErrorInvalidValue;
    switch (rk4_generic_tile_rows(a.Nc, a.Nr)) {
        case 4: return launch_chain_ty<real, 4>(a, ch, s);
        case 8: return launch_chain_ty<real, 8>(a, ch, s);
        default: return launch_chain_ty<real, 16>(a, ch, s);
    }
}

template hipError_t launch_rk_chain<float>(const RkGenArgs<float>&, const RkChainArgs<float>&, hipStream_t);
template hipError_t launch_rk_chain<double>(const RkGenArgs<double>&, const RkChainArgs<double>&, hipStream_t);

} // namespace phx
