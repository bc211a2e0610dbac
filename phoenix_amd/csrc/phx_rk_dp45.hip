/*
 * phx_rk_dp45.hip -- the adaptive Dormand-Prince 5(4) kernel in tiles of 8 and 16 rows (the tall FP32 TE-TM
 * ones: phx_rk_dp45t.hip), in a translation unit of its own.
 */
#include "phx_rk_generic.h"

namespace phx {

template <typename real>
hipError_t launch_dp45_adaptive(const RkGenArgs<real>& a, int ty, hipStream_t s) {
    if (ty == 8) return dispatch_flags<real, TabDP45Adaptive, 8>(a, s);
    return dispatch_flags<real, TabDP45Adaptive, kRkGenTileRows>(a, s);
}

template hipError_t launch_dp45_adaptive<float>(const RkGenArgs<float>&, int, hipStream_t);
template hipError_t launch_dp45_adaptive<double>(const RkGenArgs<double>&, int, hipStream_t);

} // namespace phx
