/*
 * phx_rk4_f64.hip -- FP64 instantiations of the one-step RK4 kernel of phx_rk4.h (the two
 * precisions live in separate translation units so that they compile in parallel).
 */
#include "phx_rk4.h"

namespace phx {

template hipError_t launch_rk4_scalar<double>(const Rk4Args<double>&, const Rk4Tune&, hipStream_t);

} // namespace phx
