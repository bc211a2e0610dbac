/*
 * phx_rk4_batch.hip -- FP32 instantiations of the batched RK4 kernel of phx_rk4.h (in translation units of
 * their own, so that they compile in parallel).
 */
#include "phx_rk4.h"

namespace phx {

template hipError_t launch_rk4_batched<float>(const Rk4BatchArgs<float>&, int, bool, bool, bool, hipStream_t);

} // namespace phx
