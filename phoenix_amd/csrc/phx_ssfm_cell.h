/*
 * phx_ssfm_cell.h -- device math of the split-step iterator's pointwise steps (library functions).
 */
#pragma once
#include <hip/hip_runtime.h>

namespace phx {

__device__ __forceinline__ void phx_sincos_dev(float x, float& s, float& c) { sincosf(x, &s, &c); }
__device__ __forceinline__ void phx_sincos_dev(double x, double& s, double& c) { sincos(x, &s, &c); }
__device__ __forceinline__ float phx_exp_dev(float x) { return expf(x); }
__device__ __forceinline__ double phx_exp_dev(double x) { return exp(x); }

} // namespace phx
