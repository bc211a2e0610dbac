/*
 * phx_fft_cx.h -- complex values of the LDS transforms and the order in which column groups are
 * handed out, shared by phx_fft.hip and phx_fft_mixed.hip.
 */
#pragma once
#include <hip/hip_runtime.h>

#include "custom_rhs.h"

namespace phx {

/* aligned to its full size, so an element moves with one 64-bit (FP32) / 128-bit (FP64) LDS access */
template <typename real>
struct alignas(2 * sizeof(real)) Cx {
    real r, i;
};

template <typename real>
__device__ __forceinline__ Cx<real> cmul(Cx<real> a, Cx<real> w) {
    return {phx_fma(a.r, w.r, -(a.i * w.i)), phx_fma(a.r, w.i, a.i * w.r)};
}

/* Column groups are handed out XCD by XCD (block b runs on XCD b % 8): consecutive
   groups share cache lines, so they go to the same L2. */
__device__ __forceinline__ int fft_xcd_group(int b, int nblocks) {
    const int q = nblocks >> 3, r = nblocks & 7;
    const int x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

} // namespace phx
