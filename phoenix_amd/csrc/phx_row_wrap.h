/*
 * phx_row_wrap.h -- periodic row index of the streaming kernels, in plain C++ so that it compiles for the
 * host too.
 */
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define PHX_HD __host__ __device__ __forceinline__
#else
#define PHX_HD inline
#endif

namespace phx {

/* Periodic row wrap without branches, so that a fully unrolled row loop stays one
   basic block (a branch there splits it, and DPP moves then no longer fold into the
   adds that consume them).  With x = g + bias >= 0 and magic = floor((2^32 - 1) / Nr),
   mulhi(x, magic) is x / Nr or one less for every x < 2^32 and Nr >= 1 (magic is short of 2^32 / Nr by
   at most one, so the product by at most x / 2^32 < 1), hence one conditional subtraction;
   g >= -halo, and bias = Nr (Nr >= halo) or Nr * halo keeps x from going negative. */
struct RowWrap {
    uint32_t nr, magic, bias;
};
PHX_HD RowWrap make_row_wrap(int Nr, int halo) {
    RowWrap w;
    w.nr = (uint32_t)Nr;
    w.magic = 0xFFFFFFFFu / (uint32_t)Nr;
    w.bias = Nr >= halo ? (uint32_t)Nr : (uint32_t)(Nr * halo);
    return w;
}
/* Row of tile row g: wrapped into [0, Nr) (for a zero boundary `in` says whether g lies in the grid, the
   wrapped row is then unused). */
PHX_HD uint32_t tile_row(int g, const RowWrap& w, int periodic, bool& in) {
    in = periodic || (g >= 0 && g < (int)w.nr);
    const uint32_t x = (uint32_t)g + w.bias;
    const uint32_t r = x - (uint32_t)(((uint64_t)x * w.magic) >> 32) * w.nr; /* in [0, 2 Nr) */
    const uint32_t less = r - w.nr;                                          /* past every r where r < Nr */
    return r < less ? r : less;
}

} // namespace phx
