/*
 * phx_row_wrap.h -- grid rows of a tile's rows in the streaming kernels, in plain C++ so that it compiles for
 * the host too.
 */
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define PHX_HD __host__ __device__ __forceinline__
#else
#define PHX_HD inline
#endif

namespace phx {

/* Walk over the grid rows of consecutive tile rows, upwards (dir 1) or downwards (dir -1), without branches, so that
   a fully unrolled row loop stays one basic block (a branch there splits it, and DPP moves then no longer fold into
   the adds that consume them): one add, one compare and one select a row.  A periodic axis turns at its end, whatever
   its length; beyond a zero boundary the row is out of range (next_row says so) and counts on.  (A quotient by a
   reciprocal took four scalar operations a row and was wrong for one row and for more than 37837; six made it exact.
   us per pass with four, six and the walk: FP64 512 x 512 with a pulse, 10 steps, 44.6 / 46.4 / 44.3; FP64 spinor DP45 of
   134 x 134 1675 / 1740 / 1672; FP32 adjoint of 12 x 185 x 153 1235 / 1246 / 1206.) */
struct RowWalk {
    uint32_t row, step, stop, turn, nr;
};
/* from tile row `first` >= -halo on: next_row moves there first */
PHX_HD RowWalk make_row_walk(int first, int dir, int Nr, int halo, bool periodic) {
    RowWalk w;
    w.nr = (uint32_t)Nr;
    w.step = (uint32_t)dir;
    const uint32_t before = (uint32_t)(first - dir);
    const uint32_t bias = Nr > halo ? w.nr : w.nr * (uint32_t)(halo + 1); /* a multiple of Nr past halo */
    w.row = periodic ? (before + bias) % w.nr : before;
    w.stop = periodic ? (dir > 0 ? w.nr : 0xFFFFFFFFu) : 0x80000000u; /* the last: never reached */
    w.turn = dir > 0 ? 0u : w.nr - 1u;
    return w;
}
/* the next row; whether it lies in the grid */
PHX_HD bool next_row(RowWalk& w) {
    const uint32_t t = w.row + w.step;
    w.row = t == w.stop ? w.turn : t;
    return w.row < w.nr;
}

} // namespace phx
