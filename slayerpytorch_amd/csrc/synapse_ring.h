// 3x3 gathers with stride 1 that keep three source rows in LDS (synapse_ring.hip).
#ifndef SLAYER_CSRC_SYNAPSE_RING_H
#define SLAYER_CSRC_SYNAPSE_RING_H

#include "common.h"

namespace slayer {

// dst[n][m][a][b][t] = sum over source channels q of m's group and taps (i, j) of weight(m, q, i, j) src[n][q][y][x][t], with
// y = a - padH + i, x = b - padW + j (forward) or y = a + padH - i, x = b + padW - j (the input gradient)
struct RingGeom {
    const float *src, *w;
    float *dst;
    int N, SC, SH, SW, DC, DH, DW, T, groups, Qg, Mg, Cg, Og, padH, padW;
};

// SLAYER_EUNSUPPORTED (nothing launched) for geometries that the kernel does not take - it takes 16 or 32 source and at least
// 16 destination channels per group, rows of whole vectors or at least 32 samples - and for sizes at which another is faster.
template <bool BACKWARD> int launch_gather_ring(const RingGeom &s, hipStream_t st);

// The weight gradient of the same geometry, src the input [N][SC][SH][SW][T], dst (read) the output gradient: rows of partial
// sums [Og groups][Cg][9] in `workspace`, ring_wgrad_rows() of them (0: not a geometry for it, or another kernel is faster), to be added up.
int ring_wgrad_rows(const RingGeom &s);
int launch_wgrad_ring(const RingGeom &s, float *workspace, hipStream_t st);

}  // namespace slayer

#endif
