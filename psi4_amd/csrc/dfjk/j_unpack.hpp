// J from its partial sums (kernels.hip; kernels_f64.hip runs it beside the reduction of K).
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"

namespace p4a {
namespace {

// J from the partials of every Q chunk.  A workgroup sums 128 elements (4 rows) of one tile, the
// chunks dealt to 8 groups of threads and added in LDS in a fixed order, and writes each element
// with its mirror image, so J is exactly symmetric.  Bound by latency at small sizes: one thread
// per element of J walking every chunk took 145 us at nbf 96 (464 chunks) and 36 us at nbf 576
// (24 chunks); this takes 9 us and 11 us.  Tiles that are not stored stay at the caller's zeros
// (or are zeroed by k_j_clear when not accumulating).
constexpr int kJuGroups = 8;
__device__ __forceinline__ void j_unpack_block(const JUnpack& u, int t, int part, int p, double* red) {
    const int el = threadIdx.x & 127, grp = threadIdx.x >> 7;
    const int e = part * 128 + el;
    const double* __restrict__ Jp = u.Jpart + p * u.pstride + static_cast<size_t>(t) * TILE2 + e;
    double s = 0.0;
#pragma unroll 4
    for (int c = grp; c < u.nchunk; c += kJuGroups) s += Jp[static_cast<size_t>(c) * u.ntp * TILE2];
    red[grp * 128 + el] = s;
    __syncthreads();
    if (grp != 0) return;
    double v = red[el];
#pragma unroll
    for (int g = 1; g < kJuGroups; ++g) v += red[g * 128 + el];
    const int2 IJ = u.tiles[t];
    const int m = IJ.x * TILE + e / TILE, n = IJ.y * TILE + e % TILE;
    if (m >= u.nbf || n >= u.nbf || m > n) return;  // the lower triangle of a diagonal tile is its mirror image
    double* __restrict__ J = u.out.J[p];
    double* o = J + static_cast<size_t>(m) * u.ldJ + n;
    *o = u.alpha * v + (u.accumulate ? *o : 0.0);
    if (m != n) {
        double* ot = J + static_cast<size_t>(n) * u.ldJ + m;
        *ot = u.alpha * v + (u.accumulate ? *ot : 0.0);
    }
}

}  // namespace
}  // namespace p4a
