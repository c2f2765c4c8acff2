// Launchers of the FP32 K path (kernels_f32.hip): the wave-level kernels of the FP64 path with FP32
// operands, FP32 MFMA and FP64 partial sums.  Columns come in groups padded to 16; X and the
// half-transform's operand are stored in MFMA fragment order, 16 columns (rows) deep.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "kernels_f64.hpp"

namespace p4a {

// CA32 [nbfp/16][ncb][64][4]
void launch_pack_frag32(const ColGroups& cg, int nbf, int nbfp, float* CA, hipStream_t s);
// X[q][nbfp/16][ncb][64][4] = B_q C, q < nq, from the FP32 copy of B
void launch_ht_f32(const TileGeom& g, const float* B, int nq, const float* CA, int ncb, int rt, float* X, const void* zt,
                   hipStream_t s);
// Output blocks of 64 rows x 32 columns over nT 32-column blocks; a partial sum is kc32_partial doubles
int kc32_blocks(int nT, bool upper);
constexpr size_t kc32_partial = 2048;
// P[split][block][8 sub-tiles][4][64] (+)= the passes (KcSeg with k in units of 16 columns)
void launch_kc_f32(const float* X, size_t qstride, int nkx, int nT, int nq, const KcSegs& segs, bool upper, double* P,
                   int accumulate, hipStream_t s);
int kc32_choose_splits(int nT, bool upper, int steps, int nseg, int max_splits);
void launch_kc32_reduce(const double* P, int nT, int n, bool upper, const KcOuts& outs, int accumulate, hipStream_t s);

}  // namespace p4a
