// Launchers of the set-up's dense algebra on the device: the diagonal blocks of the metric's Cholesky
// factor, and the fit B = M (P|mn).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace p4a {

constexpr int kCholBlock = 128;
// A_kk (nb x nb at A, leading dimension lda, lower triangle read, nb <= kCholBlock) = L L^T:
// X (leading dimension ldx) = L^-1 with zeros above the diagonal, LiT [nb][nb] = (L^-1)^T.
// *info becomes min(*info, k0 + k) at a pivot k that is not positive.
void launch_chol_inverse(const double* A, int lda, int nb, int k0, double* X, int ldx, double* LiT, int* info,
                         hipStream_t s);

// Doubles of the packed metric factor
size_t fit_packed_size(int na);
// M [na][na] -> MF, the fit's operand in MFMA fragment order
void launch_fit_pack(const double* M, int na, double* MF, hipStream_t s);
// out[i][j] = sum_k M[i][k] A[k][j] for i < na, j < w (w a multiple of 1024); lower: M[i][k] = 0 for k > i
void launch_fit(const double* MF, int na, const double* A, size_t lda, size_t w, double* out, size_t ldo, bool lower,
                hipStream_t s);

}  // namespace p4a
