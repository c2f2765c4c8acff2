// Dense algebra of the set-up for gfx950: diagonal blocks of the metric's Cholesky factor, and the
// fit B = M (P|mn) by the FP64 MFMA.
//
// MFMA lane layout, 16x16x4 f64: A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k, D[i][j] in lane
// j + 16 (i % 4), register i / 4.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "kernels_fit.hpp"

namespace p4a {

namespace {

typedef double d2_t __attribute__((ext_vector_type(2)));
constexpr int kXCD = 8;

__device__ inline d2_t ld2(const double* base, unsigned off) {
    return *reinterpret_cast<const d2_t*>(reinterpret_cast<const char*>(base) + off);
}
__device__ inline double ld1(const double* base, unsigned off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
}

// 1 / sqrt(x): the hardware's estimate and one step of third order, e = 1 - x y^2, y + y e (1/2 + 3/8 e), which
// leaves (5/16) e^3: with |e| < 2^-23 (the estimate is within 2^-24.1 on 4 million x in [1, 4)) that is
// below 2^-70, and the result within 2^-52.6 there, where 1 / sqrt(x) by a rounded root and division is within 2^-52.4.  A
// sixth of the latency of those.
__device__ inline double rsqrt_refined(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// ------------------------------------------------------------------ L_kk^-1
// One workgroup, the block in registers: thread (ty, tx) holds rows ty + 32 a, columns tx + 32 b.  At
// step k, with r = 1 / sqrt(T_kk), row i > k takes T_ij -= l_i w_j, l_i = T_ik r, where column j > k
// still holds A (w_j = l_j) and column j < k already holds L^-1 (w_j = T_kj r); row k becomes row k of
// L^-1.  Row and column k go through LDS, double buffered: one barrier a step.  Bound by that chain
// (root, barrier, LDS): 128 steps take 74 us, of the 32 x 32 blocks only those that still change and lie on or
// below the diagonal (88 us with every block and a division; 114 us when every wave computes the
// root); factor and inverse on the host, with the copies to and from it, took 7 ms per 256 rows.
__global__ __launch_bounds__(1024) void k_chol_inverse(const double* __restrict__ A, int lda, int nb, int k0,
                                                       double* __restrict__ X, int ldx, double* __restrict__ LiT,
                                                       int* __restrict__ info) {
    __shared__ double vb[2][kCholBlock], cb[2][kCholBlock], rb[2];
    const int ty = threadIdx.x >> 5, tx = threadIdx.x & 31;
    double T[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = ty + 32 * a, j = tx + 32 * b;
            // rows and columns past nb: the identity
            T[a][b] = (i < nb && j <= i) ? A[static_cast<size_t>(i) * lda + j] : (i == j ? 1.0 : 0.0);
        }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll 1
        for (int kk = 0; kk < 32; ++kk) {
            const int k = 32 * kb + kk, par = kk & 1;
            if (tx == kk) {
#pragma unroll
                for (int a = kb; a < 4; ++a) cb[par][ty + 32 * a] = T[a][kb];
                // the pivot's reciprocal root, by the one wave that holds it
                if (ty == kk) {
                    if (!(T[kb][kb] > 0.0)) atomicMin(info, k0 + k);
                    rb[par] = rsqrt_refined(T[kb][kb]);
                }
            }
            if (ty == kk)
#pragma unroll
                for (int b = 0; b <= kb; ++b) vb[par][tx + 32 * b] = T[kb][b];
            __syncthreads();
            const double r = rb[par];
            double l[4], w[4];
#pragma unroll
            for (int a = kb; a < 4; ++a) l[a] = cb[par][ty + 32 * a] * r;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int j = tx + 32 * b;
                w[b] = (j < k ? vb[par][j] : cb[par][j]) * r;
            }
#pragma unroll
            for (int a = kb; a < 4; ++a)
#pragma unroll
                for (int b = 0; b <= a; ++b) {
                    const int i = ty + 32 * a, j = tx + 32 * b;
                    if (i > k)
                        T[a][b] = j == k ? -l[a] * r : fma(-l[a], w[b], T[a][b]);
                    else if (i == k)
                        T[a][b] = j < k ? w[b] : r;
                }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = ty + 32 * a, j = tx + 32 * b;
            if (i >= nb || j >= nb) continue;
            const double v = j <= i ? T[a][b] : 0.0;
            X[static_cast<size_t>(i) * ldx + j] = v;
            LiT[static_cast<size_t>(j) * nb + i] = v;
        }
}

// ------------------------------------------------------------------ fit
// MF[k8][16 rows][lane][2]: row lane % 16, column 8 kb + 2 (lane / 16) + e
__global__ __launch_bounds__(256) void k_fit_pack(const double* __restrict__ M, int na, int nrb, int nkb,
                                                  double* __restrict__ MF) {
    const size_t n = static_cast<size_t>(nrb) * nkb * 128;
    for (size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; idx < n; idx += static_cast<size_t>(gridDim.x) * 256) {
        const int e = idx & 1, lane = static_cast<int>(idx >> 1) & 63;
        const size_t rest = idx >> 7;
        const int kb = static_cast<int>(rest / nrb), rb = static_cast<int>(rest % nrb);
        const int i = 16 * rb + (lane & 15), k = 8 * kb + 2 * (lane >> 4) + e;
        MF[idx] = (i < na && k < na) ? M[static_cast<size_t>(i) * na + k] : 0.0;
    }
}

// One wave: NC 16-row blocks x 64 columns
template <int NC>
__device__ __forceinline__ void fit_body(const double* __restrict__ MF, int na, int nrb, int rb0, int kend,
                                         const double* __restrict__ A, size_t lda, double* __restrict__ out, size_t ldo) {
    const int lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const unsigned off_m = lane * 16, off_a = static_cast<unsigned>((2 * lg * lda + lj) * 8);
    d4_t acc[4][NC];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < NC; ++i) acc[f][i] = d4_t{0.0, 0.0, 0.0, 0.0};
    d2_t a0[4], a1[4], m0[NC], m1[NC];
    const int nfull = kend / 8;  // whole steps of 8 rows of A
    auto mload = [&](int kb, d2_t* m) {
        const double* p = MF + (static_cast<size_t>(kb) * nrb + rb0) * 128;
#pragma unroll
        for (int i = 0; i < NC; ++i) m[i] = ld2(p + 128 * i, off_m);
    };
    auto load = [&](int kb, d2_t* a, d2_t* m) {
        kb = min(kb, nfull - 1);
        const double* p = A + static_cast<size_t>(8 * kb) * lda;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            a[f].x = ld1(p + 16 * f, off_a);
            a[f].y = ld1(p + 16 * f + lda, off_a);
        }
        mload(kb, m);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const d2_t* a, const d2_t* m) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    acc[f][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[i][e], a[f][e], acc[f][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (nfull > 0) {
        load(0, a0, m0);
        int kb = 0;
        for (; kb + 1 < nfull; kb += 2) {
            load(kb + 1, a1, m1);
            mul(a0, m0);
            load(kb + 2, a0, m0);
            mul(a1, m1);
        }
        if (kb < nfull) mul(a0, m0);
    }
    if (kend % 8) {
        // the last rows: those past na read row na - 1, against zeros of M
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                a0[f][e] = A[static_cast<size_t>(min(8 * nfull + 2 * lg + e, na - 1)) * lda + 16 * f + lj];
        mload(nfull, m0);
        mul(a0, m0);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (rb0 + i) + 4 * r + lg;
            if (row < na)
#pragma unroll
                for (int f = 0; f < 4; ++f) out[static_cast<size_t>(row) * ldo + 16 * f + lj] = acc[f][i][r];
        }
}

// Groups of NC (the first ones) and NC - 1 row blocks; 16 strips of 64 columns go to one XCD, all row
// groups of a strip with them, the longest (last) rows first, so that the waves in flight share
// rows of M and columns of A in the XCD's L2.  Bound by the MFMA pipes: na 5568 / 682 k columns (2.1e13
// flops of the lower triangle) take 291 ms (73 TFLOP/s), and took 383 ms with 128 x 128 LDS tiles; na
// 1856 / 80 k columns 4.6 ms against 5.5.
template <int NC>
__global__ __launch_bounds__(256, 2) void k_fit(const double* __restrict__ MF, int na, int nrb, int nrg,
                                                const double* __restrict__ A, size_t lda, int ngroups,
                                                double* __restrict__ out, size_t ldo, int lower) {
    const int wg = blockIdx.x, lw = (wg / kXCD) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int items = nrg * 16, group = (lw / items) * kXCD + wg % kXCD, item = lw % items;
    if (group >= ngroups) return;
    const int rg = nrg - 1 - item / 16;
    const size_t j0 = (static_cast<size_t>(group) * 16 + item % 16) * 64;
    const int nwide = nrb - nrg * (NC - 1);
    const int rb0 = rg * NC - max(0, rg - nwide);
    const int n = rg < nwide ? NC : NC - 1;
    const int kend = lower ? min(na, 16 * (rb0 + n)) : na;
    if (rg < nwide)
        fit_body<NC>(MF, na, nrb, rb0, kend, A + j0, lda, out + j0, ldo);
    else if constexpr (NC > 1)
        fit_body<NC - 1>(MF, na, nrb, rb0, kend, A + j0, lda, out + j0, ldo);
}

inline int fit_row_blocks(int na) { return (na + 15) / 16; }

}  // namespace

void launch_chol_inverse(const double* A, int lda, int nb, int k0, double* X, int ldx, double* LiT, int* info,
                         hipStream_t s) {
    require(nb > 0 && nb <= kCholBlock && lda >= nb && ldx >= nb, "chol_inverse");
    hipLaunchKernelGGL(k_chol_inverse, dim3(1), dim3(1024), 0, s, A, lda, nb, k0, X, ldx, LiT, info);
}

size_t fit_packed_size(int na) { return static_cast<size_t>(fit_row_blocks(na)) * ((na + 7) / 8) * 128; }

void launch_fit_pack(const double* M, int na, double* MF, hipStream_t s) {
    require(na > 0, "fit_pack");
    const size_t nb = std::min<size_t>((fit_packed_size(na) + 255) / 256, size_t(1) << 16);
    hipLaunchKernelGGL(k_fit_pack, dim3(static_cast<unsigned>(nb)), dim3(256), 0, s, M, na, fit_row_blocks(na),
                       (na + 7) / 8, MF);
}

void launch_fit(const double* MF, int na, const double* A, size_t lda, size_t w, double* out, size_t ldo, bool lower,
                hipStream_t s) {
    // a lane's offset into A (6 rows) is a 32-bit byte count
    require(na > 0 && w > 0 && w % 1024 == 0 && lda >= w && ldo >= w && 8 * lda * 8 < (size_t(1) << 32), "fit");
    const int nrb = fit_row_blocks(na), nrg = (nrb + 4) / 5, nc = (nrb + nrg - 1) / nrg;
    const int ngroups = static_cast<int>(w / 1024);
    const long long per = static_cast<long long>((ngroups + kXCD - 1) / kXCD) * nrg * 16;
    const dim3 grid(static_cast<unsigned>(kXCD * ((per + 3) / 4)));
#define P4A_FIT(N)                                                                                                    \
    case N:                                                                                                           \
        hipLaunchKernelGGL((k_fit<N>), grid, dim3(256), 0, s, MF, na, nrb, nrg, A, lda, ngroups, out, ldo, lower ? 1 : 0); \
        break;
    switch (nc) { P4A_FIT(1) P4A_FIT(2) P4A_FIT(3) P4A_FIT(4) P4A_FIT(5) }
#undef P4A_FIT
}

}  // namespace p4a
