// DF-JK device kernels for gfx950 (CDNA4), FP64 path.
//
// Data layout in HBM (all row-major, FP64):
//   B      [naux][ntp][TILE][TILE]  fitted three-index tensor, stored as the
//          TILE x TILE blocks (I,J), I <= J, of each symmetric B_Q; diagonal
//          blocks hold both triangles.  Blocks with no Schwarz-significant pair
//          are not stored (tile-granular screening).
//   C      [nbfp][ldc]              orbital coefficients, zero-padded.
//
// MFMA lane layouts used here (verified on the device):
//   v_mfma_f64_16x16x4f64: A[i][k] in lane i+16k, B[k][j] in lane j+16k,
//                          D[i][j] in lane j+16*(i%4), register i/4.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "j_unpack.hpp"
#include "kernels.hpp"

namespace p4a {

namespace {

inline dim3 grid1(size_t n, int block) { return dim3(static_cast<unsigned>((n + block - 1) / block)); }

// ------------------------------------------------------------------ J path
__global__ void k_pack_w(const double* __restrict__ D, int ldD, int nbf, const int2* __restrict__ tiles,
                         double* __restrict__ W) {
    const int t = blockIdx.x;
    const int2 IJ = tiles[t];
    for (int e = threadIdx.x; e < TILE2; e += blockDim.x) {
        const int r = e / TILE, c = e % TILE;
        const int m = IJ.x * TILE + r, n = IJ.y * TILE + c;
        double v = 0.0;
        if (m < nbf && n < nbf) {
            v = D[static_cast<size_t>(m) * ldD + n];
            if (IJ.x != IJ.y) v += D[static_cast<size_t>(n) * ldD + m];
        }
        W[static_cast<size_t>(t) * TILE2 + e] = v;
    }
}

// Element loaders of the resident tensor for the J path (FP64 accumulation in every case).
// load4 / load8 read 4 / 8 consecutive elements (i a multiple of 4 / 8) with 16-byte vector
// loads per lane.
typedef double d2_t __attribute__((ext_vector_type(2)));
typedef float f4v_t __attribute__((ext_vector_type(4)));
struct BSrcF64 {
    const double* p;
    __device__ void load4(size_t i, double* v) const {
        const d2_t a = *reinterpret_cast<const d2_t*>(p + i), b = *reinterpret_cast<const d2_t*>(p + i + 2);
        v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    }
    __device__ void load8(size_t i, double* v) const {
        load4(i, v);
        load4(i + 4, v + 4);
    }
};
struct BSrcF32 {
    const float* p;
    __device__ void load4(size_t i, double* v) const {
        const f4v_t a = *reinterpret_cast<const f4v_t*>(p + i);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    }
    __device__ void load8(size_t i, double* v) const {
        load4(i, v);
        load4(i + 4, v + 4);
    }
};
// d_Q partials: one wave per Q, the density tile of pair t held in registers (lane l holds
// elements 8l..8l+7 and 512+8l..512+8l+7).  Each wave takes two Q per pass, so two tiles
// are in flight.  grid = (ntp, ceil((q1-q0)/qblk)), 256 threads.
template <class BS>
__global__ __launch_bounds__(256) void k_j1(BS B, const double* __restrict__ W, int ntp, int naux, int q0, int q1,
                                            int qblk, double* __restrict__ dpart) {
    const int t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double* Wt = W + static_cast<size_t>(t) * TILE2;
    double w[16];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) w[8 * c + e] = Wt[512 * c + 8 * lane + e];
    const int qa = q0 + blockIdx.y * qblk;
    const int qb = min(q1, qa + qblk);
    auto dot = [&](int Q) {
        const size_t base = (static_cast<size_t>(Q) * ntp + t) * TILE2 + 8 * lane;
        double v[16];
        B.load8(base, v);
        B.load8(base + 512, v + 8);
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) s = fma(v[k], w[k], s);
        return s;
    };
    for (int Q = qa + wave; Q < qb; Q += 8) {
        const int Q2 = Q + 4;
        double s = dot(Q);
        double s2 = Q2 < qb ? dot(Q2) : 0.0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            s += __shfl_xor(s, off);
            s2 += __shfl_xor(s2, off);
        }
        if (lane == 0) {
            dpart[static_cast<size_t>(t) * naux + Q] = s;
            if (Q2 < qb) dpart[static_cast<size_t>(t) * naux + Q2] = s2;
        }
    }
}

// d_Q = sum over the tile pairs of the partials.  64 Q per workgroup, the tile pairs dealt to 16
// waves (a wave's loads are 512 contiguous bytes, several in flight), their sums added in LDS in a
// fixed order.  Bound by latency: one thread per Q walking every pair took 70 us at 171 pairs /
// 2784 Q and 33 us at 78 / 1856; this takes 5 us at both.
constexpr int kJ1Groups = 16;
__global__ __launch_bounds__(64 * kJ1Groups) void k_j1_reduce(const double* __restrict__ dpart, int ntp, int naux,
                                                             double* __restrict__ d) {
    __shared__ double red[kJ1Groups][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int Q = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (Q < naux) {
#pragma unroll 8
        for (int t = grp; t < ntp; t += kJ1Groups) s += dpart[static_cast<size_t>(t) * naux + Q];
    }
    red[grp][lane] = s;
    __syncthreads();
    if (grp == 0 && Q < naux) {
        double v = red[0][lane];
#pragma unroll
        for (int g = 1; g < kJ1Groups; ++g) v += red[g][lane];
        d[Q] = v;
    }
}

// J partials over a chunk of Q: grid = (ntp, nchunk), 256 threads, 4 consecutive elements per
// thread (vector loads), two Q per pass.  NP densities share the pass over B (d[p * ldd + Q], partials
// at Jpart + p * pstride): bound by reading B, so a second density costs next to nothing.
template <class BS, int NP>
__global__ __launch_bounds__(256) void k_j2(BS B, const double* __restrict__ d, int ldd, int ntp, int naux, int qchunk,
                                            double* __restrict__ Jpart, size_t pstride) {
    const int t = blockIdx.x, c = blockIdx.y;
    const int qa = c * qchunk, qb = min(naux, qa + qchunk);
    const int e0 = 4 * threadIdx.x;
    double a[NP][4] = {};
    int Q = qa;
    for (; Q + 1 < qb; Q += 2) {
        const size_t base = (static_cast<size_t>(Q) * ntp + t) * TILE2 + e0;
        double v0[4], v1[4];
        B.load4(base, v0);
        B.load4(base + static_cast<size_t>(ntp) * TILE2, v1);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const double d0 = d[static_cast<size_t>(p) * ldd + Q], d1 = d[static_cast<size_t>(p) * ldd + Q + 1];
#pragma unroll
            for (int k = 0; k < 4; ++k) a[p][k] = fma(v1[k], d1, fma(v0[k], d0, a[p][k]));
        }
    }
    if (Q < qb) {
        double v0[4];
        B.load4((static_cast<size_t>(Q) * ntp + t) * TILE2 + e0, v0);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const double d0 = d[static_cast<size_t>(p) * ldd + Q];
#pragma unroll
            for (int k = 0; k < 4; ++k) a[p][k] = fma(v0[k], d0, a[p][k]);
        }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        double* o = Jpart + p * pstride + (static_cast<size_t>(c) * ntp + t) * TILE2 + e0;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = a[p][k];
    }
}

__global__ __launch_bounds__(128 * kJuGroups) void k_j_unpack(JUnpack u) {
    __shared__ double red[128 * kJuGroups];
    j_unpack_block(u, blockIdx.x, blockIdx.y, blockIdx.z, red);
}
// J = 0 on the 32 x 32 blocks that have no stored tile
__global__ void k_j_clear(const int* __restrict__ tidx, int nT, int nbf, JOut out, int ldJ) {
    double* __restrict__ J = out.J[blockIdx.z];
    const int I = blockIdx.y, Jt = blockIdx.x;
    if (tidx[min(I, Jt) * nT + max(I, Jt)] >= 0) return;
    for (int e = threadIdx.x; e < TILE2; e += blockDim.x) {
        const int m = I * TILE + e / TILE, n = Jt * TILE + e % TILE;
        if (m < nbf && n < nbf) J[static_cast<size_t>(m) * ldJ + n] = 0.0;
    }
}

// ------------------------------------------------------------------ K path
// Sum of the split partials into the dense result.  A workgroup owns a 16 x 16 output block, the
// splits dealt to 4 groups of 256 threads and added in LDS in a fixed order.  With sym only the
// blocks on and above the diagonal run and write their mirror image too.  Bound by latency at small
// sizes and by HBM at large ones: one thread per output element walking every split, both triangles
// read separately, took 154 us at nbf 96 (464 splits), 301 us at nbf 576 (136 splits of 15 tiles)
// and 360 us in the cross form there; this takes 18, 42 and 59 us.
constexpr int kTrGroups = 4;
__global__ __launch_bounds__(256 * kTrGroups) void k_tile_reduce(const double* __restrict__ P, int nsplit, int ntile,
                                                                const int* __restrict__ tile_of, int nB, int sym, int M,
                                                                int N, double* __restrict__ out, int ldo, double alpha,
                                                                int accumulate) {
    const int bj = blockIdx.x, bi = blockIdx.y;
    if (sym && bi > bj) return;
    __shared__ double s1[kTrGroups][256], s2[kTrGroups][16][17];
    const int el = threadIdx.x & 255, grp = threadIdx.x >> 8;
    const int r = el >> 4, c = el & 15;
    const int t1 = tile_of[(bi >> 3) * nB + (bj >> 3)];
    const size_t o1 = static_cast<size_t>((bi & 7) * 16 + r) * 128 + (bj & 7) * 16 + c;
    double a = 0.0, b = 0.0;
    if (t1 >= 0) {
        const double* p = P + static_cast<size_t>(t1) * 16384 + o1;
#pragma unroll 8
        for (int sp = grp; sp < nsplit; sp += kTrGroups) a += p[static_cast<size_t>(sp) * ntile * 16384];
    }
    s1[grp][el] = a;
    if (sym == 2) {
        // the mirror block of the cross form, M^T
        const int t2 = tile_of[(bj >> 3) * nB + (bi >> 3)];
        const size_t o2 = static_cast<size_t>((bj & 7) * 16 + r) * 128 + (bi & 7) * 16 + c;
        if (t2 >= 0) {
            const double* p = P + static_cast<size_t>(t2) * 16384 + o2;
#pragma unroll 8
            for (int sp = grp; sp < nsplit; sp += kTrGroups) b += p[static_cast<size_t>(sp) * ntile * 16384];
        }
        s2[grp][r][c] = b;
    }
    __syncthreads();
    if (grp != 0) return;
    double v = s1[0][el];
#pragma unroll
    for (int g = 1; g < kTrGroups; ++g) v += s1[g][el];
    if (sym == 2) {
        double w = s2[0][c][r];
#pragma unroll
        for (int g = 1; g < kTrGroups; ++g) w += s2[g][c][r];
        v += w;
    }
    const int m = bi * 16 + r, n = bj * 16 + c;
    if (m >= M || n >= N || (sym && m > n)) return;
    double* o = out + static_cast<size_t>(m) * ldo + n;
    *o = alpha * v + (accumulate ? *o : 0.0);
    if (sym && m != n) {
        double* ot = out + static_cast<size_t>(n) * ldo + m;
        *ot = alpha * v + (accumulate ? *ot : 0.0);
    }
}

// Row-major C = alpha*A*B + beta*C, 128x128 output tiles, FP64 MFMA, 4 waves of 64x64.
// grid = (ceil(N/128), ceil(M/128), batch); operand z is offset by z * stride (0 = shared).
// lower_a: A is lower triangular (A[m][k] = 0 for k > m), so row block m0 stops at k = m0 + 128.
// lower_c: only the 128 x 128 blocks on and below the diagonal of C are formed.
// K-step 16, double-buffered LDS: the next step's operands are loaded into registers before
// the current step's MFMAs and stored to the other buffer after them, one barrier per step.
// Out-of-range elements load as zero.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_gemm_nn_f64(
    const double* __restrict__ A, int lda, const double* __restrict__ Bm, int ldb, double* __restrict__ Cm, int ldc,
    int M, int N, int K, double alpha, double beta, size_t sA, size_t sB, size_t sC, int lower_a, int lower_c) {
    constexpr int KS = 16;
    if (lower_c && blockIdx.x > blockIdx.y) return;
    __shared__ double As[2][128][17];
    __shared__ double Bs[2][16][132];
    A += blockIdx.z * sA;
    Bm += blockIdx.z * sB;
    Cm += blockIdx.z * sC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int m0 = blockIdx.y * 128, n0 = blockIdx.x * 128;
    const int kend = lower_a ? min(K, m0 + 128) : K;
    const int nsteps = (kend + KS - 1) / KS;
    d4_t acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = d4_t{0.0, 0.0, 0.0, 0.0};
    // thread slots: A element (r, kk) = (e >> 4, e & 15), B element (kb, cc) = (e >> 7, e & 127)
    double ra[8], rb[8];
    auto gload = [&](int st) {
        const int k0 = st * KS;
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int e = tid + 256 * it;
            const int r = e >> 4, kk = e & 15;
            ra[it] = (m0 + r < M && k0 + kk < K) ? A[static_cast<size_t>(m0 + r) * lda + k0 + kk] : 0.0;
            const int kb = e >> 7, cc = e & 127;
            rb[it] = (k0 + kb < K && n0 + cc < N) ? Bm[static_cast<size_t>(k0 + kb) * ldb + n0 + cc] : 0.0;
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int e = tid + 256 * it;
            As[buf][e >> 4][e & 15] = ra[it];
            Bs[buf][e >> 7][e & 127] = rb[it];
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < KS; ks += 4) {
            double a[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[buf][wr * 64 + i * 16 + (lane & 15)][ks + (lane >> 4)];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[j] = Bs[buf][ks + (lane >> 4)][wc * 64 + j * 16 + (lane & 15)];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i * 4 + j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], bv[j], acc[i * 4 + j], 0, 0, 0);
        }
    };
    if (nsteps > 0) {
        gload(0);
        lstore(0);
        __syncthreads();
        int buf = 0;
        for (int st = 0; st < nsteps; ++st) {
            const bool more = st + 1 < nsteps;
            if (more) gload(st + 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(buf);
            if (more) lstore(buf ^ 1);
            __syncthreads();
            buf ^= 1;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wr * 64 + i * 16 + 4 * r + (lane >> 4);
                const int col = n0 + wc * 64 + j * 16 + (lane & 15);
                if (row < M && col < N) {
                    double* o = Cm + static_cast<size_t>(row) * ldc + col;
                    *o = alpha * acc[i * 4 + j][r] + (beta != 0.0 ? beta * *o : 0.0);
                }
            }
}

// ------------------------------------------------------------------ synthetic B
__device__ inline void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c[0];
        const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c[2];
        const uint32_t hi0 = static_cast<uint32_t>(p0 >> 32), lo0 = static_cast<uint32_t>(p0);
        const uint32_t hi1 = static_cast<uint32_t>(p1 >> 32), lo1 = static_cast<uint32_t>(p1);
        const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ inline double synth_normal(uint32_t m, uint32_t n, uint32_t Q, uint32_t k0, uint32_t k1) {
    uint32_t c[4] = {m, n, Q, 0u};
    philox4x32_10(c, k0, k1);
    const uint64_t i1 = (static_cast<uint64_t>(c[0]) << 21) | (c[1] >> 11);
    const uint64_t i2 = (static_cast<uint64_t>(c[2]) << 21) | (c[3] >> 11);
    const double u1 = static_cast<double>(i1 + 1) * 0x1.0p-53;
    const double u2 = static_cast<double>(i2) * 0x1.0p-53;
    return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

// grid = (ntp, q1-q0), 256 threads.
__global__ void k_synth_b(const int2* __restrict__ tiles, int ntp, int nbf, const double* __restrict__ decay,
                          uint32_t k0, uint32_t k1, int q0, double* __restrict__ B) {
    const int t = blockIdx.x, Q = q0 + blockIdx.y;
    const int2 IJ = tiles[t];
    const double sQ = 1.0 / sqrt(static_cast<double>(Q) + 1.0);
    double* Bt = B + (static_cast<size_t>(Q) * ntp + t) * TILE2;
    for (int e = threadIdx.x; e < TILE2; e += blockDim.x) {
        const int m = IJ.x * TILE + e / TILE, n = IJ.y * TILE + e % TILE;
        double v = 0.0;
        if (m < nbf && n < nbf) {
            const double g = 0.5 * (synth_normal(m, n, Q, k0, k1) + synth_normal(n, m, Q, k0, k1));
            v = sQ * decay[m > n ? m - n : n - m] * g;
        }
        Bt[e] = v;
    }
}

}  // namespace

// ------------------------------------------------------------------ launchers
void launch_pack_w(const TileGeom& g, const double* D, int ldD, double* W, hipStream_t s) {
    require(g.ntp > 0 && ldD >= g.nbf, "pack_w");
    hipLaunchKernelGGL(k_pack_w, dim3(g.ntp), dim3(256), 0, s, D, ldD, g.nbf, g.d_tiles, W);
}

template <class F>
void with_bsrc(const JSource& b, F&& f) {
    if (b.kind == JSource::F64)
        f(BSrcF64{static_cast<const double*>(b.a)});
    else
        f(BSrcF32{static_cast<const float*>(b.a)});
}

void launch_j1(const TileGeom& g, const JSource& B, const double* W, int naux, int q0, int q1, double* dpart,
               hipStream_t s) {
    require(q0 >= 0 && q1 <= naux && q0 < q1, "j1 q range");
    require(B.a != nullptr, "j1 source");
    const int qblk = 64;
    dim3 grid(g.ntp, (q1 - q0 + qblk - 1) / qblk);
    with_bsrc(B, [&](auto src) {
        hipLaunchKernelGGL(k_j1<decltype(src)>, grid, dim3(256), 0, s, src, W, g.ntp, naux, q0, q1, qblk, dpart);
    });
}

void launch_j1_reduce(const TileGeom& g, const double* dpart, int naux, double* d, hipStream_t s) {
    hipLaunchKernelGGL(k_j1_reduce, grid1(naux, 64), dim3(64 * kJ1Groups), 0, s, dpart, g.ntp, naux, d);
}

void launch_j2(const TileGeom& g, const JSource& B, const double* d, int ldd, int np, int naux, int qchunk,
               double* Jpart, size_t pstride, hipStream_t s) {
    require(qchunk > 0, "j2 qchunk");
    require(B.a != nullptr && np >= 1 && np <= 4 && (np == 1 || ldd >= naux), "j2 source");
    dim3 grid(g.ntp, (naux + qchunk - 1) / qchunk);
    require(np == 1 || pstride >= static_cast<size_t>(grid.y) * g.q_stride(), "j2 partials");
    with_bsrc(B, [&](auto src) {
#define P4A_J2(N)                                                                                                    \
    case N:                                                                                                          \
        hipLaunchKernelGGL((k_j2<decltype(src), N>), grid, dim3(256), 0, s, src, d, ldd, g.ntp, naux, qchunk, Jpart, \
                           pstride);                                                                                 \
        break;
        switch (np) { P4A_J2(1) P4A_J2(2) P4A_J2(3) P4A_J2(4) }
#undef P4A_J2
    });
}

JUnpack prepare_j_unpack(const TileGeom& g, const double* Jpart, size_t pstride, int nchunk, const JOut& out, int np,
                         int ldJ, double alpha, int accumulate, hipStream_t s) {
    require(ldJ >= g.nbf && g.ntp > 0 && nchunk > 0 && np >= 1 && np <= 4, "j_unpack");
    if (!accumulate && g.ntp < g.nT * (g.nT + 1) / 2)
        hipLaunchKernelGGL(k_j_clear, dim3(g.nT, g.nT, np), dim3(256), 0, s, g.d_tidx, g.nT, g.nbf, out, ldJ);
    return JUnpack{Jpart, pstride, nchunk, g.ntp, np, g.d_tiles, g.nbf, out, ldJ, alpha, accumulate};
}
void launch_j_unpack(const TileGeom& g, const double* Jpart, size_t pstride, int nchunk, const JOut& out, int np, int ldJ,
                     double alpha, int accumulate, hipStream_t s) {
    const JUnpack u = prepare_j_unpack(g, Jpart, pstride, nchunk, out, np, ldJ, alpha, accumulate, s);
    hipLaunchKernelGGL(k_j_unpack, dim3(g.ntp, TILE2 / 128, np), dim3(128 * kJuGroups), 0, s, u);
}

void launch_tile_reduce(const double* P, int nsplit, int ntile, const int* d_tile_of, int nB, int sym, int M, int N,
                        double* out, int ldo, double alpha, int accumulate, hipStream_t s) {
    require(M <= nB * 128 && N <= nB * 128 && ldo >= N, "tile_reduce");
    dim3 grid((N + 15) / 16, (M + 15) / 16);
    hipLaunchKernelGGL(k_tile_reduce, grid, dim3(256 * kTrGroups), 0, s, P, nsplit, ntile, d_tile_of, nB, sym, M, N, out, ldo,
                       alpha, accumulate);
}

void launch_gemm_nn_f64(const double* A, int lda, const double* B, int ldb, double* C, int ldc, int M, int N, int K,
                        double alpha, double beta, hipStream_t s, int batch, size_t sA, size_t sB, size_t sC,
                        int lower_a, int lower_c) {
    require(lda >= K && ldb >= N && ldc >= N && batch >= 1 && batch <= 65535, "gemm_nn_f64");
    if (M <= 0 || N <= 0) return;
    dim3 grid((N + 127) / 128, (M + 127) / 128, batch);
    hipLaunchKernelGGL(k_gemm_nn_f64, grid, dim3(256), 0, s, A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, sA, sB, sC,
                       lower_a, lower_c);
}

// ---- adjoint helpers ----
__global__ void k_axpby_mat(const double* __restrict__ X, double a, const double* Y, double b, double* Z, size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        Z[i] = a * X[i] + b * Y[i];
}
// A = (A + A^T) / 2 in place (Matrix::hermitivitize, matrix.cc:2681-2700): the thread of
// (r, c), c > r, owns the pair
__global__ void k_hermitivitize(double* __restrict__ A, int n, int lda) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (c > r && c < n) {
        const size_t rc = static_cast<size_t>(r) * lda + c, cr = static_cast<size_t>(c) * lda + r;
        const double v = 0.5 * (A[rc] + A[cr]);
        A[rc] = v;
        A[cr] = v;
    }
}
__global__ void k_transpose(const double* __restrict__ A, int rows, int cols, int lda, double* __restrict__ AT,
                            int ldt) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (c < cols) AT[static_cast<size_t>(c) * ldt + r] = A[static_cast<size_t>(r) * lda + c];
}
// p[0..n) = 0 (a kernel, not hipMemsetAsync: a caller may capture this work in a graph)
__global__ void k_zero(double* __restrict__ p, size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        p[i] = 0.0;
}
void launch_zero(double* p, size_t n, hipStream_t s) {
    if (n == 0) return;
    const size_t nb = std::min<size_t>((n + 255) / 256, size_t(1) << 16);
    hipLaunchKernelGGL(k_zero, dim3(static_cast<unsigned>(nb)), dim3(256), 0, s, p, n);
}

// out[r][c] = f[r] * A[r][c]
__global__ void k_scale_rows(const double* __restrict__ A, int rows, int cols, const double* __restrict__ f,
                             double* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (c < cols) out[static_cast<size_t>(r) * cols + c] = f[r] * A[static_cast<size_t>(r) * cols + c];
}
void launch_scale_rows(const double* A, int rows, int cols, const double* f, double* out, hipStream_t s) {
    require(rows >= 1 && rows <= 65535 && cols >= 1, "scale_rows");
    hipLaunchKernelGGL(k_scale_rows, dim3((cols + 255) / 256, rows), dim3(256), 0, s, A, rows, cols, f, out);
}
void launch_axpby_mat(const double* X, double a, const double* Y, double b, double* Z, size_t n, hipStream_t s) {
    const size_t nb = std::min<size_t>((n + 255) / 256, size_t(1) << 20);
    if (nb == 0) return;
    hipLaunchKernelGGL(k_axpby_mat, dim3(static_cast<unsigned>(nb)), dim3(256), 0, s, X, a, Y, b, Z, n);
}
void launch_hermitivitize(double* A, int n, int lda, hipStream_t s) {
    require(n >= 1 && n <= 65535 && lda >= n, "hermitivitize");
    hipLaunchKernelGGL(k_hermitivitize, dim3((n + 255) / 256, n), dim3(256), 0, s, A, n, lda);
}
void launch_transpose(const double* A, int rows, int cols, int lda, double* AT, int ldt, hipStream_t s) {
    require(lda >= cols && ldt >= rows, "transpose");
    hipLaunchKernelGGL(k_transpose, dim3((cols + 255) / 256, rows), dim3(256), 0, s, A, rows, cols, lda, AT, ldt);
}
// Dense [nq][nbf][nbf] -> stored tiles of Q = q0 .. q0+nq-1; pairs outside the Schwarz mask are zero.
__global__ __launch_bounds__(256) void k_pack_dense(const double* __restrict__ src, const int2* __restrict__ tiles,
                                                    int ntp, int nbf, const uint8_t* __restrict__ mask, int q0,
                                                    double* __restrict__ B) {
    const int t = blockIdx.x, q = blockIdx.y;
    const int2 IJ = tiles[t];
    const double* S = src + static_cast<size_t>(q) * nbf * nbf;
    double* o = B + (static_cast<size_t>(q0 + q) * ntp + t) * TILE2;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = threadIdx.x + 256 * k;
        const int r = e >> 5, c = e & 31;
        const int m = IJ.x * TILE + r, n = IJ.y * TILE + c;
        double v = 0.0;
        if (m < nbf && n < nbf) {
            const size_t mn = static_cast<size_t>(m) * nbf + n;
            if (mask[mn]) v = S[mn];
        }
        o[e] = v;
    }
}

void launch_pack_dense(const TileGeom& g, const double* src, const uint8_t* mask, int q0, int nq, double* B,
                       hipStream_t s) {
    require(q0 >= 0 && nq >= 1 && nq <= 65535, "pack_dense");
    hipLaunchKernelGGL(k_pack_dense, dim3(g.ntp, nq), dim3(256), 0, s, src, g.d_tiles, g.ntp, g.nbf, mask, q0, B);
}

void launch_synth_b(const TileGeom& g, const double* decay, uint64_t seed, int q0, int q1, double* B, hipStream_t s) {
    require(q0 >= 0 && q1 > q0, "synth_b");
    dim3 grid(g.ntp, q1 - q0);
    hipLaunchKernelGGL(k_synth_b, grid, dim3(256), 0, s, g.d_tiles, g.ntp, g.nbf, decay,
                       static_cast<uint32_t>(seed & 0xffffffffu), static_cast<uint32_t>(seed >> 32), q0, B);
}

}  // namespace p4a
