// FP32 K path for gfx950: X_Q = B_Q C and K = sum_Q X_Q X'_Q^T with FP32 MFMA (16x16x4, 32 cycles for
// 2 x 256 bytes of operands, the FP64 ratio) by the scheme of kernels_f64.hip: independent waves
// whose operands go straight into the MFMA registers one step ahead.  A step is 16 rows of the sum:
// a lane holds 4 consecutive FP32 values per operand.
//
// MFMA lane layout (checked on the device), f32 16x16x4: A[i][k] in lane i + 16 k, B[k][j] in lane
// j + 16 k, D[i][j] in lane j + 16 (i / 4), register i % 4.  (B_Q C)^T = C^T B_Q leaves row m of X and
// columns 4 (lane / 16) + r in a lane, which is an operand of the contraction over columns as it is.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernels_f32.hpp"
#include "wave_kernels.hpp"

namespace p4a {

namespace {

typedef float v4_t __attribute__((ext_vector_type(4)));
__device__ inline v4_t ld4f(const float* base, unsigned off) {
    return *reinterpret_cast<const v4_t*>(reinterpret_cast<const char*>(base) + off);
}
__device__ inline float ld1f(const float* base, unsigned off) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off);
}

// [16 rows][column block][lane][4]: row 16 kb + 4 (lane / 16) + e, column lane % 16
__global__ __launch_bounds__(256) void k_pack_frag32(ColGroups cg, int nbf, int nbfp, float* __restrict__ CA) {
    const ColGroup G = cg.g[blockIdx.y];
    const int n = nbfp * 16 * G.ncb;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < n; idx += gridDim.x * 256) {
        const int e = idx & 3, lane = (idx >> 2) & 63, rest = idx >> 8;
        const int kb = rest / G.ncb, cb = rest % G.ncb;
        const int m = 16 * kb + 4 * (lane >> 4) + e, c = 16 * cb + (lane & 15);
        const int sc = G.cmap ? G.cmap[c] : (c < G.ncol ? c : -1);
        CA[((static_cast<size_t>(kb) * cg.ncb + G.cb0 + cb) * 64 + lane) * 4 + e] =
            (m < nbf && sc >= 0) ? static_cast<float>(G.src[static_cast<size_t>(m) * G.ld + sc]) : 0.0f;
    }
}

// One wave: RT row tiles (32 rows each) x NC column blocks of X_q^T = C^T B_q.
template <int RT, int NC>
__device__ __forceinline__ void ht32_body(const float* __restrict__ BQ, const int* __restrict__ tidx, int nT, int I0,
                                          const float* __restrict__ CA, int ncb, int cb0, float* __restrict__ Xq,
                                          const float* __restrict__ zt) {
    constexpr int NF = 2 * RT;  // 16-row fragments
    const int lane = threadIdx.x & 63, lm = lane & 15, lg = lane >> 4;
    f4_t acc[NF][NC];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[f][c] = f4_t{0, 0, 0, 0};
    v4_t a0[NF], a1[NF], c0[NC], c1[NC];
    // lane offsets (bytes): row lm, columns 4 lg.. of a tile used as it is stored; row 4 lg, column lm
    // of one used transposed
    const unsigned off_n = (lm * TILE + 4 * lg) * 4, off_t = (4 * lg * TILE + lm) * 4, off_c = lane * 16;
    const float* tp[RT];
    TileRow<RT> row(tidx, nT, I0);
    auto seek = [&](const float** t) {
        int o[RT];
        const int j = row.next(o);
        if (j < nT) {
#pragma unroll
            for (int s = 0; s < RT; ++s) t[s] = o[s] >= 0 ? BQ + static_cast<size_t>(o[s]) * TILE2 : zt;
        }
        return j;
    };
    // Step s (16 rows of the sum) of column tile J; orientations as in the FP64 kernel
    auto load = [&](auto tr, int J, const float* const* t, int s, v4_t* a, v4_t* c) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if constexpr (decltype(tr)::value) {
                const float* b = t[f >> 1] + 16 * s * TILE + 16 * (f & 1);
#pragma unroll
                for (int e = 0; e < 4; ++e) a[f][e] = ld1f(b + e * TILE, off_t);
            } else {
                a[f] = ld4f(t[f >> 1] + 16 * (f & 1) * TILE + 16 * s, off_n);
            }
        }
        const float* cp = CA + (static_cast<size_t>(2 * J + s) * ncb + cb0) * 256;
#pragma unroll
        for (int i = 0; i < NC; ++i) c[i] = ld4f(cp + 256 * i, off_c);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const v4_t* a, const v4_t* c) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    acc[f][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[i][e], a[f][e], acc[f][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    const float* tn[RT];
    int J = seek(tp), Jn;
    // tile J, its step 0 already loaded, and step 0 of tile Jn (past the last tile: of J again)
    auto tile = [&](auto tr, auto trn) {
        load(tr, J, tp, 1, a1, c1);
        mul(a0, c0);
        const bool last = Jn >= nT;
        const float* tl[RT];
#pragma unroll
        for (int s = 0; s < RT; ++s) tl[s] = last ? tp[s] : tn[s];
        load(trn, last ? J : Jn, tl, 0, a0, c0);
        mul(a1, c1);
        J = Jn;
#pragma unroll
        for (int s = 0; s < RT; ++s) tp[s] = tl[s];
    };
    using Tr = std::true_type;
    using As = std::false_type;
    if (J <= I0) {
        load(Tr{}, J, tp, 0, a0, c0);
        Jn = seek(tn);
        while (Jn <= I0) {
            tile(Tr{}, Tr{});
            Jn = seek(tn);
        }
        tile(Tr{}, As{});
    } else if (J < nT) {
        load(As{}, J, tp, 0, a0, c0);
    }
    while (J < nT) {
        Jn = seek(tn);
        tile(As{}, As{});
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < NC; ++i)
            *reinterpret_cast<f4_t*>(reinterpret_cast<char*>(
                                         Xq + (static_cast<size_t>(2 * I0 + f) * ncb + cb0 + i) * 256) + off_c) = acc[f][i];
}

// Bound by FP32 MFMA issue at the clock the power limit leaves (79 % of the cycles busy at 2.05 GHz).
// Naux 1856 / nbf 384 / 160 columns: 0.81 ms, 108 TFLOP/s; the LDS-tiled kernel before it, whose
// columns were padded to 64, took 1.34 ms.  One wave per SIMD (launch_ht_f32): two waves of this
// kernel on a SIMD get in each other's way - 108 us each where one alone takes 35, at 5 column blocks, with all
// operands in cache too - and workgroups are dispatched in order over the shader engines, so the
// engine that is full holds the others back (1.25 ms).  With the registers of the whole SIMD a wave
// takes up to 10 column blocks (0.81 ms; 5: 0.83), which halves the reads of B.
template <int RT, int NC>
__global__ __launch_bounds__(256, NC <= 5 ? 2 : 1) void k_ht_f32(const float* __restrict__ B, const int* __restrict__ tidx, int nT,
                                                   int ntp, int nq, const float* __restrict__ CA, int ncb, int ncg,
                                                   float* __restrict__ X, const float* __restrict__ zt) {
    const int nrg = (nT + RT - 1) / RT;
    const WaveItem w = wave_item(nrg * ncg);
    if (w.group >= nq) return;
    const int q = w.group, rg = w.item / ncg, cg = w.item % ncg;
    // the first nwide column groups are NC blocks wide, the others NC - 1
    const int nwide = ncb - ncg * (NC - 1);
    const int cb0 = cg * NC - max(0, cg - nwide);
    const bool wide = cg < nwide;
    const int I0 = RT * rg;
    const float* BQ = B + static_cast<size_t>(q) * ntp * TILE2;
    float* Xq = X + static_cast<size_t>(q) * nT * 2 * ncb * 256;
    if (RT == 1 || I0 + RT <= nT) {
        if (wide)
            ht32_body<RT, NC>(BQ, tidx, nT, I0, CA, ncb, cb0, Xq, zt);
        else if constexpr (NC > 1)
            ht32_body<RT, NC - 1>(BQ, tidx, nT, I0, CA, ncb, cb0, Xq, zt);
    } else if constexpr (RT == 2) {
        if (wide)
            ht32_body<1, NC>(BQ, tidx, nT, I0, CA, ncb, cb0, Xq, zt);
        else if constexpr (NC > 1)
            ht32_body<1, NC - 1>(BQ, tidx, nT, I0, CA, ncb, cb0, Xq, zt);
    }
}

// k-terms an FP32 accumulator holds before it is folded into FP64
constexpr int kFold = 512;

// One wave: NI x NJ 16-row fragments of X X'^T over a range of (q, k) steps of 16 columns.  SKIP: the
// block touches the diagonal of a symmetric result, its row fragment i and column fragment j + DJ:
// sub-tiles below it are not formed.  The FP32 accumulators are folded into FP64 totals every 512
// k-terms, so the error of a sum does not grow with the auxiliary functions a split covers; the totals
// are what limits the block to 64 x 32.  Naux 1856 / nbf 384, every block over 80 columns: 0.45 ms, 97 TFLOP/s
// (LDS-tiled 128 x 128 tiles before: 0.51 ms); one wave per SIMD instead of two 0.63, half the splits 0.49.
template <int NI, int NJ, bool SKIP, int DJ>
__device__ __forceinline__ void kc32_body(const float* __restrict__ X, size_t qstride, int nkx, int ra, int rb, int ka,
                                          int kb, int nk, int s0, int s1, double alpha, int accumulate,
                                          double* __restrict__ Pb) {
    const int lane = threadIdx.x & 63;
    const unsigned off = lane * 16;
    f4_t acc[NI][NJ];
    d4_t tot[NI][NJ];
    auto formed = [](int i, int j) { return !SKIP || i <= j + DJ; };
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            acc[i][j] = f4_t{0, 0, 0, 0};
            tot[i][j] = d4_t{0, 0, 0, 0};
        }
    v4_t a0[NI], b0[NJ], a1[NI], b1[NJ];
    int q = s0 / nk, k = s0 % nk, left = s1 - s0;
    auto load = [&](v4_t* a, v4_t* b) {
        const float* pa = X + q * qstride + (static_cast<size_t>(ra) * nkx + ka + k) * 256;
#pragma unroll
        for (int i = 0; i < NI; ++i) a[i] = ld4f(pa + static_cast<size_t>(i) * nkx * 256, off);
        const float* pb = X + q * qstride + (static_cast<size_t>(rb) * nkx + kb + k) * 256;
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = ld4f(pb + static_cast<size_t>(j) * nkx * 256, off);
        if (--left > 0) {
            if (++k == nk) {
                k = 0;
                ++q;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const v4_t* a, const v4_t* b) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    if (formed(i, j))
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                if (formed(i, j)) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[i][j][r] += static_cast<double>(acc[i][j][r]);
                    acc[i][j] = f4_t{0, 0, 0, 0};
                }
    };
    const int n = s1 - s0;
    if (n > 0) {
        load(a0, b0);
        int st = 0;
        while (st + 1 < n) {
            // up to one fold's worth of step pairs
            const int end = min(n - 1, st + kFold / 16);
            for (; st < end; st += 2) {
                load(a1, b1);
                mul(a0, b0);
                load(a0, b0);
                mul(a1, b1);
            }
            fold();
        }
        if (st < n) mul(a0, b0);
        fold();
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (formed(i, j))
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double* o = Pb + (i * 2 + j) * 256 + r * 64 + lane;
                    *o = alpha * tot[i][j][r] + (accumulate ? *o : 0.0);
                }
}

// Block b of the upper set: row block I (64 rows) takes the column blocks (32) J >= 2 I
__device__ inline void upper_block32(int b, int nT, int& I, int& J) {
    I = 0;
    while (b >= nT - 2 * I) {
        b -= nT - 2 * I;
        ++I;
    }
    J = 2 * I + b;
}

template <bool UPPER>
__global__ __launch_bounds__(64, 2) void k_kc_f32(const float* __restrict__ X, size_t qstride, int nkx, int nT, int nq,
                                                  KcSegs segs, int nblk, double* __restrict__ P, int accumulate) {
    const WaveItem w = wave_item(nblk);
    if (w.group >= segs.nsplit) return;
    int is = 0;
    while (w.group >= segs.s[is].sp0 + segs.s[is].nsp) ++is;
    const KcSeg sg = segs.s[is];
    int I, J;
    if (UPPER) {
        upper_block32(w.item, nT, I, J);
    } else {
        I = w.item / nT;
        J = w.item % nT;
    }
    const long long steps = static_cast<long long>(nq) * sg.nk;
    const int sp = w.group - sg.sp0;
    const int s0 = uni(static_cast<int>(steps * sp / sg.nsp)), s1 = uni(static_cast<int>(steps * (sp + 1) / sg.nsp));
    const bool fi = 2 * I + 2 <= nT;  // a last block row holds two fragments when nT is odd
    double* Pb = P + (static_cast<size_t>(w.group) * nblk + w.item) * kc32_partial;
#define P4A_KC32(NI, S, DJ) \
    kc32_body<NI, 2, S, DJ>(X, qstride, nkx, 4 * I, 2 * J, sg.ka, sg.kb, sg.nk, s0, s1, sg.alpha, accumulate, Pb)
    if (UPPER && J == 2 * I)
        P4A_KC32(2, true, 0);  // rows 32.. of the block lie below the diagonal
    else if (UPPER && J == 2 * I + 1)
        P4A_KC32(4, true, 2);
    else if (fi)
        P4A_KC32(4, false, 0);
    else
        P4A_KC32(2, false, 0);
#undef P4A_KC32
}

constexpr int kRed32 = 4;
__global__ __launch_bounds__(256 * kRed32) void k_kc32_reduce(const double* __restrict__ P, int nblk, int nT, int n,
                                                             int upper, KcOuts outs, int accumulate) {
    __shared__ double red[kRed32][256];
    const int blk = blockIdx.x, st = blockIdx.y;
    const KcOut O = outs.o[blockIdx.z];
    int I, J;
    if (upper) {
        upper_block32(blk, nT, I, J);
    } else {
        I = blk / nT;
        J = blk % nT;
    }
    const int m0 = 64 * I + 16 * (st >> 1), n0 = 32 * J + 16 * (st & 1);
    if (m0 >= n || n0 >= n || (upper && m0 > n0)) return;
    const int el = threadIdx.x & 255, grp = threadIdx.x >> 8;
    const double* p = P + static_cast<size_t>(blk) * kc32_partial + st * 256 + el;
    double a = 0.0;
#pragma unroll 8
    for (int sp = grp; sp < O.nsp; sp += kRed32) a += p[static_cast<size_t>(O.sp0 + sp) * nblk * kc32_partial];
    red[grp][el] = a;
    __syncthreads();
    if (grp) return;
    double v = red[0][el];
#pragma unroll
    for (int g = 1; g < kRed32; ++g) v += red[g][el];
    // register r, lane l: row 4 (l / 16) + r, column l % 16
    const int m = m0 + 4 * ((el & 63) >> 4) + (el >> 6), c = n0 + (el & 15);
    if (m >= n || c >= n || (upper && m > c)) return;
    double* o = O.out + static_cast<size_t>(m) * n + c;
    *o = v + (accumulate ? *o : 0.0);
    if (upper && m != c) {
        double* ot = O.out + static_cast<size_t>(c) * n + m;
        *ot = v + (accumulate ? *ot : 0.0);
    }
}

}  // namespace

// ------------------------------------------------------------------ launchers
void launch_pack_frag32(const ColGroups& cg, int nbf, int nbfp, float* CA, hipStream_t s) {
    require(cg.n >= 1 && cg.n <= kMaxGroups && nbfp % TILE == 0 && nbfp >= nbf, "pack_frag32");
    int most = 0;
    for (int i = 0; i < cg.n; ++i) {
        const ColGroup& G = cg.g[i];
        require(G.ncb > 0 && G.cb0 >= 0 && G.cb0 + G.ncb <= cg.ncb && G.src && G.ld >= (G.cmap ? 1 : G.ncol) &&
                    (G.cmap || G.ncol <= 16 * G.ncb),
                "pack_frag32 group");
        most = std::max(most, G.ncb);
    }
    require(static_cast<long long>(nbfp) * 16 * most < (1LL << 31), "pack_frag32 size");
    hipLaunchKernelGGL(k_pack_frag32, dim3(std::min(4096, (nbfp * 16 * most + 255) / 256), cg.n), dim3(256), 0, s, cg, nbf,
                       nbfp, CA);
}

// Column groups of up to 10 blocks, evenly divided
constexpr int kNC = 10;
// LDS a workgroup asks for and does not use: more than half a CU's, so that each SIMD runs one wave
constexpr int kOneWave = 84 << 10;

template <int RT>
static void ht_f32_rt(const TileGeom& g, const float* B, int nq, const float* CA, int ncb, float* X, const float* zt,
                      hipStream_t s) {
    const int ncg = (ncb + kNC - 1) / kNC, nc = (ncb + ncg - 1) / ncg;
    const dim3 grid(wave_grid(nq, ht_row_groups(g.nT, RT) * ncg, 4));
#define P4A_HT32(N)                                                                                                     \
    case N:                                                                                                             \
        hipLaunchKernelGGL((k_ht_f32<RT, N>), grid, dim3(256), kOneWave, s, B, g.d_tidx, g.nT, g.ntp, nq, CA, ncb, ncg, \
                           X, zt);                                                                                      \
        break;
    switch (nc) {
        P4A_HT32(1) P4A_HT32(2) P4A_HT32(3) P4A_HT32(4) P4A_HT32(5)
        P4A_HT32(6) P4A_HT32(7) P4A_HT32(8) P4A_HT32(9) P4A_HT32(10)
    }
#undef P4A_HT32
}
void launch_ht_f32(const TileGeom& g, const float* B, int nq, const float* CA, int ncb, int rt, float* X, const void* zt,
                   hipStream_t s) {
    require(nq > 0 && ncb > 0 && (rt == 1 || rt == 2) && g.nT > 0 && g.nT <= 256 && g.nbfp == g.nT * TILE && zt &&
                static_cast<double>(nq) * ht_row_groups(g.nT, rt) * ((ncb + kNC - 1) / kNC) < 4.0e9,
            "ht_f32 shape");
    if (rt == 1)
        ht_f32_rt<1>(g, B, nq, CA, ncb, X, static_cast<const float*>(zt), s);
    else
        ht_f32_rt<2>(g, B, nq, CA, ncb, X, static_cast<const float*>(zt), s);
}

int kc32_blocks(int nT, bool upper) {
    const int nbr = (nT + 1) / 2;
    return upper ? nbr * nT - nbr * (nbr - 1) : nbr * nT;
}
int kc32_choose_splits(int nT, bool upper, int steps, int nseg, int max_splits) {
    return balanced_splits(static_cast<long long>(kc32_blocks(nT, upper)) * nseg, steps, max_splits);
}

void launch_kc_f32(const float* X, size_t qstride, int nkx, int nT, int nq, const KcSegs& segs, bool upper, double* P,
                   int accumulate, hipStream_t s) {
    require(segs.n >= 1 && segs.n <= kMaxSegs && nq > 0 && nkx > 0 && nT > 0 && segs.nsplit > 0, "kc_f32 shape");
    int at = 0;
    for (int i = 0; i < segs.n; ++i) {
        const KcSeg& g = segs.s[i];
        require(g.sp0 == at && g.nsp > 0 && g.nk > 0 && g.ka >= 0 && g.kb >= 0 && g.ka + g.nk <= nkx &&
                    g.kb + g.nk <= nkx && (!upper || g.ka == g.kb) && static_cast<long long>(nq) * g.nk < (1LL << 31),
                "kc_f32 pass");
        at += g.nsp;
    }
    require(at == segs.nsplit, "kc_f32 splits");
    const int nblk = kc32_blocks(nT, upper);
    const dim3 grid(wave_grid(segs.nsplit, nblk, 1));
    if (upper)
        hipLaunchKernelGGL((k_kc_f32<true>), grid, dim3(64), 0, s, X, qstride, nkx, nT, nq, segs, nblk, P, accumulate);
    else
        hipLaunchKernelGGL((k_kc_f32<false>), grid, dim3(64), 0, s, X, qstride, nkx, nT, nq, segs, nblk, P, accumulate);
}

void launch_kc32_reduce(const double* P, int nT, int n, bool upper, const KcOuts& outs, int accumulate, hipStream_t s) {
    require(outs.n >= 1 && outs.n <= 2 * kMaxPairs && n > 0 && n <= nT * TILE, "kc32_reduce");
    const int nblk = kc32_blocks(nT, upper);
    hipLaunchKernelGGL(k_kc32_reduce, dim3(nblk, 8, outs.n), dim3(256 * kRed32), 0, s, P, nblk, nT, n, upper ? 1 : 0, outs,
                       accumulate);
}

}  // namespace p4a
