// FP64 J/K path for gfx950: X_Q = B_Q C, d_Q = <X_Q, C_right> and K = sum_Q X_Q X'_Q^T.
//
// The FP64 MFMA (16x16x4) takes 64 cycles for 2 x 512 bytes of operands, so a wave that owns a
// 64 x 80 (or 64 x 64) output tile needs 14-16 bytes per clock and CU: the vector caches deliver
// that, and staging through LDS would only add barriers that make the waves of a workgroup wait for
// one another.  Every wave here is independent: it loads its operands straight into the MFMA
// registers one step ahead and never synchronises.
//
// MFMA lane layout (checked on the device), 16x16x4: A[i][k] in lane i + 16 k, B[k][j] in lane
// j + 16 k, D[i][j] in lane j + 16 (i % 4), register i / 4.
//
// Fragment order.  The half-transform computes (B_Q C)^T = C^T B_Q, so a lane ends up with one row m
// of X (m = lane % 16) and the columns 4 r + lane / 16, r = 0..3, of a 16-column block.  That is
// exactly an MFMA operand of the contraction over columns: register r of both operands holds the
// same four columns, and the sum over columns does not care which four.  X is therefore stored as it
// lies in the registers, [q][16 rows][8 columns][lane][2], and the contraction loads 16 contiguous
// bytes per lane, 1 KB per wave.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "j_unpack.hpp"
#include "kernels_f64.hpp"
#include "wave_kernels.hpp"

namespace p4a {

namespace {

// ------------------------------------------------------------------ packing
__global__ __launch_bounds__(256) void k_pack_frag(ColGroups cg, int nbf, int nbfp, double* __restrict__ CA,
                                                   double* __restrict__ CD) {
    const ColGroup G = cg.g[blockIdx.y];
    const int n = nbfp * 16 * G.ncb;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < n; idx += gridDim.x * 256) {
        const int e = idx & 1, lane = (idx >> 1) & 63, rest = idx >> 7;
        if (CA) {
            // [k8 of rows][column block][lane][2]: row 8 kb + 2 (lane / 16) + e, column lane % 16
            const int kb = rest / G.ncb, cb = rest % G.ncb;
            const int m = 8 * kb + 2 * (lane >> 4) + e, c = 16 * cb + (lane & 15);
            const int sc = G.cmap ? G.cmap[c] : (c < G.ncol ? c : -1);
            CA[((static_cast<size_t>(kb) * cg.ncb + G.cb0 + cb) * 64 + lane) * 2 + e] =
                (m < nbf && sc >= 0) ? G.src[static_cast<size_t>(m) * G.ld + sc] : 0.0;
        }
        if (CD) {
            // [16 rows][k8 of columns][lane][2]: row lane % 16, column 8 kb + 4 e + lane / 16
            const int rb = rest / (2 * G.ncb), kb = rest % (2 * G.ncb);
            const int m = 16 * rb + (lane & 15), c = 8 * kb + 4 * e + (lane >> 4);
            const int sc = G.cmap ? G.cmap[c] : (c < G.ncol ? c : -1);
            CD[((static_cast<size_t>(rb) * 2 * cg.ncb + 2 * G.cb0 + kb) * 64 + lane) * 2 + e] =
                (G.partner && m < nbf && sc >= 0) ? G.partner[static_cast<size_t>(m) * G.ld + sc] : 0.0;
        }
    }
}

// ------------------------------------------------------------------ half-transform
// One wave: RT row tiles (32 rows each) x NC column blocks of X_q^T = C^T B_q.
template <int RT, int NC>
__device__ __forceinline__ void ht_body(const double* __restrict__ BQ, const int* __restrict__ tidx, int nT, int I0,
                               const double* __restrict__ CA, int ncb, int cb0, const double* __restrict__ CD,
                               double* __restrict__ Xq, double* __restrict__ dp, const double* __restrict__ zt) {
    constexpr int NF = 2 * RT;  // 16-row fragments
    const int lane = threadIdx.x & 63, lm = lane & 15, lg = lane >> 4;
    d4_t acc[NF][NC];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[f][c] = d4_t{0.0, 0.0, 0.0, 0.0};

    d2_t a0[NF], a1[NF], c0[NC], c1[NC];
    // lane offsets (bytes) inside a tile: row lm, columns 2 lg.. of a tile used as it is stored, and
    // row 2 lg, column lm of one used transposed
    const unsigned off_n = (lm * TILE + 2 * lg) * 8, off_t = (2 * lg * TILE + lm) * 8, off_c = lane * 16;
    const double* tp[RT];
    TileRow<RT> row(tidx, nT, I0);
    auto seek = [&](const double** t) {  // the next tile's rows (an absent one reads zeros)
        int o[RT];
        const int j = row.next(o);
        if (j < nT) {
#pragma unroll
            for (int s = 0; s < RT; ++s) t[s] = o[s] >= 0 ? BQ + static_cast<size_t>(o[s]) * TILE2 : zt;
        }
        return j;
    };
    // Step s (8 rows of the sum) of column tile J.  For J <= I0 every row tile reads the stored block
    // (J, I) transposed (the diagonal block holds both triangles), for J > I0 the block (I, J), or the
    // diagonal one, as it is stored.
    auto load = [&](auto tr, int J, const double* const* t, int s, d2_t* a, d2_t* c) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if constexpr (decltype(tr)::value) {
                const double* b = t[f >> 1] + 8 * s * TILE + 16 * (f & 1);
                a[f].x = ld1(b, off_t);
                a[f].y = ld1(b + TILE, off_t);
            } else {
                a[f] = ld2(t[f >> 1] + 16 * (f & 1) * TILE + 8 * s, off_n);
            }
        }
        const double* cp = CA + (static_cast<size_t>(4 * J + s) * ncb + cb0) * 128;
#pragma unroll
        for (int i = 0; i < NC; ++i) c[i] = ld2(cp + 128 * i, off_c);
    };
    auto mul = [&](const d2_t* a, const d2_t* c) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    acc[f][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(c[i][e], a[f][e], acc[f][i], 0, 0, 0);
    };
    // load the next step's operands while this one's are multiplied
    auto step = [&](auto tr, int J, const double* const* t, int s, d2_t* an, d2_t* cn, const d2_t* a, const d2_t* c) {
        load(tr, J, t, s, an, cn);
        mul(a, c);
        interleave<(decltype(tr)::value ? 2 : 1) * NF + NC, 2 * NF * NC>();
    };
    // Tile J, its step 0 already loaded, and step 0 of tile Jn (past the last tile: of J again, never
    // used), so that every path through the loops issues the same loads and a wait for one step's
    // operands leaves the next step's in flight.
    const double* tn[RT];
    int J = seek(tp), Jn;
    auto tile = [&](auto tr, auto trn) {
        step(tr, J, tp, 1, a1, c1, a0, c0);
        step(tr, J, tp, 2, a0, c0, a1, c1);
        step(tr, J, tp, 3, a1, c1, a0, c0);
        const bool last = Jn >= nT;
        const double* tl[RT];
#pragma unroll
        for (int s = 0; s < RT; ++s) tl[s] = last ? tp[s] : tn[s];
        step(trn, last ? J : Jn, tl, 0, a0, c0, a1, c1);
        J = Jn;
#pragma unroll
        for (int s = 0; s < RT; ++s) tp[s] = tl[s];
    };
    using Tr = std::true_type;
    using As = std::false_type;
    if (J <= I0) {
        load(Tr{}, J, tp, 0, a0, c0);
        __builtin_amdgcn_sched_barrier(0);
        Jn = seek(tn);
        while (Jn <= I0) {
            tile(Tr{}, Tr{});
            Jn = seek(tn);
        }
        tile(Tr{}, As{});
    } else if (J < nT) {
        load(As{}, J, tp, 0, a0, c0);
        __builtin_amdgcn_sched_barrier(0);
    }
    while (J < nT) {
        Jn = seek(tn);
        tile(As{}, As{});
    }
    // X in fragment order, and the wave's share of d_q per column block
    const int nkx = 2 * ncb;
    auto at = [&](int f) { return (static_cast<size_t>(2 * I0 + f) * nkx + 2 * cb0) * 128; };
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 2 * NC; ++i)
            *reinterpret_cast<d2_t*>(reinterpret_cast<char*>(Xq + at(f) + 128 * i) + off_c) =
                d2_t{acc[f][i >> 1][2 * (i & 1)], acc[f][i >> 1][2 * (i & 1) + 1]};
    if (CD) {
        double ds[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) ds[i] = 0.0;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int i = 0; i < 2 * NC; ++i) {
                const d2_t w = ld2(CD + at(f) + 128 * i, off_c);
                ds[i >> 1] = fma(acc[f][i >> 1][2 * (i & 1) + 1], w.y,
                                 fma(acc[f][i >> 1][2 * (i & 1)], w.x, ds[i >> 1]));
            }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) ds[i] += __shfl_xor(ds[i], o);
            if (lane == 0) dp[i] = ds[i];
        }
    }
}

// Bound by the FP64 MFMA pipes (90 % busy at 2.3 GHz, where a library product of 8192^3 reaches
// 72.6 TFLOP/s): 2000 Q at nbf 1500 / 300 columns take 39.5 ms (68 TFLOP/s of the 2 nbf^2 ncol
// products) against 50.7 through LDS with 128 x 320 tiles and a barrier per 8 rows of the sum;
// nbf 576 / 120 columns / 2784 Q 3.8 ms against 5.8.  Columns are cut into near-equal groups of at
// most 80, in 16s: 80 columns cost 5 blocks, not two 64s.  Four waves per workgroup: the column groups
// of one row block mostly share a CU's vector cache (one wave per workgroup: 3 % slower).  64 x 128 and
// 64 x 160 with one wave per SIMD were 8 % slower and spilled; waves that draw their items from counters fill
// the slots that uneven waves leave empty (a quarter at nbf 413) and were 3-7 % slower all the same.
template <int RT, int NC>
__global__ __launch_bounds__(256, 2) void k_ht_f64(
    const double* __restrict__ B, const int* __restrict__ tidx, int nT, int ntp, int nq, const double* __restrict__ CA,
    const double* __restrict__ CD, int ncb, int ncg, double* __restrict__ X, double* __restrict__ dpart,
    const double* __restrict__ zt) {
    const int nrg = (nT + RT - 1) / RT;
    const WaveItem w = wave_item(nrg * ncg);
    if (w.group >= nq) return;
    const int q = w.group, rg = w.item / ncg, cg = w.item % ncg;
    // the first nwide column groups are NC blocks wide, the others NC - 1
    const int nwide = ncb - ncg * (NC - 1);
    const int cb0 = cg * NC - max(0, cg - nwide);
    const bool wide = cg < nwide;
    const int I0 = RT * rg;
    const double* BQ = B + static_cast<size_t>(q) * ntp * TILE2;
    double* Xq = X + static_cast<size_t>(q) * nT * 4 * ncb * 128;
    double* dp = dpart ? dpart + (static_cast<size_t>(q) * nrg + rg) * ncb + cb0 : nullptr;
    if (RT == 1 || I0 + RT <= nT) {
        if (wide)
            ht_body<RT, NC>(BQ, tidx, nT, I0, CA, ncb, cb0, CD, Xq, dp, zt);
        else if constexpr (NC > 1)
            ht_body<RT, NC - 1>(BQ, tidx, nT, I0, CA, ncb, cb0, CD, Xq, dp, zt);
    } else if constexpr (RT == 2) {
        if (wide)
            ht_body<1, NC>(BQ, tidx, nT, I0, CA, ncb, cb0, CD, Xq, dp, zt);
        else if constexpr (NC > 1)
            ht_body<1, NC - 1>(BQ, tidx, nT, I0, CA, ncb, cb0, CD, Xq, dp, zt);
    }
}

// d[p][q]: one wave per (q, pair), the partials in a fixed order
__global__ __launch_bounds__(256) void k_dpart_reduce(const double* __restrict__ dpart, int nq, int nrg, int ncb,
                                                      DRanges r, double* __restrict__ d, int ldd) {
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, p = blockIdx.y;
    if (q >= nq) return;
    const int nc = r.ncb[p], n = nrg * nc;
    const double* src = dpart + static_cast<size_t>(q) * nrg * ncb + r.cb0[p];
    double s = 0.0;
    for (int i = lane; i < n; i += 64) s += src[(i / nc) * ncb + i % nc];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) d[static_cast<size_t>(p) * ldd + q] = s;
}

// ------------------------------------------------------------------ contraction
// One wave: a block of NI x NJ 16-row fragments of X X'^T over a range of (q, k) steps.  DIAG: the
// two row ranges are the same and so are the column ranges (a symmetric result): the operands are
// loaded once and only the sub-tiles on and above the diagonal are formed.
template <int NI, int NJ, bool DIAG>
__device__ __forceinline__ void kc_body(const double* __restrict__ XA, const double* __restrict__ XB, size_t qstride, int nkx,
                               int ra, int rb, int ka, int kb, int nk, int s0, int s1, double alpha, int accumulate,
                               double* __restrict__ Pb) {
    const int lane = threadIdx.x & 63;
    const unsigned off = lane * 16;
    d4_t acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
    d2_t a0[NI], b0[NJ], a1[NI], b1[NJ];
    // the step being loaded; loads past the end read the last step again
    int q = s0 / nk, k = s0 % nk, left = s1 - s0;
    auto load = [&](d2_t* a, d2_t* b) {
        const double* pa = XA + q * qstride + (static_cast<size_t>(ra) * nkx + ka + k) * 128;
#pragma unroll
        for (int i = 0; i < NI; ++i) a[i] = ld2(pa + static_cast<size_t>(i) * nkx * 128, off);
        if constexpr (!DIAG) {
            const double* pb = XB + q * qstride + (static_cast<size_t>(rb) * nkx + kb + k) * 128;
#pragma unroll
            for (int j = 0; j < NJ; ++j) b[j] = ld2(pb + static_cast<size_t>(j) * nkx * 128, off);
        }
        if (--left > 0) {
            if (++k == nk) {
                k = 0;
                ++q;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const d2_t* a, const d2_t* b) {
        const d2_t* bb = DIAG ? a : b;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    if (!DIAG || i <= j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], bb[j][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int n = s1 - s0;
    if (n > 0) {
        load(a0, b0);
        int st = 0;
        for (; st + 1 < n; st += 2) {
            load(a1, b1);
            mul(a0, b0);
            load(a0, b0);
            mul(a1, b1);
        }
        if (st < n) mul(a0, b0);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (!DIAG || i <= j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double* o = Pb + (i * 4 + j) * 256 + r * 64 + lane;
                    *o = alpha * acc[i][j][r] + (accumulate ? *o : 0.0);
                }
}

// Bound by the MFMA pipes and, under them, the power limit: at nbf 1500 the wave reads 4 bytes of X
// per 256 flops, and X (10 GB per Q-block) streams through the L2s, which serve all output blocks of
// a split as long as the waves of the split stay within a few Q of one another.  Nothing holds them
// together, so the splits are short (kc_choose_splits): 3000 Q at nbf 1500 / 300 columns took 36.5 ms
// in 96 splits of 1190 steps (192 GB fetched, 1.5e9 L2 misses, 2.07 GHz) and take 32.1 ms in 384 of
// 297; 2 x 2 blocks per workgroup held together by a barrier per step (0.87e9 misses) took 35.9.
// One wave per workgroup: a wave's slot is refilled when it ends, not when its three neighbours do
// (2.58 against 2.88 ms at nbf 576).  Before, through LDS with 128 x 128 tiles: 34.1 ms there.
template <bool UPPER>
__global__ __launch_bounds__(64, 2) void k_kc_f64(
    const double* __restrict__ XA, const double* __restrict__ XB, size_t qstride, int nkx, int nT, int nq, KcSegs segs,
    int nbr, int nblk, double* __restrict__ P, int accumulate) {
    const WaveItem w = wave_item(nblk);
    if (w.group >= segs.nsplit) return;
    int is = 0;
    while (w.group >= segs.s[is].sp0 + segs.s[is].nsp) ++is;
    const KcSeg sg = segs.s[is];
    int I, J;
    if (UPPER) {
        // upper blocks row by row
        I = 0;
        int r = w.item;
        while (r >= nbr - I) {
            r -= nbr - I;
            ++I;
        }
        J = I + r;
    } else {
        I = w.item / nbr;
        J = w.item % nbr;
    }
    const long long steps = static_cast<long long>(nq) * sg.nk;
    const int sp = w.group - sg.sp0;
    const int s0 = uni(static_cast<int>(steps * sp / sg.nsp)), s1 = uni(static_cast<int>(steps * (sp + 1) / sg.nsp));
    const int ra = 4 * I, rb = 4 * J;
    const bool fi = ra + 4 <= 2 * nT, fj = rb + 4 <= 2 * nT;  // a last block row holds two fragments when nT is odd
    double* Pb = P + (static_cast<size_t>(w.group) * nblk + w.item) * 4096;
#define P4A_KC(NI, NJ, D) \
    kc_body<NI, NJ, D>(XA, XB, qstride, nkx, ra, rb, sg.ka, sg.kb, sg.nk, s0, s1, sg.alpha, accumulate, Pb)
    if constexpr (UPPER) {
        if (I == J) {
            if (fi)
                P4A_KC(4, 4, true);
            else
                P4A_KC(2, 2, true);
        } else if (fj) {
            P4A_KC(4, 4, false);
        } else {
            P4A_KC(4, 2, false);
        }
    } else {
        if (fi && fj)
            P4A_KC(4, 4, false);
        else if (fi)
            P4A_KC(4, 2, false);
        else if (fj)
            P4A_KC(2, 4, false);
        else
            P4A_KC(2, 2, false);
    }
#undef P4A_KC
}

// Sum over a pair's splits of one 16 x 16 sub-tile, the splits dealt to 4 groups of 256 threads and
// added in LDS in a fixed order.  J's reduction rides in the same launch (z past the outputs): bound by
// latency both, the two in a row cost 8 us at nbf 24.
constexpr int kRedGroups = 4;
__global__ __launch_bounds__(256 * kRedGroups) void k_kc_reduce(const double* __restrict__ P, int nblk, int nbr, int n,
                                                               int upper, KcOuts outs, int accumulate, JUnpack ju) {
    __shared__ double red[kRedGroups][256];
    const int blk = blockIdx.x, st = blockIdx.y;
    if (static_cast<int>(blockIdx.z) >= outs.n) {
        const int i = ((blockIdx.z - outs.n) * 16 + st) * nblk + blk, per = ju.ntp * (TILE2 / 128);
        if (i < per * ju.np) j_unpack_block(ju, i % per % ju.ntp, i % per / ju.ntp, i / per, &red[0][0]);
        return;
    }
    const KcOut O = outs.o[blockIdx.z];
    int I = 0, J = 0;
    if (upper) {
        int r = blk;
        while (r >= nbr - I) {
            r -= nbr - I;
            ++I;
        }
        J = I + r;
    } else {
        I = blk / nbr;
        J = blk % nbr;
    }
    const int m0 = 64 * I + 16 * (st >> 2), n0 = 64 * J + 16 * (st & 3);
    if (m0 >= n || n0 >= n || (upper && m0 > n0)) return;
    const int el = threadIdx.x & 255, grp = threadIdx.x >> 8;
    const double* p = P + static_cast<size_t>(blk) * 4096 + st * 256 + el;
    double a = 0.0;
#pragma unroll 8
    for (int sp = grp; sp < O.nsp; sp += kRedGroups) a += p[static_cast<size_t>(O.sp0 + sp) * nblk * 4096];
    red[grp][el] = a;
    __syncthreads();
    if (grp) return;
    double v = red[0][el];
#pragma unroll
    for (int g = 1; g < kRedGroups; ++g) v += red[g][el];
    // register r, lane l: row 4 r + l / 16, column l % 16
    const int m = m0 + 4 * (el >> 6) + ((el & 63) >> 4), c = n0 + (el & 15);
    if (m >= n || c >= n || (upper && m > c)) return;
    double* o = O.out + static_cast<size_t>(m) * n + c;
    *o = v + (accumulate ? *o : 0.0);
    if (upper && m != c) {
        double* ot = O.out + static_cast<size_t>(c) * n + m;
        *ot = v + (accumulate ? *ot : 0.0);
    }
}

// K (+)= M + M^T: the pair (m, c), (c, m) gets the same sum
__global__ __launch_bounds__(256) void k_add_transpose(const double* __restrict__ M, int n, double* __restrict__ K,
                                                       int accumulate) {
    __shared__ double t[16][17];
    const int bi = blockIdx.y, bj = blockIdx.x;
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    const int tm = bj * 16 + r, tc = bi * 16 + c;
    t[r][c] = (tm < n && tc < n) ? M[static_cast<size_t>(tm) * n + tc] : 0.0;
    __syncthreads();
    const int m = bi * 16 + r, q = bj * 16 + c;
    if (m >= n || q >= n) return;
    const double a = M[static_cast<size_t>(m) * n + q], b = t[c][r];
    double* o = K + static_cast<size_t>(m) * n + q;
    *o = a + b + (accumulate ? *o : 0.0);
}

// ------------------------------------------------------------------ adjoint
// With X_Q = B_Q C, Y_Q = C^T X_Q (o x o) and d_Q = tr Y_Q, every term of the adjoint of
// E = tr(D (2J - K)) comes from X and Z_Q = 2 d_Q 1 - Y_Q, with neither J, K nor D:
//   E = sum_Q tr(Y_Q Z_Q), dE/dC = 4 sum_Q X_Q Z_Q, dE/dB_Q = 2 C Z_Q C^T.
// For o = n/5 that is 0.4 of the products that J, K, (2J - K) C and 4 d D - 2 (C Y) C^T take, and B
// is read once.  All operands are again register images of the kernel before.
__global__ __launch_bounds__(256) void k_pack_rows(const double* __restrict__ C, int ld, int ncol, int nbf, int n,
                                                   int ncb, double* __restrict__ CB) {
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < n; idx += gridDim.x * 256) {
        const int e = idx & 1, lane = (idx >> 1) & 63, rest = idx >> 7;
        const int kb = rest / ncb, cb = rest % ncb;
        const int m = 8 * kb + 4 * e + (lane >> 4), c = 16 * cb + (lane & 15);
        CB[idx] = (m < nbf && c < ncol) ? C[static_cast<size_t>(m) * ld + c] : 0.0;
    }
}

// NC-wide groups of ncb blocks: the first ncb - ng (NC - 1) are NC wide, the others NC - 1
__device__ inline int group_start(int g, int ncb, int ng, int NC) {
    return g * NC - max(0, g - (ncb - ng * (NC - 1)));
}

// Y and Z of one q: blocks [i0, i0 + NI) x [j0, j0 + NJ) of the symmetric Y, the ones below the diagonal
// (DIAG: i0 = j0) stored as mirror images.  X is gathered 8 bytes per lane in the transposed sense (rows
// along the sum); each 16 x 16 piece feeds NI MFMA steps, so the gather (32 cache cycles) hides under
// them.  1856 Q / nbf 384 / 80 columns: 0.152 ms, 15 of 25 sub-tiles (every sub-tile in four waves: 0.265).
template <int NI, int NJ, bool DIAG>
__device__ __forceinline__ void adj_z_body(const double* __restrict__ CB, const double* __restrict__ Xq, int nkb, int ncb,
                                           int i0, int j0, double dq, double* __restrict__ Zq,
                                           double* __restrict__ ep) {
    const int lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const unsigned off_c = lane * 16;
    const unsigned off_x = ((lj >> 3) * 128 + (lj & 3) * 32 + ((lj >> 2) & 1) + lg * 2) * 8;
    const int nkx = 2 * ncb;
    d4_t acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
    d2_t a0[NI], a1[NI], b0[NJ], b1[NJ];
    auto load = [&](int kb, d2_t* a, d2_t* b) {
        kb = min(kb, nkb - 1);
        const double* ca = CB + (static_cast<size_t>(kb) * ncb + i0) * 128;
#pragma unroll
        for (int i = 0; i < NI; ++i) a[i] = ld2(ca + 128 * i, off_c);
        const double* x = Xq + (static_cast<size_t>(kb >> 1) * nkx + 2 * j0) * 128 + 16 * (kb & 1);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            b[j].x = ld1(x + 256 * j, off_x);
            b[j].y = ld1(x + 256 * j + 8, off_x);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const d2_t* a, const d2_t* b) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    if (!DIAG || i <= j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    load(0, a0, b0);
    for (int kb = 0; kb < nkb; kb += 2) {  // nkb is even
        load(kb + 1, a1, b1);
        mul(a0, b0);
        load(kb + 2, a0, b0);
        mul(a1, b1);
    }
    // mirror image: element 4 r + lg of a row in lane lj is row lj, element 4 r + lg
    const unsigned off_m = ((lj >> 3) * ncb * 128 + ((lj & 3) * 16 + lg) * 2 + ((lj >> 2) & 1)) * 8;
    double es = 0.0;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (DIAG && i > j) continue;
            double ts = 0.0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                d2_t z;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const double y = acc[i][j][2 * h + e];
                    const bool diag = DIAG && i == j && 8 * h + 4 * e + lg == lj;
                    z[e] = (diag ? 2.0 * dq : 0.0) - y;
                    ts = fma(y, z[e], ts);
                }
                *reinterpret_cast<d2_t*>(reinterpret_cast<char*>(
                                             Zq + (static_cast<size_t>(2 * (i0 + i) + h) * ncb + j0 + j) * 128) + off_c) = z;
            }
            if (!DIAG || i < j) {
                ts *= 2.0;
                double* zm = Zq + (static_cast<size_t>(2 * (j0 + j)) * ncb + i0 + i) * 128;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *reinterpret_cast<double*>(reinterpret_cast<char*>(zm + 8 * r) + off_m) = -acc[i][j][r];
            }
            es += ts;
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) es += __shfl_xor(es, o);
    if (lane == 0) *ep = es;
}

__global__ __launch_bounds__(256, 2) void k_adj_z(const double* __restrict__ CB, const double* __restrict__ X, int nT,
                                                  int ncb, int ng, int nc, int nq, const double* __restrict__ d,
                                                  double* __restrict__ Z, double* __restrict__ epart) {
    const int items = ng * (ng + 1) / 2;
    const WaveItem w = wave_item(items);
    if (w.group >= nq) return;
    int gi = 0, gj = w.item;
    while (gj >= ng - gi) {
        gj -= ng - gi;
        ++gi;
    }
    gj += gi;
    const int q = w.group;
    const int i0 = group_start(gi, ncb, ng, nc), j0 = group_start(gj, ncb, ng, nc);
    const int ni = group_start(gi + 1, ncb, ng, nc) - i0, nj = group_start(gj + 1, ncb, ng, nc) - j0;
    const double* Xq = X + static_cast<size_t>(q) * nT * 4 * ncb * 128;
    double* Zq = Z + static_cast<size_t>(q) * 2 * ncb * ncb * 128;
    double* ep = epart + static_cast<size_t>(q) * items + w.item;
    const double dq = d[q];
#define P4A_Z(NI, NJ, DIAG)                        \
    if (ni == NI && nj == NJ && (gi == gj) == DIAG) \
    return adj_z_body<NI, NJ, DIAG>(CB, Xq, 4 * nT, ncb, i0, j0, dq, Zq, ep)
    P4A_Z(5, 5, true);
    P4A_Z(4, 4, true);
    P4A_Z(3, 3, true);
    P4A_Z(2, 2, true);
    P4A_Z(1, 1, true);
    P4A_Z(4, 4, false);
    P4A_Z(4, 3, false);
    P4A_Z(3, 3, false);
#undef P4A_Z
}

// One wave of a product whose right operand is shared or not: NF row fragments x NC column blocks of
// the transposed product, summed over steps; the caller gives the operand addresses of a step.
template <int NF, int NC, class LA, class LC>
__device__ __forceinline__ void frag_product(d4_t (&acc)[NF][NC], int steps, LA&& la, LC&& lc) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[f][c] = d4_t{0.0, 0.0, 0.0, 0.0};
    if (steps <= 0) return;
    d2_t a0[NF], a1[NF], c0[NC], c1[NC];
    auto load = [&](int st, d2_t* a, d2_t* c) {
        st = min(st, steps - 1);
        la(st, a);
        lc(st, c);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](const d2_t* a, const d2_t* c) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    acc[f][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(c[i][e], a[f][e], acc[f][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    load(0, a0, c0);
    int st = 0;
    for (; st + 1 < steps; st += 2) {
        load(st + 1, a1, c1);
        mul(a0, c0);
        load(st + 2, a0, c0);
        mul(a1, c1);
    }
    if (st < steps) mul(a0, c0);
}

// P_q^T = Z_q C^T: rows of C as the row operand, Z as the column operand
template <int NF, int NC>
__device__ __forceinline__ void adj_p_body(const double* __restrict__ Zq, const double* __restrict__ CD, int ncb, int rb0,
                                           int cb0, double* __restrict__ Pq) {
    const unsigned off = (threadIdx.x & 63) * 16;
    const int nkx = 2 * ncb;
    d4_t acc[NF][NC];
    frag_product<NF, NC>(
        acc, nkx,
        [&](int st, d2_t* a) {
#pragma unroll
            for (int f = 0; f < NF; ++f) a[f] = ld2(CD + (static_cast<size_t>(rb0 + f) * nkx + st) * 128, off);
        },
        [&](int st, d2_t* c) {
#pragma unroll
            for (int i = 0; i < NC; ++i) c[i] = ld2(Zq + (static_cast<size_t>(st) * ncb + cb0 + i) * 128, off);
        });
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 2 * NC; ++i)
            *reinterpret_cast<d2_t*>(reinterpret_cast<char*>(
                                         Pq + (static_cast<size_t>(rb0 + f) * nkx + 2 * cb0 + i) * 128) + off) =
                d2_t{acc[f][i >> 1][2 * (i & 1)], acc[f][i >> 1][2 * (i & 1) + 1]};
}
template <int NC>
__global__ __launch_bounds__(256, 2) void k_adj_p(const double* __restrict__ Z, const double* __restrict__ CD, int nT,
                                                  int ncb, int ng, int nq, double* __restrict__ P) {
    const int nrg = (nT + 1) / 2;
    const WaveItem w = wave_item(nrg * ng);
    if (w.group >= nq) return;
    const int q = w.group, rg = w.item / ng, gc = w.item % ng;
    const int cb0 = group_start(gc, ncb, ng, NC);
    const bool wide = group_start(gc + 1, ncb, ng, NC) - cb0 == NC;
    const double* Zq = Z + static_cast<size_t>(q) * 2 * ncb * ncb * 128;
    double* Pq = P + static_cast<size_t>(q) * nT * 4 * ncb * 128;
    const bool full = 2 * rg + 2 <= nT;
    if (full) {
        if (wide)
            adj_p_body<4, NC>(Zq, CD, ncb, 4 * rg, cb0, Pq);
        else if constexpr (NC > 1)
            adj_p_body<4, NC - 1>(Zq, CD, ncb, 4 * rg, cb0, Pq);
    } else {
        if (wide)
            adj_p_body<2, NC>(Zq, CD, ncb, 4 * rg, cb0, Pq);
        else if constexpr (NC > 1)
            adj_p_body<2, NC - 1>(Zq, CD, ncb, 4 * rg, cb0, Pq);
    }
}

// G_q = 2 P_q C^T, a 64 x 64 block on or above the diagonal, written with its mirror image.  Bound
// by writing G (8 n^2 bytes per q).  The mirror image is turned in registers, so that a lane stores 32
// consecutive bytes; stores pass the caches by.  Nbf 384 / 1856 Q (2.19 GB) / 80 columns: 0.71 ms, 3.1 TB/s
// (8-byte mirror stores: 0.84; cached ones 0.74; without the product 0.44; 32 x 64 blocks at twice the
// occupancy 0.82).
template <int NI, int NJ, bool DIAG>
__device__ __forceinline__ void adj_g_body(const double* __restrict__ Pq, const double* __restrict__ CD, int nkx, int nk,
                                           int rb0, int cb0, int n, double* __restrict__ G) {
    const int lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const unsigned off = lane * 16;
    d4_t acc[NJ][NI];
    // the transposed product: rows of G along the MFMA rows, columns along its columns
    frag_product<NJ, NI>(
        acc, nk,
        [&](int st, d2_t* a) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) a[j] = ld2(CD + (static_cast<size_t>(cb0 + j) * nkx + st) * 128, off);
        },
        [&](int st, d2_t* c) {
#pragma unroll
            for (int i = 0; i < NI; ++i) c[i] = ld2(Pq + (static_cast<size_t>(rb0 + i) * nkx + st) * 128, off);
        });
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (DIAG && i > j) continue;
            const bool diag = DIAG && i == j;
            const int m0 = 16 * (rb0 + i), c = 16 * (cb0 + j) + lj;
            double v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + 4 * r + lg;
                v[r] = 2.0 * acc[j][i][r];
                if (m < n && c < n && (!diag || m <= c)) __builtin_nontemporal_store(v[r], G + static_cast<size_t>(m) * n + c);
            }
            transpose4(v);
            const int m = m0 + 4 * lg;
            double* g = G + static_cast<size_t>(c) * n + m;
            if (!diag && m + 4 <= n) {
                if (c < n) {
                    __builtin_nontemporal_store(d2u_t{v[0], v[1]}, reinterpret_cast<d2u_t*>(g));
                    __builtin_nontemporal_store(d2u_t{v[2], v[3]}, reinterpret_cast<d2u_t*>(g + 2));
                }
            } else if (c < n) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (m + r < n && (!diag || m + r <= c)) g[r] = v[r];
            }
        }
}
__global__ __launch_bounds__(256, 2) void k_adj_g(const double* __restrict__ P, const double* __restrict__ CD, int nT,
                                                  int ncb, int nk, int nq, int n, int nbr, int nblk,
                                                  double* __restrict__ G) {
    const WaveItem w = wave_item(nblk);
    if (w.group >= nq) return;
    int I = 0, r = w.item;
    while (r >= nbr - I) {
        r -= nbr - I;
        ++I;
    }
    const int J = I + r, nkx = 2 * ncb;
    const double* Pq = P + static_cast<size_t>(w.group) * nT * 4 * ncb * 128;
    double* Gq = G + static_cast<size_t>(w.group) * n * n;
    const bool fj = 4 * J + 4 <= 2 * nT;
    if (I == J) {
        if (fj)
            adj_g_body<4, 4, true>(Pq, CD, nkx, nk, 4 * I, 4 * J, n, Gq);
        else
            adj_g_body<2, 2, true>(Pq, CD, nkx, nk, 4 * I, 4 * J, n, Gq);
    } else if (fj) {
        adj_g_body<4, 4, false>(Pq, CD, nkx, nk, 4 * I, 4 * J, n, Gq);
    } else {
        adj_g_body<4, 2, false>(Pq, CD, nkx, nk, 4 * I, 4 * J, n, Gq);
    }
}

// sum over (q, k) of X_q Z_q: one wave takes 4 (or 2) row fragments x NC column blocks of one split
template <int NF, int NC>
__device__ __forceinline__ void adj_dc_body(const double* __restrict__ X, const double* __restrict__ Z, size_t xq,
                                            size_t zq, int ncb, int nk, int rb0, int cb0, int s0, int s1,
                                            double* __restrict__ part, int accumulate) {
    const int lane = threadIdx.x & 63;
    const unsigned off = lane * 16;
    const int nkx = 2 * ncb;
    d4_t acc[NF][NC];
    // steps are taken in order: (q, k) of the step being loaded
    int q = s0 / nk, k = s0 % nk, at = 0;
    auto advance = [&](int st) {
        if (st > at) {
            at = st;
            if (++k == nk) {
                k = 0;
                ++q;
            }
        }
    };
    frag_product<NF, NC>(
        acc, s1 - s0,
        [&](int st, d2_t* a) {
            advance(st);
            const double* p = X + q * xq + (static_cast<size_t>(rb0) * nkx + k) * 128;
#pragma unroll
            for (int f = 0; f < NF; ++f) a[f] = ld2(p + static_cast<size_t>(f) * nkx * 128, off);
        },
        [&](int, d2_t* c) {
            const double* p = Z + q * zq + (static_cast<size_t>(k) * ncb + cb0) * 128;
#pragma unroll
            for (int i = 0; i < NC; ++i) c[i] = ld2(p + 128 * i, off);
        });
    // acc holds the transposed product: lane m + 16 (column % 4), register column / 4
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double* o = part + (static_cast<size_t>(rb0 + f) * ncb + cb0 + i) * 256 + r * 64 + lane;
                *o = acc[f][i][r] + (accumulate ? *o : 0.0);
            }
}
template <int NC>
__global__ __launch_bounds__(64, 2) void k_adj_dc(const double* __restrict__ X, const double* __restrict__ Z, int nT,
                                                  int ncb, int ng, int nk, int nq, int nsplit,
                                                  double* __restrict__ partial, int accumulate) {
    const int nrg = (nT + 1) / 2;
    const WaveItem w = wave_item(nrg * ng);
    if (w.group >= nsplit) return;
    const int sp = w.group, rg = w.item / ng, gc = w.item % ng;
    const int cb0 = group_start(gc, ncb, ng, NC);
    const bool wide = group_start(gc + 1, ncb, ng, NC) - cb0 == NC;
    const long long steps = static_cast<long long>(nq) * nk;
    const int s0 = uni(static_cast<int>(steps * sp / nsplit)), s1 = uni(static_cast<int>(steps * (sp + 1) / nsplit));
    const size_t xq = static_cast<size_t>(nT) * 4 * ncb * 128, zq = static_cast<size_t>(2) * ncb * ncb * 128;
    double* part = partial + static_cast<size_t>(sp) * 2 * nT * ncb * 256;
#define P4A_DC(NF, N) adj_dc_body<NF, N>(X, Z, xq, zq, ncb, nk, 4 * rg, cb0, s0, s1, part, accumulate)
    if (2 * rg + 2 <= nT) {
        if (wide)
            P4A_DC(4, NC);
        else if constexpr (NC > 1)
            P4A_DC(4, NC - 1);
    } else {
        if (wide)
            P4A_DC(2, NC);
        else if constexpr (NC > 1)
            P4A_DC(2, NC - 1);
    }
#undef P4A_DC
}
__global__ __launch_bounds__(256 * kRedGroups) void k_adj_dc_reduce(const double* __restrict__ partial, int nsplit,
                                                                   size_t stride, int ncb, int n, int ncol, double alpha,
                                                                   double* __restrict__ out) {
    __shared__ double red[kRedGroups][256];
    const int cb = blockIdx.x, rb = blockIdx.y;
    const int el = threadIdx.x & 255, grp = threadIdx.x >> 8;
    const double* p = partial + (static_cast<size_t>(rb) * ncb + cb) * 256 + el;
    double a = 0.0;
#pragma unroll 8
    for (int sp = grp; sp < nsplit; sp += kRedGroups) a += p[sp * stride];
    red[grp][el] = a;
    __syncthreads();
    if (grp) return;
    double v = red[0][el];
#pragma unroll
    for (int g = 1; g < kRedGroups; ++g) v += red[g][el];
    const int m = 16 * rb + (el & 15), c = 16 * cb + 4 * (el >> 6) + ((el & 63) >> 4);
    if (m < n && c < ncol) out[static_cast<size_t>(m) * ncol + c] = alpha * v;
}

}  // namespace

// ------------------------------------------------------------------ launchers
void launch_pack_frag(const ColGroups& cg, int nbf, int nbfp, double* CA, double* CD, hipStream_t s) {
    require(cg.n >= 1 && cg.n <= kMaxGroups && nbfp % TILE == 0 && nbfp >= nbf && (CA || CD), "pack_frag");
    int most = 0;
    for (int i = 0; i < cg.n; ++i) {
        const ColGroup& G = cg.g[i];
        require(G.ncb > 0 && G.cb0 >= 0 && G.cb0 + G.ncb <= cg.ncb && G.src && G.ld >= (G.cmap ? 1 : G.ncol) &&
                    (G.cmap || G.ncol <= 16 * G.ncb),
                "pack_frag group");
        most = std::max(most, G.ncb);
    }
    require(static_cast<long long>(nbfp) * 16 * most < (1LL << 31), "pack_frag size");
    const int nb = std::min(4096, (nbfp * 16 * most + 255) / 256);
    hipLaunchKernelGGL(k_pack_frag, dim3(nb, cg.n), dim3(256), 0, s, cg, nbf, nbfp, CA, CD);
}

// Row tiles per wave.  Two halve the traffic of the C operand and are faster once the launch fills
// the chip several times over; with fewer waves than that one tile per wave wastes less of the last
// round.  Time in units of one row tile over all columns: rounds of the XCD's wave slots x tiles per
// wave (a 2-tile wave costs a little less than two 1-tile waves).
int ht_row_tiles(int nT, int nq, int ncb) {
    const int ncg = (ncb + 4) / 5;
    auto rounds = [&](int rt) {
        const double w = std::ceil(nq / static_cast<double>(kXCD)) * ht_row_groups(nT, rt) * ncg / kSlots;
        return w < 8.0 ? std::ceil(w) : w + 0.5;
    };
    return 1.8 * rounds(2) <= rounds(1) ? 2 : 1;
}

template <int RT>
static void ht_f64_rt(const TileGeom& g, const double* B, int nq, const double* CA, const double* CD, int ncb,
                      double* X, double* dpart, const double* zt, hipStream_t s) {
    const int ncg = (ncb + 4) / 5, nc = (ncb + ncg - 1) / ncg;
    const dim3 grid(wave_grid(nq, ht_row_groups(g.nT, RT) * ncg, 4));
#define P4A_HT(N)                                                                                                     \
    case N:                                                                                                           \
        hipLaunchKernelGGL((k_ht_f64<RT, N>), grid, dim3(256), 0, s, B, g.d_tidx, g.nT, g.ntp, nq, CA, CD, ncb, ncg, X, \
                           dpart, zt);                                                                                \
        break;
    switch (nc) { P4A_HT(1) P4A_HT(2) P4A_HT(3) P4A_HT(4) P4A_HT(5) }
#undef P4A_HT
}

void launch_ht_f64(const TileGeom& g, const double* B, int nq, const double* CA, const double* CD, int ncb, int rt,
                   double* X, double* dpart, const void* zt, hipStream_t s) {
    require(nq > 0 && ncb > 0 && (rt == 1 || rt == 2) && g.nT > 0 && g.nT <= 256 && g.nbfp == g.nT * TILE && zt &&
                (!CD || dpart) &&
                static_cast<double>(nq) * ht_row_groups(g.nT, rt) * ((ncb + 4) / 5) < 4.0e9,
            "ht_f64 shape");
    if (rt == 1)
        ht_f64_rt<1>(g, B, nq, CA, CD, ncb, X, dpart, static_cast<const double*>(zt), s);
    else
        ht_f64_rt<2>(g, B, nq, CA, CD, ncb, X, dpart, static_cast<const double*>(zt), s);
}

void launch_dpart_reduce(const double* dpart, int nq, int nrg, int ncb, const DRanges& r, double* d, int ldd,
                         hipStream_t s) {
    require(r.n >= 1 && r.n <= kMaxPairs && nq > 0 && ldd >= nq, "dpart_reduce");
    hipLaunchKernelGGL(k_dpart_reduce, dim3((nq + 3) / 4, r.n), dim3(256), 0, s, dpart, nq, nrg, ncb, r, d, ldd);
}

int kc_block_rows(int nT) { return (nT + 1) / 2; }

int kc_choose_splits(int nT, bool upper, int steps, int nseg, int max_splits) {
    return balanced_splits(static_cast<long long>(kc_blocks(nT, upper)) * nseg, steps, max_splits);
}

void launch_kc_f64(const double* XA, const double* XB, size_t qstride, int nkx, int nT, int nq, const KcSegs& segs,
                   bool upper, double* P, int accumulate, hipStream_t s) {
    require(segs.n >= 1 && segs.n <= kMaxSegs && nq > 0 && nkx > 0 && nT > 0 && segs.nsplit > 0, "kc_f64 shape");
    int at = 0;
    for (int i = 0; i < segs.n; ++i) {
        const KcSeg& g = segs.s[i];
        require(g.sp0 == at && g.nsp > 0 && g.nk > 0 && g.ka >= 0 && g.kb >= 0 && g.ka + g.nk <= nkx &&
                    g.kb + g.nk <= nkx && (!upper || g.ka == g.kb) && static_cast<long long>(nq) * g.nk < (1LL << 31),
                "kc_f64 pass");
        at += g.nsp;
    }
    require(at == segs.nsplit && (!upper || XA == XB), "kc_f64 splits");
    const int nbr = kc_block_rows(nT), nblk = kc_blocks(nT, upper);
    const dim3 grid(wave_grid(segs.nsplit, nblk, 1));
    if (upper)
        hipLaunchKernelGGL((k_kc_f64<true>), grid, dim3(64), 0, s, XA, XB, qstride, nkx, nT, nq, segs, nbr, nblk, P,
                           accumulate);
    else
        hipLaunchKernelGGL((k_kc_f64<false>), grid, dim3(64), 0, s, XA, XB, qstride, nkx, nT, nq, segs, nbr, nblk, P,
                           accumulate);
}

void launch_kc_reduce(const double* P, int nT, int n, bool upper, const KcOuts& outs, int accumulate, hipStream_t s,
                      const JUnpack* ju) {
    static_assert(256 * kRedGroups == 128 * kJuGroups, "one workgroup size");
    require(outs.n >= 1 && outs.n <= 2 * kMaxPairs && n > 0 && n <= nT * TILE, "kc_reduce");
    const int nblk = kc_blocks(nT, upper);
    const int nj = ju ? ju->ntp * (TILE2 / 128) * ju->np : 0;
    hipLaunchKernelGGL(k_kc_reduce, dim3(nblk, 16, outs.n + (nj + 16 * nblk - 1) / (16 * nblk)), dim3(256 * kRedGroups), 0,
                       s, P, nblk, kc_block_rows(nT), n, upper ? 1 : 0, outs, accumulate, ju ? *ju : JUnpack{});
}

void launch_add_transpose(const double* M, int n, double* K, int accumulate, hipStream_t s) {
    const int nb = (n + 15) / 16;
    hipLaunchKernelGGL(k_add_transpose, dim3(nb, nb), dim3(256), 0, s, M, n, K, accumulate);
}

// ---- adjoint ----
void launch_pack_rows(const double* C, int ld, int ncol, int nbf, int nbfp, int ncb, double* CB, hipStream_t s) {
    require(ncol > 0 && ld >= ncol && ncol <= 16 * ncb && nbfp >= nbf && nbfp % TILE == 0 &&
                static_cast<long long>(nbfp) * 16 * ncb < (1LL << 31),
            "pack_rows");
    const int n = nbfp * 16 * ncb;
    hipLaunchKernelGGL(k_pack_rows, dim3(std::min(4096, (n + 255) / 256)), dim3(256), 0, s, C, ld, ncol, nbf, n, ncb, CB);
}

// Up to 5 blocks in one group (the upper 15 of 25 sub-tiles fit the registers), more in groups of 3 or 4
static int z_groups(int ncb) { return ncb <= 5 ? 1 : (ncb + 3) / 4; }
int adj_z_waves(int ncb) { return z_groups(ncb) * (z_groups(ncb) + 1) / 2; }
void launch_adj_z(const double* CB, const double* X, int nT, int ncb, int nq, const double* d, double* Z, double* epart,
                  hipStream_t s) {
    require(nT > 0 && ncb > 0 && nq > 0, "adj_z");
    const int ng = z_groups(ncb), nc = (ncb + ng - 1) / ng;
    hipLaunchKernelGGL(k_adj_z, dim3(wave_grid(nq, adj_z_waves(ncb), 4)), dim3(256), 0, s, CB, X, nT, ncb, ng, nc, nq, d,
                       Z, epart);
}

template <class F>
static void with_groups(int ncb, F&& f) {
    const int ng = (ncb + 4) / 5, nc = (ncb + ng - 1) / ng;
    switch (nc) {
        case 1: f(std::integral_constant<int, 1>{}, ng); break;
        case 2: f(std::integral_constant<int, 2>{}, ng); break;
        case 3: f(std::integral_constant<int, 3>{}, ng); break;
        case 4: f(std::integral_constant<int, 4>{}, ng); break;
        default: f(std::integral_constant<int, 5>{}, ng); break;
    }
}
void launch_adj_p(const double* Z, const double* CD, int nT, int ncb, int nq, double* P, hipStream_t s) {
    require(nT > 0 && ncb > 0 && nq > 0, "adj_p");
    with_groups(ncb, [&](auto nc, int ng) {
        constexpr int NC = decltype(nc)::value;
        hipLaunchKernelGGL((k_adj_p<NC>), dim3(wave_grid(nq, kc_block_rows(nT) * ng, 4)), dim3(256), 0, s, Z, CD, nT, ncb,
                           ng, nq, P);
    });
}
void launch_adj_g(const double* P, const double* CD, int nT, int ncb, int nk, int nq, int n, double* G, hipStream_t s) {
    require(nT > 0 && nk > 0 && nk <= 2 * ncb && nq > 0 && n <= nT * TILE, "adj_g");
    const int nblk = kc_blocks(nT, true);
    hipLaunchKernelGGL(k_adj_g, dim3(wave_grid(nq, nblk, 4)), dim3(256), 0, s, P, CD, nT, ncb, nk, nq, n,
                       kc_block_rows(nT), nblk, G);
}
int adj_dc_splits(int nT, int ncb, int steps) {
    return balanced_splits(kc_block_rows(nT) * ((ncb + 4) / 5), steps, 4096);
}
void launch_adj_dc(const double* X, const double* Z, int nT, int ncb, int nk, int nq, int nsplit, double* partial,
                   int accumulate, hipStream_t s) {
    require(nT > 0 && nk > 0 && nk <= 2 * ncb && nq > 0 && nsplit > 0 && static_cast<long long>(nq) * nk < (1LL << 31),
            "adj_dc");
    with_groups(ncb, [&](auto nc, int ng) {
        constexpr int NC = decltype(nc)::value;
        hipLaunchKernelGGL((k_adj_dc<NC>), dim3(wave_grid(nsplit, kc_block_rows(nT) * ng, 1)), dim3(64), 0, s, X, Z, nT,
                           ncb, ng, nk, nq, nsplit, partial, accumulate);
    });
}
void launch_adj_dc_reduce(const double* partial, int nsplit, int nT, int ncb, int n, int ncol, double alpha, double* out,
                          hipStream_t s) {
    require(nsplit > 0 && n <= nT * TILE && ncol <= 16 * ncb, "adj_dc_reduce");
    hipLaunchKernelGGL(k_adj_dc_reduce, dim3(ncb, 2 * nT), dim3(256 * kRedGroups), 0, s, partial, nsplit,
                       adj_dc_partial(nT, ncb), ncb, n, ncol, alpha, out);
}

}  // namespace p4a
