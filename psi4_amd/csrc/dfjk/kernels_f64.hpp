// Launchers of the FP64 J/K path (kernels_f64.hip): wave-level MFMA kernels whose operands are
// stored in MFMA fragment order, so every load is a contiguous 1 KB per wave and neither LDS nor
// barriers are needed.
//
// Columns come in groups (one orbital matrix each), padded to blocks of 16 columns and laid side by
// side; a "k8" is 8 columns of X, the depth of one contraction step (two MFMAs).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "kernels.hpp"

namespace p4a {

constexpr int kMaxGroups = 8;   // column groups of one half-transform
constexpr int kMaxPairs = 4;    // density pairs of one batch
constexpr int kMaxSegs = 8;     // contraction passes of one launch

// One group of columns: src [nbf][ld]; partner (or null): the matrix whose product with X gives d_Q;
// cmap (or null): source column of each padded column (-1: zero).
struct ColGroup {
    const double* src;
    const double* partner;
    const int* cmap;
    int ld, ncol;
    int cb0, ncb;  // first 16-column block and their number
};
struct ColGroups {
    int n = 0, ncb = 0;  // groups, column blocks over all groups
    ColGroup g[kMaxGroups];
};

// CA: the half-transform's operand [nbfp/8][ncb][64][2]; CD: the partners in X's own layout
// [nbfp/16][2 ncb][64][2].  Either may be null.
void launch_pack_frag(const ColGroups& cg, int nbf, int nbfp, double* CA, double* CD, hipStream_t s);

// X[q][nbfp/16][2 ncb][64][2] = B_q C for q < nq, and with CD also
// dpart[q][row groups][ncb] = sum over the rows of the group and the columns of the block of X * CD.
// ht_row_tiles: row tiles (32 rows) per wave, 1 or 2, for this shape.
int ht_row_tiles(int nT, int nq, int ncb);
inline int ht_row_groups(int nT, int rt) { return (nT + rt - 1) / rt; }
void launch_ht_f64(const TileGeom& g, const double* B, int nq, const double* CA, const double* CD, int ncb, int rt,
                   double* X, double* dpart, const void* zt, hipStream_t s);
// d[p * ldd + q] = sum of dpart[q][*][cb0_p .. cb0_p + ncb_p)
struct DRanges {
    int n = 0;
    int cb0[kMaxPairs], ncb[kMaxPairs];
};
void launch_dpart_reduce(const double* dpart, int nq, int nrg, int ncb, const DRanges& r, double* d, int ldd,
                         hipStream_t s);

// One pass of the contraction: splits [sp0, sp0 + nsp) of P take
// alpha * sum_{q, k < nk} X[q][rows][ka + k] . X[q][rows'][kb + k]^T
struct KcSeg {
    int sp0, nsp, ka, kb, nk;
    double alpha;
};
struct KcSegs {
    int n = 0, nsplit = 0;
    KcSeg s[kMaxSegs];
};
// 64 x 64 output blocks of the contraction: (I, J) over ceil(nbfp / 64) block rows, I <= J first
int kc_block_rows(int nT);
inline int kc_blocks(int nT, bool upper) {
    const int n = kc_block_rows(nT);
    return upper ? n * (n + 1) / 2 : n * n;
}
// P[split][block][16 sub-tiles][4][64] (+)= the passes.  XA, XB: [q][nrb][nkx][64][2].
void launch_kc_f64(const double* XA, const double* XB, size_t qstride, int nkx, int nT, int nq, const KcSegs& segs,
                   bool upper, double* P, int accumulate, hipStream_t s);
// Splits of one pass with `steps` = nq * nk steps when `nseg` passes of this size share the launch.
int kc_choose_splits(int nT, bool upper, int steps, int nseg, int max_splits);
struct KcOut {
    int sp0, nsp;
    double* out;
};
struct KcOuts {
    int n = 0;
    KcOut o[2 * kMaxPairs];  // K and D of each pair
};
// out (+)= sum over the pair's splits; upper: written with its mirror image (exactly symmetric)
// ju (or null): J's reduction, taken along in the same launch
void launch_kc_reduce(const double* P, int nT, int n, bool upper, const KcOuts& outs, int accumulate, hipStream_t s,
                      const JUnpack* ju = nullptr);
// K (+)= M + M^T (n x n)
void launch_add_transpose(const double* M, int n, double* K, int accumulate, hipStream_t s);

// ---- adjoint of E = tr(D (2J - K)), D = C C^T, with ncb 16-column blocks of C ----
// CB [nbfp/8][ncb][64][2]: C in the row order of X's fragments (rows 8 kb + 4 e + lane / 16)
void launch_pack_rows(const double* C, int ld, int ncol, int nbf, int nbfp, int ncb, double* CB, hipStream_t s);
// Y_q = C^T X_q, Z_q = 2 d_q 1 - Y_q as [2 ncb][ncb][64][2]; epart[q][adj_z_waves(ncb)] sums Y Z
int adj_z_waves(int ncb);
void launch_adj_z(const double* CB, const double* X, int nT, int ncb, int nq, const double* d, double* Z, double* epart,
                  hipStream_t s);
// P_q = C Z_q in X's layout
void launch_adj_p(const double* Z, const double* CD, int nT, int ncb, int nq, double* P, hipStream_t s);
// G_q = 2 P_q C^T, dense [nq][n][n], exactly symmetric; nk: k8 steps (ceil(ncol / 8))
void launch_adj_g(const double* P, const double* CD, int nT, int ncb, int nk, int nq, int n, double* G, hipStream_t s);
// partial[split][row block][column block][4][64] (+)= sum_{q, k} X_q[rows][k] Z_q[k][columns]
int adj_dc_splits(int nT, int ncb, int steps);
inline size_t adj_dc_partial(int nT, int ncb) { return static_cast<size_t>(2) * nT * ncb * 256; }  // doubles per split
void launch_adj_dc(const double* X, const double* Z, int nT, int ncb, int nk, int nq, int nsplit, double* partial,
                   int accumulate, hipStream_t s);
// out[n][ncol] = alpha * sum over splits
void launch_adj_dc_reduce(const double* partial, int nsplit, int nT, int ncb, int n, int ncol, double alpha, double* out,
                          hipStream_t s);

}  // namespace p4a
