// Device helpers of the wave-level MFMA kernels (kernels_f64.hip, kernels_f32.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace p4a {
namespace {

typedef double d2_t __attribute__((ext_vector_type(2)));

constexpr int kXCD = 8;
constexpr int kSlots = 256;  // waves one XCD holds: 32 CUs x 4 SIMDs x 2 waves

// 16 bytes at a wave-uniform base plus a per-lane byte offset
__device__ inline d2_t ld2(const double* base, unsigned off) {
    return *reinterpret_cast<const d2_t*>(reinterpret_cast<const char*>(base) + off);
}
__device__ inline double ld1(const double* base, unsigned off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
}
__device__ inline int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
// v[r] in lane group g (lanes 16 g ..) becomes v[g] in lane group r: after an FP64 MFMA, four consecutive rows
// of a column in a lane instead of four rows 4 apart.
__device__ __forceinline__ void transpose4(double* v) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef unsigned u2_t __attribute__((ext_vector_type(2)));
    auto swap = [](double& a, double& b, auto&& f) {
        u2_t x = __builtin_bit_cast(u2_t, a), y = __builtin_bit_cast(u2_t, b);
        const u2_t l = f(x[0], y[0]), h = f(x[1], y[1]);
        a = __builtin_bit_cast(double, u2_t{l[0], h[0]});
        b = __builtin_bit_cast(double, u2_t{l[1], h[1]});
    };
    // lanes 32..63 of the first with lanes 0..31 of the second; odd 16-lane rows with even ones
    auto s32 = [](unsigned x, unsigned y) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
        return u2_t{r[0], r[1]};
    };
    auto s16 = [](unsigned x, unsigned y) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        return u2_t{r[0], r[1]};
    };
    swap(v[0], v[2], s32);
    swap(v[1], v[3], s32);
    swap(v[0], v[1], s16);
    swap(v[2], v[3], s16);
#endif
}

// Workgroups go round-robin to the XCDs (each with its own L2): wave w of the launch belongs to XCD
// (workgroup % 8); consecutive waves of an XCD take the items of one group (the row and column blocks
// of one Q, the output blocks of one split), so a group's operands meet in one L2.
struct WaveItem {
    int group, item;
};
__device__ inline WaveItem wave_item(int items) {
    const int wg = blockIdx.x, lw = (wg / kXCD) * (blockDim.x >> 6) + uni(threadIdx.x >> 6);
    return {(lw / items) * kXCD + wg % kXCD, lw % items};
}
inline unsigned wave_grid(int ngroups, int items, int wpw) {  // wpw: waves per workgroup
    const long long per = static_cast<long long>((ngroups + kXCD - 1) / kXCD) * items;  // waves per XCD
    return static_cast<unsigned>(kXCD * ((per + wpw - 1) / wpw));
}

// Order of a step's instructions: each of its NL loads is followed by its share of the NM MFMAs.  Loads issued in
// one burst hold up the wave's MFMAs for as long as the four SIMDs' bursts occupy the address path.  With
// the tile rows below it took the FP64 half-transform at nbf 413 / 144 columns from 1.96 to 1.87 ms; the
// contractions, whose operands come from further away, were 1-9 % slower with it and load in one burst.
template <int NL, int NM>
__device__ __forceinline__ void interleave() {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, NM / NL, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NM - NM / NL * NL, 0);
    __builtin_amdgcn_sched_barrier(0);
}

// The column tiles of a row of tiles (RT tile rows taken together) in order, absent ones passed over:
// a lane holds the tile indices of one column, so the next tile is a find-first-set and a lane read
// instead of a chain of scalar loads (about 1 us each, in the open between two steps).
template <int RT>
struct TileRow {
    const int* tidx;
    int nT, I0, base;
    int o[RT];
    unsigned long long mask;
    __device__ __forceinline__ void fill(int b) {
        base = b;
        const int lane = threadIdx.x & 63, j = min(b + lane, nT - 1);
        bool any = false;
#pragma unroll
        for (int s = 0; s < RT; ++s) {
            const int I = I0 + s;
            o[s] = tidx[min(I, j) * nT + max(I, j)];
            any |= o[s] >= 0;
        }
        mask = __ballot(any && b + lane < nT);
    }
    __device__ __forceinline__ TileRow(const int* t, int n, int I) : tidx(t), nT(n), I0(I) { fill(0); }
    // column of the next tile (nT: none left) and its index in each row (-1: absent)
    __device__ __forceinline__ int next(int* idx) {
        while (!mask) {
            if (base + 64 >= nT) return nT;
            fill(base + 64);
        }
        const int l = __builtin_ctzll(mask);
        mask &= mask - 1;
#pragma unroll
        for (int s = 0; s < RT; ++s) idx[s] = __builtin_amdgcn_readlane(o[s], l);
        return base + l;
    }
};

// Splits of `steps` steps when a split is nw waves.  A wave's partial sums (32 KB written and read
// again) cost about as much as 10 steps, and the waves of a launch end unevenly, which costs about half a
// round of the chip's 2048 wave slots: 10 ns / steps + 1024 / (ns nw) is least at ns = sqrt(102 steps / nw)
// (nbf 576 / 120 columns / 2784 Q in FP64: 307; measured 2.43, 2.23, 2.17, 2.19 ms with 96, 144, 288, 384).
// Where the launch streams more X than the L2s hold, about 320 steps a split keep a split's waves
// within 8 Q of one another (see k_kc_f64).  A launch of between one and three rounds is cut to whole ones (2000
// k8 steps of 3 x 3 x 3 blocks: 0.19 -> 0.165 ms; the adjoint's dE/dC at nbf 384: 0.206 -> 0.170).  At least 4
// steps; multiples of 8, one split per XCD.
inline int balanced_splits(long long nw, int steps, int max_splits) {
    constexpr double slots = kXCD * kSlots;
    long long ns = std::max<long long>(steps / 320, std::llround(std::sqrt(102.0 * steps / nw)));
    const double rounds = ns * static_cast<double>(nw) / slots;
    if (rounds > 1 && rounds < 3) ns = static_cast<long long>(std::floor(rounds) * slots / nw);
    ns = std::max<long long>(1, std::min<long long>({ns, steps / 4, max_splits}));
    return static_cast<int>(ns >= 8 ? ns / 8 * 8 : ns);
}

}  // namespace
}  // namespace p4a
