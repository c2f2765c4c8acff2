// BF16x3 K-path kernels for gfx950: half-transform X_Q = B_Q C and the contraction
// K = sum_Q X_Q S X_Q^T (S = diag of column signs, or a second operand X') in 3-term BF16 split
// precision, staged through LDS, and the conversions and column tests of the mixed modes.
//
// MFMA lane layout (checked on the device):
//   bf16 16x16x32: A[i][8g+e] lane i+16g elem e; B[8g+e][j] lane j+16g elem e;
//   D[i][j] lane j+16(i/4), reg i%4
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.hpp"
#include "kernels_k.hpp"

namespace p4a {

namespace {

__device__ inline uint16_t f2bf(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}
__device__ inline float bf2f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

// Workgroups are dispatched round-robin over the XCDs (flat id w runs on XCD w % 8,
// each XCD with its own L2).  xcd_map turns the flat id into (group, item) so that
// all items of one group -- the row blocks of one Q in the half-transform, the
// output tiles of one Q-split in the contraction -- run on the same XCD and share
// its L2.  The launch uses 8 * ceil(ngroups/8) * items workgroups.
constexpr int kXCD = 8;
struct XcdItem {
    int group, item;
    bool valid;
};
__device__ inline XcdItem xcd_map(int wg, int items, int ngroups) {
    const int xcd = wg % kXCD, local = wg / kXCD;
    XcdItem d;
    d.group = (local / items) * kXCD + xcd;
    d.item = local % items;
    d.valid = d.group < ngroups;
    return d;
}
inline unsigned xcd_grid(int ngroups, int items) {
    return static_cast<unsigned>(kXCD * ((ngroups + kXCD - 1) / kXCD) * items);
}

// Per-workgroup list of the column tiles J that meet at least one of the
// workgroup's RT row tiles, with the element offset of each (row tile, J) block
// in B_Q (or -1), built once in LDS at kernel start (one thread per column tile, positions
// from ballots: two barriers), so the K loop does no dependent tile-table lookups.
constexpr int kMaxColTiles = 256;  // nbf <= 8192
// k-terms an FP32 MFMA accumulator of the K contraction holds before it is folded into FP64
constexpr int kFold32 = 512;

template <int RT>
struct StepList {
    int soff[kMaxColTiles * RT];   // by step
    int J[kMaxColTiles];
    int cnt[kMaxColTiles / 64];
    int n;
};

template <int RT>
__device__ inline void build_steps(StepList<RT>& sl, const int* __restrict__ tidx, int nT, int I0, int tid) {
    const int lane = tid & 63, wv = tid >> 6;
    int off[RT];
    bool present = false;
    unsigned long long mask = 0;
    if (tid < kMaxColTiles) {  // whole waves
        const int j = tid;
#pragma unroll
        for (int s = 0; s < RT; ++s) {
            const int I = I0 + s;
            int t = -1;
            if (j < nT && I < nT) t = tidx[min(I, j) * nT + max(I, j)];
            off[s] = t >= 0 ? t * TILE2 : -1;
            present |= t >= 0;
        }
        mask = __ballot(present);
        if (lane == 0) sl.cnt[wv] = __popcll(mask);
    }
    __syncthreads();
    if (present) {
        int k = __popcll(mask & ((1ull << lane) - 1));
        for (int i = 0; i < wv; ++i) k += sl.cnt[i];
        sl.J[k] = tid;
#pragma unroll
        for (int s = 0; s < RT; ++s) sl.soff[k * RT + s] = off[s];
    }
    if (tid == 0) {
        int n = 0;
        for (int i = 0; i < kMaxColTiles / 64; ++i) n += sl.cnt[i];
        sl.n = n;
    }
    __syncthreads();
}

// BF16 LDS tiles of 32 k per row (64 bytes): the four 16-byte chunks of row r are stored at
// chunk c ^ ((r>>1)&3), so fragment reads (16 rows x one chunk per 16 lanes) and row-segment
// stores (4 lanes per row) are free of bank conflicts.
__device__ inline int kg_swz(int row, int chunk) { return row * 32 + ((chunk ^ ((row >> 1) & 3)) << 3); }

// Split 8 FP32 values into BF16 hi = RNE(x) and lo = RNE(x - hi), packed two per word
// (v_cvt_pk_bf16_f32 rounds to nearest even, as f2bf does).
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef float f2v_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf4v_t __attribute__((ext_vector_type(4)));
typedef unsigned int v4u_t __attribute__((ext_vector_type(4)));
__device__ inline void split_bf16x8(const v4f_t& x, const v4f_t& y, v4u_t& h, v4u_t& l) {
    auto hi = [](float a, float b) { return __builtin_convertvector(f2v_t{a, b}, bf2v_t); };
    auto lo = [](float a, float b, bf2v_t hb) {
        return __builtin_convertvector(f2v_t{a, b} - __builtin_convertvector(hb, f2v_t), bf2v_t);
    };
    const bf2v_t h0 = hi(x[0], x[1]), h1 = hi(x[2], x[3]), h2 = hi(y[0], y[1]), h3 = hi(y[2], y[3]);
    const bf2v_t l0 = lo(x[0], x[1], h0), l1 = lo(x[2], x[3], h1), l2 = lo(y[0], y[1], h2), l3 = lo(y[2], y[3], h3);
    h = v4u_t{__builtin_bit_cast(unsigned int, h0), __builtin_bit_cast(unsigned int, h1),
              __builtin_bit_cast(unsigned int, h2), __builtin_bit_cast(unsigned int, h3)};
    l = v4u_t{__builtin_bit_cast(unsigned int, l0), __builtin_bit_cast(unsigned int, l1),
              __builtin_bit_cast(unsigned int, l2), __builtin_bit_cast(unsigned int, l3)};
}

// =====================================================================================
// Half-transform, 3-term BF16 split: X = Bh Ch + Bh Cl + Bl Ch with FP32 accumulation.
// B is read from its FP32 copies and split into hi/lo in registers before the LDS store (the
// same 4 bytes per element as stored hi/lo copies); a block used in the transposed
// orientation is read from the tile-transposed FP32 copy, so every A vector is a 32-byte
// row segment.
// C transposed ([ldc][nbfp], k contiguous) hi/lo.  K-step = one column tile (32).  WM x WN
// waves, workgroup tile 64*WM rows x 16*NBW*WN columns (WN = 4: one 8-wave workgroup per CU;
// WN = 2: two 4-wave workgroups per CU, whose barriers are independent).  DC: the C panel
// goes global -> LDS by direct loads (no staging registers, no LDS store instructions)
// instead of through registers.  Output X split again into hi/lo BF16 ([nq][xrows][ldc]).
// =====================================================================================
// s_waitcnt immediate (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
// that waits until at most n vector-memory operations of this wave are outstanding
constexpr int wait_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
__device__ inline void fence_compiler() { __asm__ __volatile__("" ::: "memory"); }
// (the target builtins below exist only in the device pass; the host pass of a kernel
// template that calls them directly would drop the kernel's launch stub)
template <int N>
__device__ inline void wait_vmem() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_s_waitcnt(wait_vm(N));
#endif
}
// Workgroup barrier that publishes this wave's LDS stores and the direct loads older than its n
// youngest vector-memory operations, and leaves those n in flight (__syncthreads waits for all).
template <int N>
__device__ inline void barrier_vmem() {
    fence_compiler();
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_s_waitcnt(wait_vm(N) & ~0x0F00);
    __builtin_amdgcn_s_barrier();
#endif
    fence_compiler();
}
template <int P>
__device__ inline void set_priority() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_s_setprio(P);
#endif
}
// 16 bytes per lane from global memory straight into LDS: lane L of the wave writes
// lds + 16 L bytes (lds is wave-uniform)
__device__ inline void load_lds16(const uint16_t* src, uint16_t* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(src), lds, 16, 0, 0);
#endif
}

template <int NBW, int WM, int WN, bool DC>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_ht_bf3(const float* __restrict__ B,
                                                     const float* __restrict__ BT,
                                                     const int* __restrict__ tidx, int nT, int ntp, int q0, int nq,
                                                     int npanel, const uint16_t* __restrict__ CTh,
                                                     const uint16_t* __restrict__ CTl,
                                                     int nbfp, int ldc, uint16_t* __restrict__ Xh,
                                                     uint16_t* __restrict__ Xl, int xrows,
                                                     const float* __restrict__ ztile) {
    constexpr int NTHR = WM * WN * 64;
    constexpr int RT = 2 * WM;
    constexpr int ROWS = 64 * WM;
    constexpr int PAN = 16 * NBW * WN;
    constexpr int A_SZ = ROWS * 32;          // swizzled 64-byte rows (kg_swz)
    constexpr int C_SZ = PAN * 32;
    constexpr int NAV = ROWS * 4 / NTHR;     // 16-byte A vectors per thread per array
    constexpr int NCV = PAN * 4 / NTHR;      // full rounds of 16-byte C vectors per thread per array
    constexpr int NCV_R = (PAN * 4) % NTHR;  // vectors in the last partial round
    static_assert((NAV == 1 || NAV == 2) && NAV * NTHR == ROWS * 4, "one or two A vectors per thread");
    static_assert(NCV + (NCV_R ? 1 : 0) <= 5, "C staging slots");
    static_assert(NCV_R % 4 == 0, "whole C rows per partial round");
    static_assert(NTHR >= kMaxColTiles, "build_steps takes one thread per column tile");
    constexpr int NSLOT = NCV + (NCV_R ? 1 : 0);  // C vector rounds per thread
    // the two stage buffers are separate arrays, so the compiler can tell a direct load into
    // one from the fragment reads of the other and need not wait for it before them
    __shared__ __align__(16) uint16_t Ls0[2 * A_SZ + 2 * C_SZ];
    __shared__ __align__(16) uint16_t Ls1[2 * A_SZ + 2 * C_SZ];
    auto lbuf = [&](int buf) { return buf ? Ls1 : Ls0; };
    __shared__ StepList<RT> sl;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int nrb = xrows / ROWS;
    const XcdItem xi = xcd_map(blockIdx.x, nrb * npanel, nq);
    if (!xi.valid) return;
    const int rb = xi.item / npanel;
    const int I0 = RT * rb;
    const int q = xi.group;
    const int col0 = (xi.item % npanel) * PAN;
    const size_t qoff = static_cast<size_t>(q0 + q) * ntp * TILE2;

    build_steps<RT>(sl, tidx, nT, I0, tid);
    const int nsteps = sl.n;

    f4_t acc[4][NBW];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NBW; ++j) acc[i][j] = f4_t{0, 0, 0, 0};

    // A: per row tile 32x32 = 128 vectors of 8; RT row tiles -> NAV vectors per thread per
    // array, vector v = tid + NTHR * n in row tile v >> 7.
    // Staging registers.  The A vectors (B_Q blocks, streamed from HBM) are loaded two steps
    // before their LDS store, in two sets; the C vectors (a panel every workgroup re-reads,
    // mostly L2 hits) one step before, either into registers (C loads issued first in the
    // step, so the store's wait for them leaves the younger A loads in flight) or, with DC,
    // straight into the other LDS buffer (then the step's closing wait for the direct loads
    // waits for every vector-memory load, and the A loads have one step to land).
    typedef v4u_t v4u;
    v4f_t a0[2 * NAV], a1[2 * NAV];  // 8 FP32 of one A row segment per vector, per set
    v4u c0h, c0l, c1h, c1l, c2h, c2l, c3h, c3l, c4h, c4l;
    // column tile of step st; steps past the end re-read the last one (their data is never used)
    auto jof = [&](int st) { return sl.J[min(st, nsteps - 1)]; };
    // direct C loads: the panel's 16-row groups (PAN/16 per array, hi then lo) are dealt to
    // the waves; a load writes 16 rows of 64 bytes, lane L into 16-byte slot L, so lane L
    // fetches the logical chunk that the swizzle of kg_swz places in that slot
    constexpr int NWAVE = WM * WN;
    constexpr int NRG = PAN / 16;
    constexpr int NLD = 2 * NRG / NWAVE;
    static_assert(!DC || NLD * NWAVE == 2 * NRG, "whole direct loads per wave");
    const int w = __builtin_amdgcn_readfirstlane(wave);
    const uint16_t* csrc[NLD];  // wave-uniform: the group's first row
    int cdst[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int idx = w + NWAVE * i, arr = idx / NRG, rg = idx % NRG;
        csrc[i] = (arr ? CTl : CTh) + static_cast<size_t>(col0 + rg * 16) * nbfp;
        cdst[i] = 2 * A_SZ + arr * C_SZ + rg * 512;
    }
    const unsigned coff = ((lane >> 2) * nbfp + 8 * ((lane & 3) ^ ((lane >> 3) & 3))) * 2;  // bytes
    auto issueC = [&](int J, int buf) {
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            load_lds16(reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(csrc[i] + J * TILE) + coff),
                       lbuf(buf) + cdst[i]);
    };
    // vector f = v & 127 covers row (f>>2) of its row tile's block, k = 8*(f&3)..+7.  The block's tile
    // and offset are wave-uniform.  A block stored as (J, I) (below the diagonal) is read from the
    // tile-transposed copy, so the vector is always a row segment of this row tile's block.
    const unsigned aoff = ((tid & 127) >> 2) * TILE * 4 + 32 * (tid & 3);  // bytes
    auto gloadA_at = [&](int J, const int* off, v4f_t(&a)[2 * NAV]) {
#pragma unroll
        for (int n = 0; n < NAV; ++n) {
            const int sub = (w * 64 + NTHR * n) >> 7;
            const float* t = off[n] >= 0 ? (I0 + sub > J ? BT : B) + qoff + off[n] : ztile;
            const char* t8 = reinterpret_cast<const char*>(t) + aoff;
            a[2 * n] = *reinterpret_cast<const v4f_t*>(t8);
            a[2 * n + 1] = *reinterpret_cast<const v4f_t*>(t8 + 16);
        }
    };
    auto offs = [&](int st, int* off) {
#pragma unroll
        for (int n = 0; n < NAV; ++n)
            off[n] = __builtin_amdgcn_readfirstlane(sl.soff[min(st, nsteps - 1) * RT + ((w * 64 + NTHR * n) >> 7)]);
    };
    auto gloadA = [&](int st, v4f_t(&a)[2 * NAV]) {
        int off[NAV];
        offs(st, off);
        gloadA_at(__builtin_amdgcn_readfirstlane(jof(st)), off, a);
    };
    // the A vectors split into hi/lo (done while the previous step's MFMAs run)
    v4u_t sah[NAV], sal[NAV];
    auto splitA = [&](const v4f_t(&a)[2 * NAV]) {
#pragma unroll
        for (int n = 0; n < NAV; ++n) split_bf16x8(a[2 * n], a[2 * n + 1], sah[n], sal[n]);
    };
    auto gloadC = [&](int st) {
        const size_t kb = static_cast<size_t>(jof(st)) * TILE;
        // every lane loads (idle lanes of the partial round re-read the last vector and do
        // not store it), so every step issues the same loads
        auto cload = [&](int it, v4u& h, v4u& l) {
            const int v = min(tid + NTHR * it, PAN * 4 - 1);
            const int col = v >> 2, k8 = 8 * (v & 3);
            const size_t co = static_cast<size_t>(col0 + col) * nbfp + kb + k8;
            h = *reinterpret_cast<const v4u*>(CTh + co);
            l = *reinterpret_cast<const v4u*>(CTl + co);
        };
        if constexpr (DC) return;
        if (NSLOT > 0) cload(0, c0h, c0l);
        if (NSLOT > 1) cload(1, c1h, c1l);
        if (NSLOT > 2) cload(2, c2h, c2l);
        if (NSLOT > 3) cload(3, c3h, c3l);
        if (NSLOT > 4) cload(4, c4h, c4l);
    };
    auto lstore = [&](int buf) {
        uint16_t* Ah = lbuf(buf);
        uint16_t* Al = Ah + A_SZ;
        uint16_t* Ch = Al + A_SZ;
        uint16_t* Cl = Ch + C_SZ;
#pragma unroll
        for (int n = 0; n < NAV; ++n) {
            const int v = tid + NTHR * n, f = v & 127;
            const int ao = kg_swz((v >> 7) * 32 + (f >> 2), f & 3);
            *reinterpret_cast<v4u*>(Ah + ao) = sah[n];
            *reinterpret_cast<v4u*>(Al + ao) = sal[n];
        }
        // every loaded value has an unconditional use, so the loads stay where they are issued:
        // lanes past the end of the partial round loaded the last vector and store it again
        // to the same place (the same bytes as its own lane's store)
        auto cstore = [&](int it, const v4u& h, const v4u& l) {
            const int v = min(tid + NTHR * it, PAN * 4 - 1);
            const int o = kg_swz(v >> 2, v & 3);
            *reinterpret_cast<v4u*>(Ch + o) = h;
            *reinterpret_cast<v4u*>(Cl + o) = l;
        };
        if constexpr (DC) return;
        if (NSLOT > 0) cstore(0, c0h, c0l);
        if (NSLOT > 1) cstore(1, c1h, c1l);
        if (NSLOT > 2) cstore(2, c2h, c2l);
        if (NSLOT > 3) cstore(3, c3h, c3l);
        if (NSLOT > 4) cstore(4, c4h, c4l);
    };
    // One step's products, column block by column block: the A fragments and the first C fragments are
    // read first, then each block's C fragments while the block before it is multiplied, so the LDS
    // reads of a step are spread over its MFMAs (an accumulator's three updates are 4 MFMAs apart).  pre
    // (the next steps' operands) runs after the first block's MFMAs are issued.
    // A wave whose 16-row fragments lie past the last row tile (last row block only) skips
    // their fragment reads and MFMAs; their accumulators stay zero.
    const int nfr = __builtin_amdgcn_readfirstlane(min(4, max(0, 2 * (nT - I0 - 2 * wm))));
    auto compute = [&](int buf, auto ni, auto&& pre) {
        constexpr int NI = decltype(ni)::value;
        const uint16_t* Ah = lbuf(buf);
        const uint16_t* Al = Ah + A_SZ;
        const uint16_t* Ch = Al + A_SZ;
        const uint16_t* Cl = Ch + C_SZ;
        const int fc = lane >> 4;
        bf8_t ah[4], al[4], bh[2], bl[2];
        auto frag = [&](const uint16_t* L, int row) {
            return __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + kg_swz(row + (lane & 15), fc)));
        };
        auto cread = [&](int j) {
            bh[j & 1] = frag(Ch, wn * NBW * 16 + j * 16);
            bl[j & 1] = frag(Cl, wn * NBW * 16 + j * 16);
        };
#pragma unroll
        for (int i = 0; i < NI; ++i) ah[i] = frag(Ah, wm * 64 + i * 16);
        if constexpr (NI > 0) cread(0);
#pragma unroll
        for (int i = 0; i < NI; ++i) al[i] = frag(Al, wm * 64 + i * 16);
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            if constexpr (NI > 0)
                if (j + 1 < NBW) cread(j + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j & 1], ah[i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[j & 1], ah[i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j & 1], al[i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (j == 0) {
                pre();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Steps run in pairs so the two A sets are named statically; the loop body has no
    // branches around its loads and stores (loads past the last step re-read it, and their
    // stores land in a buffer no later compute reads).
    auto mainloop = [&](auto ni) {
        // Staged C: the step's C and A loads are issued before its fragment reads.  Direct C: the A
        // vectors that arrived are split and stored to the other buffer, then the next step's C goes
        // there (a store that follows a direct load to its buffer would wait for it), then the A loads
        // of the step after next; the wait that closes the step leaves those in flight, so a block of
        // B has two steps to arrive from HBM.  The tiles and offsets of those loads are looked up a
        // step ahead.
        int J1 = 0, J2 = 0, off2[NAV] = {};
        auto half = [&](int cur, int st, v4f_t(&have)[2 * NAV], v4f_t(&next)[2 * NAV]) {
            if constexpr (DC) {
                const int jn = sl.J[min(st + 3, nsteps - 1)];
                int on[NAV];
#pragma unroll
                for (int n = 0; n < NAV; ++n) on[n] = sl.soff[min(st + 3, nsteps - 1) * RT + ((w * 64 + NTHR * n) >> 7)];
                compute(cur, ni, [&] {
                    splitA(have);
                    lstore(cur ^ 1);
                    __builtin_amdgcn_sched_barrier(0);
                    issueC(J1, cur ^ 1);
                    fence_compiler();
                    __builtin_amdgcn_sched_barrier(0);
                    gloadA_at(J2, off2, next);
                });
                J1 = J2;
                J2 = __builtin_amdgcn_readfirstlane(jn);
#pragma unroll
                for (int n = 0; n < NAV; ++n) off2[n] = __builtin_amdgcn_readfirstlane(on[n]);
                barrier_vmem<2 * NAV>();
            } else {
                gloadC(st + 1);
                gloadA(st + 2, next);
                __builtin_amdgcn_sched_barrier(0);
                compute(cur, ni, [&] { splitA(have); });
                lstore(cur ^ 1);
                __syncthreads();
            }
        };
        if constexpr (DC) {
            issueC(__builtin_amdgcn_readfirstlane(jof(0)), 0);
            fence_compiler();
        } else {
            gloadC(0);
        }
        gloadA(0, a0);
        splitA(a0);
        lstore(0);
        gloadA(1, a1);
        J1 = __builtin_amdgcn_readfirstlane(jof(1));
        J2 = __builtin_amdgcn_readfirstlane(jof(2));
        offs(2, off2);
        if constexpr (DC) wait_vmem<0>();
        __syncthreads();
        int st = 0;
        for (; st + 1 < nsteps; st += 2) {
            half(0, st, a1, a0);
            half(1, st + 1, a0, a1);
        }
        if (st < nsteps) compute(0, ni, [] {});  // odd step count: the last step is in buffer 0
        // direct loads still in flight (steps past the end) land before the LDS is released
        if constexpr (DC) wait_vmem<0>();
    };
    // The 8-wave shape.  With all waves at the same point of a step, the fragment reads, the split and
    // the barrier (1870 of 3790 cycles per step at nbf 1500) left the MFMA pipes idle: 50 % busy, 8.49 ms
    // per 1000 Q at 600 columns.  Taking turns keeps them 62 % busy and takes 7.45 ms, now against the
    // power limit (the clock falls from 1.97 to 1.78 GHz; MFMAs alone on random data reach 2113 TFLOP/s).
    // Two groups of four waves (one wave per SIMD each) take turns: while one group multiplies a step
    // whose fragments it holds in registers, the other reads its fragments of a step from LDS, splits and
    // stores A and starts its loads.  Slots are separated by barriers; group 0 reads step s in slot 2s
    // and multiplies it in slot 2s + 1, group 1 one slot later.  The buffer of step s + 1 was last
    // read in slot 2s - 1 and is first read in slot 2s + 2: both groups start their direct loads to
    // it in slot 2s (group 0 while reading, group 1 before multiplying) and have waited for them
    // by the end of slot 2s + 1.
    auto mainloop_pp = [&](auto ni, auto grp) {
        constexpr int NI = decltype(ni)::value;
        constexpr bool G1 = decltype(grp)::value;
        bf8_t ah[4], al[4], bh[NBW], bl[NBW];
        const int fc = lane >> 4;
        auto frags = [&](int buf) {
            const uint16_t* Ah = lbuf(buf);
            const uint16_t* Al = Ah + A_SZ;
            const uint16_t* Ch = Al + A_SZ;
            const uint16_t* Cl = Ch + C_SZ;
            auto frag = [&](const uint16_t* L, int row) {
                return __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + kg_swz(row + (lane & 15), fc)));
            };
            if constexpr (NI > 0) {
#pragma unroll
                for (int i = 0; i < NI; ++i) ah[i] = frag(Ah, wm * 64 + i * 16);
#pragma unroll
                for (int j = 0; j < NBW; ++j) bh[j] = frag(Ch, wn * NBW * 16 + j * 16);
#pragma unroll
                for (int j = 0; j < NBW; ++j) bl[j] = frag(Cl, wn * NBW * 16 + j * 16);
#pragma unroll
                for (int i = 0; i < NI; ++i) al[i] = frag(Al, wm * 64 + i * 16);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto mul = [&] {
            __builtin_amdgcn_sched_barrier(0);
            set_priority<1>();
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j], ah[i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[j], ah[i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j], al[i], acc[i][j], 0, 0, 0);
            set_priority<0>();
            __builtin_amdgcn_sched_barrier(0);
        };
        // tiles and offsets of the loads, looked up a step ahead: J1 = tile of step s + 1 (group 1's
        // multiply phase: s + 2), J2 and off2 of step s + 2
        int J1, J2, off2[NAV];
        issueC(__builtin_amdgcn_readfirstlane(jof(0)), 0);
        fence_compiler();
        gloadA(0, a0);
        splitA(a0);
        lstore(0);
        gloadA(1, a1);
        J1 = __builtin_amdgcn_readfirstlane(jof(1));
        J2 = __builtin_amdgcn_readfirstlane(jof(2));
        offs(2, off2);
        wait_vmem<0>();
        __syncthreads();
        auto read_phase = [&](int cur, int st, v4f_t(&have)[2 * NAV], v4f_t(&next)[2 * NAV]) {
            const int jn = sl.J[min(st + 3, nsteps - 1)];
            int on[NAV];
#pragma unroll
            for (int n = 0; n < NAV; ++n) on[n] = sl.soff[min(st + 3, nsteps - 1) * RT + ((w * 64 + NTHR * n) >> 7)];
            frags(cur);
            splitA(have);
            lstore(cur ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!G1) {
                issueC(J1, cur ^ 1);
                fence_compiler();
                __builtin_amdgcn_sched_barrier(0);
            }
            gloadA_at(J2, off2, next);
            __builtin_amdgcn_sched_barrier(0);
            J1 = J2;
            J2 = __builtin_amdgcn_readfirstlane(jn);
#pragma unroll
            for (int n = 0; n < NAV; ++n) off2[n] = __builtin_amdgcn_readfirstlane(on[n]);
            // group 1's direct loads to the other buffer (started a slot ago) have landed; group 0's
            // have another slot
            barrier_vmem < G1 ? 2 * NAV : 63 > ();
        };
        auto mul_phase = [&](int cur, bool last) {
            if constexpr (G1) {
                // J1 is already the tile of step st + 2, whose buffer is the one just read
                issueC(J1, cur);
                fence_compiler();
            }
            mul();
            if (!last) barrier_vmem < G1 ? 63 : 2 * NAV > ();
        };
        if constexpr (G1) {
            issueC(J1, 1);
            fence_compiler();
            barrier_vmem<63>();
        }
        int st = 0;
        for (; st + 1 < nsteps; st += 2) {
            read_phase(0, st, a1, a0);
            mul_phase(0, false);
            read_phase(1, st + 1, a0, a1);
            mul_phase(1, G1 && st + 2 >= nsteps);
        }
        if (st < nsteps) {
            read_phase(0, st, a1, a0);
            mul_phase(0, G1);
        }
        wait_vmem<0>();  // direct loads of steps past the end land before the LDS is released
    };
    if (nsteps > 0) {
        auto go = [&](auto ni) {
            if constexpr (DC && NWAVE == 8) {
                if (w < 4)
                    mainloop_pp(ni, std::false_type{});
                else
                    mainloop_pp(ni, std::true_type{});
            } else {
                mainloop(ni);
            }
        };
        if (nfr == 4)
            go(std::integral_constant<int, 4>{});
        else if (nfr == 2)
            go(std::integral_constant<int, 2>{});
        else
            go(std::integral_constant<int, 0>{});
    }
    // X in fragment order (ht_bf3 above): the MFMAs formed C^T B_Q, so a lane holds row lane % 16 and four
    // consecutive columns of X, 8 bytes of a 1 KB block
    const size_t xq = static_cast<size_t>(q) * xrows * ldc;
    const int nk32 = ldc / 32, xlane = ((lane >> 5) * 16 + (lane & 15)) * 8 + 4 * ((lane >> 4) & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const int r16 = ROWS / 16 * rb + wm * 4 + i, c16 = col0 / 16 + wn * NBW + j;
            const size_t o = xq + (static_cast<size_t>(r16) * nk32 + (c16 >> 1)) * 512 + (c16 & 1) * 256 + xlane;
            const v4f_t x = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            const bf4v_t hi = __builtin_convertvector(x, bf4v_t);
            *reinterpret_cast<bf4v_t*>(Xh + o) = hi;
            *reinterpret_cast<bf4v_t*>(Xl + o) = __builtin_convertvector(x - __builtin_convertvector(hi, v4f_t), bf4v_t);
        }
}

// =====================================================================================
// K contraction, 3-term BF16 split on hi/lo X: A S B^T ~ Ah Bh + Ah Bl + Al Bh.
// 128x128 tiles, 4 waves of 64x64, K-step 32, double-buffered LDS.  X comes in fragment order, 16 rows x 32
// columns in 1 KB, so a staging load is one contiguous KB (whole cache lines; rows of X of 64 bytes
// a step took twice the L2 requests), and a fragment is read from LDS as it lies there, free of bank
// conflicts.  64 KB of LDS leave room for two workgroups per CU.  Naux 1000 / nbf 1500, every block over 304
// columns: 3.92 ms, 1.16 PFLOP/s, 57 % of the cycles busy at 1.95 GHz (rows of X: 4.58 ms): like the
// half-transform against the power limit.  Loads two steps ahead (a barrier between the fragment reads and
// the MFMAs) were no faster: 3.9-4.1 ms.
// The MFMA accumulators are folded into a second set of FP32 totals every kFold32 k-terms
// (FP64 totals would not fit beside the fragments in 256 registers): a sum of N terms then
// rounds like two chains of about sqrt(N) additions instead of one chain of N.
// DC: the operands go from global memory straight into LDS (global_load_lds_dwordx4, each
// wave 8 loads of 16 rows per step, issued after the step's fragment reads) instead of
// through staging registers.
// =====================================================================================

template <bool DC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_kgemm_bf3(
    const uint16_t* __restrict__ Ah_, const uint16_t* __restrict__ Al_, const uint16_t* __restrict__ Bh_,
    const uint16_t* __restrict__ Bl_, size_t stride, int ld, int kbeg, int kend, int nbatch, int nsplit,
    const int2* __restrict__ tiles, int ntile, double* __restrict__ P, double alpha, int accumulate, int upper,
    int nvalid) {
    constexpr int KS = 32, SZ = 128 * 32;
    __shared__ __align__(16) uint16_t Ls0[4 * SZ];
    __shared__ __align__(16) uint16_t Ls1[4 * SZ];
    auto lbuf = [&](int b) { return b ? Ls1 : Ls0; };
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const XcdItem xi = xcd_map(blockIdx.x, ntile, nsplit);
    if (!xi.valid) return;
    const int tile = xi.item, split = xi.group;
    const int2 tb = tiles[tile];
    // no MFMAs for the wave below the diagonal of a diagonal tile of a symmetric result, or
    // for one entirely in the zero padding rows / columns of X past nvalid
    const bool idle = (upper && tb.x == tb.y && wr > wc) || tb.x * 128 + wr * 64 >= nvalid ||
                      tb.y * 128 + wc * 64 >= nvalid;
    const int m0 = tb.x * 128, n0 = tb.y * 128;
    const int b0 = static_cast<int>((static_cast<long long>(nbatch) * split) / nsplit);
    const int b1 = static_cast<int>((static_cast<long long>(nbatch) * (split + 1)) / nsplit);
    const int nks = (kend - kbeg) / KS;
    const int nsteps = (b1 - b0) * nks;

    f4_t acc[16], tot[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        acc[i] = f4_t{0, 0, 0, 0};
        tot[i] = f4_t{0, 0, 0, 0};
    }
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            tot[i] += acc[i];
            acc[i] = f4_t{0, 0, 0, 0};
        }
    };

    // per step: 4 arrays x 8 blocks of 16 rows x 32 k; a thread's two 16-byte vectors per array lie in
    // blocks tid / 64 and tid / 64 + 4
    const int nk32 = ld / 32;
    auto block = [&](const uint16_t* X, int s, int r16) {
        return X + static_cast<size_t>(b0 + s / nks) * stride +
               (static_cast<size_t>(r16) * nk32 + kbeg / 32 + s % nks) * 512 + lane * 8;
    };
    const int w = __builtin_amdgcn_readfirstlane(wave);
    uint4 a0h, a0l, b0h, b0l, a1h, a1l, b1h, b1l;
    auto gload = [&](int s) {
        auto ld16 = [&](const uint16_t* X, int r16) { return *reinterpret_cast<const uint4*>(block(X, s, r16)); };
        a0h = ld16(Ah_, m0 / 16 + w);
        a0l = ld16(Al_, m0 / 16 + w);
        a1h = ld16(Ah_, m0 / 16 + w + 4);
        a1l = ld16(Al_, m0 / 16 + w + 4);
        b0h = ld16(Bh_, n0 / 16 + w);
        b0l = ld16(Bl_, n0 / 16 + w);
        b1h = ld16(Bh_, n0 / 16 + w + 4);
        b1l = ld16(Bl_, n0 / 16 + w + 4);
    };
    const int o0 = tid * 8, o1 = o0 + 2048;
    auto lstore = [&](int buf) {
        uint16_t* L = lbuf(buf);
        *reinterpret_cast<uint4*>(L + o0) = a0h;
        *reinterpret_cast<uint4*>(L + SZ + o0) = a0l;
        *reinterpret_cast<uint4*>(L + 2 * SZ + o0) = b0h;
        *reinterpret_cast<uint4*>(L + 3 * SZ + o0) = b0l;
        *reinterpret_cast<uint4*>(L + o1) = a1h;
        *reinterpret_cast<uint4*>(L + SZ + o1) = a1l;
        *reinterpret_cast<uint4*>(L + 2 * SZ + o1) = b1h;
        *reinterpret_cast<uint4*>(L + 3 * SZ + o1) = b1l;
    };
    // direct loads of step s into buf: the 32 blocks (Ah, Al, Bh, Bl x 8) are dealt to the waves
    auto issue = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int arr = i >> 1, rg = w + 4 * (i & 1);
            const uint16_t* X = arr == 0 ? Ah_ : arr == 1 ? Al_ : arr == 2 ? Bh_ : Bl_;
            load_lds16(block(X, s, (arr < 2 ? m0 : n0) / 16 + rg), lbuf(buf) + arr * SZ + rg * 512);
        }
    };
    bf8_t ah[4], al[4], bh[4], bl[4];
    auto read = [&](const uint16_t* L) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ra = (wr * 4 + i) * 512 + lane * 8, rb = (wc * 4 + i) * 512 + lane * 8;
            ah[i] = __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + ra));
            al[i] = __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + SZ + ra));
            bh[i] = __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + 2 * SZ + rb));
            bl[i] = __builtin_bit_cast(bf8_t, *reinterpret_cast<const uint4*>(L + 3 * SZ + rb));
        }
    };
    int nf = 0;
    auto mul = [&] {
        auto term = [&](const bf8_t* a, const bf8_t* b) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[i * 4 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i * 4 + j], 0, 0, 0);
        };
        term(ah, bh);
        term(ah, bl);
        term(al, bh);
        if (++nf == kFold32 / KS) {
            fold();
            nf = 0;
        }
    };

    if (nsteps > 0) {
        if constexpr (DC) {
            issue(0, 0);
            wait_vmem<0>();
        } else {
            gload(0);
            lstore(0);
        }
        __syncthreads();
        int buf = 0;
        for (int st = 0; st < nsteps; ++st) {
            const bool more = st + 1 < nsteps;
            if constexpr (!DC)
                if (more) gload(st + 1);
            if (!idle) read(lbuf(buf));
            if constexpr (DC) {
                __builtin_amdgcn_sched_barrier(0);
                if (more) issue(st + 1, buf ^ 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!idle) mul();
            if constexpr (DC)
                wait_vmem<0>();
            else if (more)
                lstore(buf ^ 1);
            __syncthreads();
            buf ^= 1;
        }
    }
    if (idle) return;
    fold();
    double* Pt = P + (static_cast<size_t>(split) * ntile + tile) * 16384;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int row = wr * 64 + i * 16 + 4 * (lane >> 4) + rr;
                const int col = wc * 64 + j * 16 + (lane & 15);
                double* o = Pt + row * 128 + col;
                *o = alpha * static_cast<double>(tot[i * 4 + j][rr]) + (accumulate ? *o : 0.0);
            }
}

// ------------------------------------------------------------------ conversions
__global__ void k_to_f32(const double* __restrict__ src, float* __restrict__ dst, size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        dst[i] = static_cast<float>(src[i]);
}
// FP32 with each 32x32 tile transposed, dstT[t][r][c] = src[t][c][r] (the half-transform reads these
// for the blocks it uses in the transposed orientation), and with dst the plain FP32 copy too, from one
// read of src.  The tile is turned in LDS, so both sides move whole lines: bound by HBM, 3.9 GB in 1.6
// ms with both copies (apart 1.0 + 1.55, the transposed one reading every line twice).
__global__ __launch_bounds__(256) void k_to_f32_t(const double* __restrict__ src, float* __restrict__ dst,
                                                  float* __restrict__ dstT, size_t ntile) {
    __shared__ float T[TILE][TILE + 1];
    const int r = threadIdx.x >> 3, c = 4 * (threadIdx.x & 7);
    for (size_t t = blockIdx.x; t < ntile; t += gridDim.x) {
        const size_t o = t * TILE2 + 4 * threadIdx.x;
        const double2 a = *reinterpret_cast<const double2*>(src + o), b = *reinterpret_cast<const double2*>(src + o + 2);
        const v4f_t v = {static_cast<float>(a.x), static_cast<float>(a.y), static_cast<float>(b.x),
                         static_cast<float>(b.y)};
        if (dst) *reinterpret_cast<v4f_t*>(dst + o) = v;
        __syncthreads();  // the tile before has been read
#pragma unroll
        for (int k = 0; k < 4; ++k) T[r][c + k] = v[k];
        __syncthreads();
        *reinterpret_cast<v4f_t*>(dstT + o) = v4f_t{T[c][r], T[c + 1][r], T[c + 2][r], T[c + 3][r]};
    }
}

// C [nbf][ld] FP64 -> transposed padded [ldc][nbfp] BF16 hi/lo, with the column map
__global__ void k_pack_cT_bf(const double* __restrict__ src, int ldsrc, int nbf, const int* __restrict__ cmap,
                             uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, int nbfp, int ldc) {
    const size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<size_t>(nbfp) * ldc) return;
    const int c = static_cast<int>(idx / nbfp), m = static_cast<int>(idx % nbfp);
    const int i = cmap[c];
    const float x = (m < nbf && i >= 0) ? static_cast<float>(src[static_cast<size_t>(m) * ldsrc + i]) : 0.0f;
    const uint16_t h = f2bf(x);
    hi[idx] = h;
    lo[idx] = f2bf(x - bf2f(h));
}

// Column signs: s[i] = +1 if Cr[:,i] == Cl[:,i], -1 if Cr[:,i] == -Cl[:,i], 0 otherwise
// (only bitwise-exact matches count).  One block per column.
// s[i] = +1 / -1 when column i of Cr is bitwise +/- column (i + shift) % ncol of Cl, else 0.
__global__ void k_column_signs(const double* __restrict__ Cl, const double* __restrict__ Cr, int ld, int nbf,
                               int ncol, int shift, int8_t* __restrict__ s) {
    const int i = blockIdx.x;
    const int il = (i + shift) % ncol;
    __shared__ int plus, minus;
    if (threadIdx.x == 0) {
        plus = 1;
        minus = 1;
    }
    __syncthreads();
    int p = 1, mi = 1;
    for (int m = threadIdx.x; m < nbf; m += blockDim.x) {
        const double a = Cl[static_cast<size_t>(m) * ld + il], b = Cr[static_cast<size_t>(m) * ld + i];
        p &= (a == b);
        mi &= (a == -b);
    }
    if (!p) atomicAnd(&plus, 0);
    if (!mi) atomicAnd(&minus, 0);
    __syncthreads();
    if (threadIdx.x == 0) s[i] = plus ? 1 : (minus ? -1 : 0);
}

inline unsigned nblocks(size_t n, int bs) {
    const size_t b = (n + bs - 1) / bs;
    return static_cast<unsigned>(b > 65535u * 16 ? 65535u * 16 : b);
}

}  // namespace

// ------------------------------------------------------------------ launchers
void ht_panel_shape(int ncol, int* nbw, int* npanel, int* ldc) {
    const int nbt = (ncol + 63) / 64;  // 64-column units
    const int np = (nbt + 4) / 5;
    const int w = (nbt + np - 1) / np;
    *nbw = w;
    *npanel = np;
    *ldc = np * 64 * w;
}

int g_ht_wm = 0;       // 0: default shape; 1, 3, 4 select others (tuning sweeps)
void set_ht_rowwaves(int wm) { g_ht_wm = (wm >= 1 && wm <= 4) ? wm : 0; }
int g_kgemm_dc = 1;    // BF16x3 contraction: operands loaded straight into LDS (1) or staged (0)
void set_kgemm_direct(int on) { g_kgemm_dc = on ? 1 : 0; }

// npanel counts panels of 64*nbw columns; the WN = 2 shape covers each with two workgroups
template <int WM, int WN, bool DC>
static void ht_bf3_wm(const TileGeom& g, const float* B, const float* BT, int q0, int nq, const uint16_t* CTh, const uint16_t* CTl,
                      int ldc, int nbw, int npanel, uint16_t* Xh, uint16_t* Xl, int xrows, const void* zt,
                      hipStream_t s) {
    const int np = npanel * 4 / WN;
    dim3 grid(xcd_grid(nq, xrows / (64 * WM) * np));
    const float* z = static_cast<const float*>(zt);
    switch (nbw) {
#define P4A_BF3(n)                                                                                                  \
    case n:                                                                                                         \
        hipLaunchKernelGGL((k_ht_bf3<n, WM, WN, DC>), grid, dim3(WM * WN * 64), 0, s, B, BT, g.d_tidx, g.nT, g.ntp, q0, nq, \
                           np, CTh, CTl, g.nbfp, ldc, Xh, Xl, xrows, z);                                           \
        break;
        P4A_BF3(1) P4A_BF3(2) P4A_BF3(3) P4A_BF3(4) P4A_BF3(5)
#undef P4A_BF3
    }
}

void launch_ht_bf3(const TileGeom& g, const float* B, const float* BT, int q0, int nq, const uint16_t* CTh, const uint16_t* CTl,
                   int ldc, int nbw, int npanel, uint16_t* Xh, uint16_t* Xl, int xrows, const void* zt,
                   hipStream_t s) {
    require(nbw >= 1 && nbw <= 5 && ldc == npanel * 64 * nbw && nq > 0 && nq <= 65535 && g.nbfp % 32 == 0 &&
                xrows == (g.nT + 3) / 4 * 128 && g.nT <= kMaxColTiles && zt != nullptr,
            "ht_bf3 shape");
    // default: one 8-wave workgroup of 128 x 64*nbw per CU, C loaded straight into LDS.
    // Kept for comparison: 1 (4 waves over 64 rows), 3 (4-wave workgroups of 128 x 32*nbw,
    // two per CU: as fast, but each B block is read by twice as many workgroups, 1.3x the
    // HBM reads), 4 (the 8-wave shape with C staged through registers).
    if (g_ht_wm == 1)
        ht_bf3_wm<1, 4, false>(g, B, BT, q0, nq, CTh, CTl, ldc, nbw, npanel, Xh, Xl, xrows, zt, s);
    else if (g_ht_wm == 3)
        ht_bf3_wm<2, 2, true>(g, B, BT, q0, nq, CTh, CTl, ldc, nbw, npanel, Xh, Xl, xrows, zt, s);
    else if (g_ht_wm == 4)
        ht_bf3_wm<2, 4, false>(g, B, BT, q0, nq, CTh, CTl, ldc, nbw, npanel, Xh, Xl, xrows, zt, s);
    else
        ht_bf3_wm<2, 4, true>(g, B, BT, q0, nq, CTh, CTl, ldc, nbw, npanel, Xh, Xl, xrows, zt, s);
}

static void kgemm_check(int xrows, int ld, int kbeg, int kend, int nbatch, int nsplit, int ntile, int ks) {
    require(ntile > 0 && nsplit > 0 && nbatch >= nsplit && xrows % 128 == 0 && kbeg >= 0 && kend <= ld &&
                kbeg < kend && kbeg % ks == 0 && kend % ks == 0,
            "kgemm shape");
}

void launch_kgemm_bf3(const uint16_t* Ah, const uint16_t* Al, const uint16_t* Bh, const uint16_t* Bl, size_t stride,
                      int xrows, int nvalid, int ld, int kbeg, int kend, int nbatch, int nsplit, const int2* tiles,
                      int ntile, double* P, double alpha, int accumulate, int upper, hipStream_t s) {
    kgemm_check(xrows, ld, kbeg, kend, nbatch, nsplit, ntile, 32);
    require(nvalid > 0 && nvalid <= xrows, "kgemm valid rows");
    hipLaunchKernelGGL(g_kgemm_dc ? k_kgemm_bf3<true> : k_kgemm_bf3<false>, dim3(xcd_grid(nsplit, ntile)), dim3(256), 0, s, Ah, Al, Bh, Bl, stride, ld, kbeg,
                       kend, nbatch, nsplit, tiles, ntile, P, alpha, accumulate, upper, nvalid);
}

void launch_to_f32(const double* src, float* dst, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_to_f32, dim3(nblocks(n, 256)), dim3(256), 0, s, src, dst, n);
}
void launch_to_f32_t(const double* src, float* dst, float* dstT, size_t n, hipStream_t s) {
    require(n % TILE2 == 0, "to_f32_t");
    if (n == 0) return;
    hipLaunchKernelGGL(k_to_f32_t, dim3(static_cast<unsigned>(std::min<size_t>(n / TILE2, 8192))), dim3(256), 0, s, src,
                       dst, dstT, n / TILE2);
}
void launch_pack_cT_bf(const double* src, int ldsrc, int nbf, const int* cmap, uint16_t* hi, uint16_t* lo, int nbfp,
                       int ldc, hipStream_t s) {
    const size_t n = static_cast<size_t>(nbfp) * ldc;
    hipLaunchKernelGGL(k_pack_cT_bf, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, src, ldsrc, nbf,
                       cmap, hi, lo, nbfp, ldc);
}
void launch_column_signs(const double* Cl, const double* Cr, int ld, int nbf, int ncol, int shift, int8_t* s,
                         hipStream_t st) {
    require(ncol > 0 && ld >= ncol && shift >= 0 && shift < ncol, "column_signs");
    hipLaunchKernelGGL(k_column_signs, dim3(ncol), dim3(256), 0, st, Cl, Cr, ld, nbf, ncol, shift, s);
}

}  // namespace p4a
