// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4_f64), grouped over
// problems and segmented along K.
//
// One launch computes every output tile of every problem in its problem
// table.  A problem is C = alpha * sum_s opA(seg s) * opB(seg s)
// + beta*C, where segment s supplies its own A/B base pointers and leading
// dimensions.  A plain DGEMM is one problem with one segment; a virtual-grid
// Cannon rank is one problem whose segments are the tiles the rotations
// would have brought in; a SUMMA rank is one problem whose segments are the
// owners' panels.
//
// Three kernels share the problem/segment tables and the tile order: problems
// whose 128x128 tiles are all interior run gemm_f64_dma_ar_kernel (A straight
// into registers, B direct to LDS); the others that take direct loads run
// gemm_f64_dma_kernel (both operands direct to LDS); both are described below.
// gemm_f64_kernel takes everything else, on 128x128, 64x64 or 32x32 tiles:
// operands that direct loads do not take (odd leading dimensions, odd K),
// strips cut off uneven problems, and what it is estimated to run faster, such
// as products with few 128x128 tiles per CU (prepare_gemm chooses; a single
// problem goes to gemm_f64_one_kernel, the same code).  It stages both
// operands through registers into a double-buffered LDS; four waves a
// workgroup, each owning a quarter of the tile.
// What bounds it: the FP64 MFMA (64 cycles each, on the vector ALU's pipes).
// Measured (TFLOP/s, against the 128x128 tiles and guarded loads before):
// 512^3 3.8 -> 32.1 (32x32 tiles; 70 -> 8.4 us), 1024^3 16.6 -> 50.4, 2000^3
// 32.8 -> 65.9, 3072^3 55.3 -> 70.9, 4097^3 (odd leading dimensions) 48.6 ->
// 64.4, TN 1500 x 1333 x 2001 22.7 -> 61.8.
// Lane l of an MFMA supplies k = 2*(l/16) + q to sub-step q for both operands,
// so the product is exact whatever k order the matrix core sums in.
// The MFMA is issued as D = B^T A^T, so each output register holds 16
// consecutive rows of one C column: the epilogue stores are 128-byte runs.
// Result layout of v_mfma_f64_16x16x4_f64: lane l, register v holds
// D(l/16 + 4v, l%16) (checked on the device by the exact-integer tests).
#include <algorithm>

#include "dg_internal.hpp"
#include "staged.hpp"

namespace dg {

namespace {

typedef double dv4 __attribute__((ext_vector_type(4)));

// Global-address-space views: loads through them compile to global_load_*
// (counted by vmcnt only), not flat_load_*, whose lgkmcnt share would make
// every LDS wait also wait for the prefetch of the next k-step.
typedef __attribute__((address_space(1))) const dv2 gdv2;
__device__ __forceinline__ dv2 gld2(const double* p) { return *(gdv2*)p; }

constexpr int GROUP_M = 8;   // tile rows per raster group

// Shapes of the register-staged kernel: BM x BN output tiles of four waves,
// each owning a WM x WN sub-tile (WM/16 x WN/16 MFMA tiles of 16 x 16);
// BK-deep k-stages (a multiple of 8), D of them in flight in registers; OCC
// workgroups per CU.
template <int BM_, int BN_, int WM_, int WN_, int BK_, int D_, int OCC_>
struct TileCfg {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, BK = BK_, D = D_, OCC = OCC_;
    static constexpr int NTH = 256;
    static constexpr int WAVES_N = BN / WN;
    static constexpr int FM = WM / 16, FN = WN / 16;
    static_assert((BM / WM) * (BN / WN) * 64 == NTH, "one wave per WM x WN sub-tile");
};
// The 128x128 kernels fill their 256 VGPRs and spill 4 to 13 values of the
// code around the steady turns (the last stages' addresses, the epilogue),
// the 64x64 walks of NN two; no steady turn touches scratch.
using Cfg128 = TileCfg<128, 128, 64, 64, 16, 1, 2>;
using Cfg64 = TileCfg<64, 64, 32, 32, 16, 2, 4>;
using Cfg32 = TileCfg<32, 32, 16, 16, 32, 2, 3>;

// Block id -> tile id so that each XCD (blocks are dealt round-robin to the
// 8 XCDs) receives one contiguous range of tiles, which the grouped raster
// below turns into a compact patch of C whose A/B panels share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int total) {
    constexpr int X = 8;
    const int q = total / X, r = total % X;
    const int x = bid % X, slot = bid / X;
    return x * q + min(x, r) + slot;
}

// f[i][q] = X(row w0 + 16i + lr, k = 8h + 2lg + q) of a stage of operand O.
template <class O, bool KC, int F>
__device__ __forceinline__ void staged_fragments(double (&f)[F][2], const char* s, int w0, int lr, int lg, int h) {
#pragma unroll
    for (int i = 0; i < F; ++i) {
        if constexpr (KC) {
            const dv2 v = *reinterpret_cast<const dv2*>(s + (w0 + 16 * i + lr) * O::LROW + (8 * h + 2 * lg) * 8);
            f[i][0] = v.x;
            f[i][1] = v.y;
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                f[i][q] = *reinterpret_cast<const double*>(s + (8 * h + 2 * lg + q) * O::LROW + (w0 + 16 * i + lr) * 8);
        }
    }
}

template <class C, bool TA, bool TB>
struct TileLds {
    using OA = Staged<double, TA, C::BM, C::BK>;    // op(A) is k-contiguous when A is transposed
    using OB = Staged<double, !TB, C::BN, C::BK>;   // op(B) when B is not
    static constexpr int STAGE = OA::BYTES + OB::BYTES;
};

// Computes one output tile of problem P.  Two LDS buffers, one barrier per
// stage: while stage s is multiplied, stages s+1 .. s+D are in flight to
// registers; s+1 is stored to the other buffer and s+1+D requested among the
// MFMAs before the last part's, one memory instruction per MFMA: issued
// together they take longer than the MFMA that runs meanwhile, and a CU with
// few resident workgroups waits (one 64x64 tile per CU, K = 4096: 148 -> 122
// us; 2048^3 249 -> 241 us).
template <class C, bool TA, bool TB>
__device__ __forceinline__ void gemm_tile(const Prob& P, const Seg* __restrict__ segs, int local, char* lds) {
    constexpr int BM = C::BM, BN = C::BN, BK = C::BK, D = C::D;
    using L = TileLds<C, TA, TB>;
    using OA = typename L::OA;
    using OB = typename L::OB;

    const int tiles_m = (int)((P.m + BM - 1) / BM), tiles_n = (int)((P.n + BN - 1) / BN);
    // Grouped raster: GROUP_M tile rows sweep the tile columns together.
    const int per_group = GROUP_M * tiles_n;
    const int group = local / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = local - group * per_group;
    const int tm = __builtin_amdgcn_readfirstlane(first_m + in_group % gsize);
    const int tn = __builtin_amdgcn_readfirstlane(in_group / gsize);

    const int64_t m0 = (int64_t)tm * BM;
    const int64_t n0 = (int64_t)tn * BN;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = (wave / C::WAVES_N) * C::WM;
    const int wn = (wave % C::WAVES_N) * C::WN;
    const int lr = lane & 15;
    const int lg = lane >> 4;

    constexpr int FM = C::FM, FN = C::FN;
    dv4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = dv4{0.0, 0.0, 0.0, 0.0};

    // load cursor over the problem's segments, one stage at a time
    const int rows = (int)min(P.m - m0, (int64_t)BM), cols = (int)min(P.n - n0, (int64_t)BN);
    const bool pairs = !(P.shift & kByElements);
    // whether the last k of a segment can be read in pairs too: no pair starts
    // at a last row (or all go along k)
    const int last = (TA || rows == BM) && (!TB || cols == BN) ? 0 : 1;
    int sg = P.seg0;
    const int sg_last = P.seg0 + P.nseg - 1;
    int64_t left;  // k of the segment from the next stage on (0 or less: past the last segment)
    OA oa;
    OB ob;
    auto enter = [&]() {
        const Seg cur = segs[sg];
        left = cur.klen;
        oa.start(cur.a, cur.lda, m0, rows);
        ob.start(cur.b, cur.ldb, n0, cols);
    };
    dv2 va[D][OA::NL], vb[D][OB::NL];
    auto read = [&](int d) {
        if (left <= 0) return;
        if (pairs && left >= BK + last) {
            oa.read(va[d]);
            ob.read(vb[d]);
        } else {
            const int real = (int)min(left, (int64_t)BK);
            oa.read_last(va[d], real, rows);
            ob.read_last(vb[d], real, cols);
        }
        left -= BK;
        if (left <= 0 && sg < sg_last) {
            ++sg;
            enter();
        }
    };
    auto store = [&](char* buf, int d) {
        OA::store(buf, va[d]);
        OB::store(buf + OA::BYTES, vb[d]);
    };
    int64_t ns = 0;
    for (int x = P.seg0; x <= sg_last; ++x) ns += (segs[x].klen + BK - 1) / BK;

    enter();
#pragma unroll
    for (int d = 0; d < D; ++d) read(d);
    store(lds, 0);
    read(0);
    __syncthreads();

    // Each 8-deep part h of a stage is one step of the direct-to-LDS kernels,
    // summed in their order: lane group lg supplies k = 8h + 2lg + q to MFMA q,
    // so every element takes the same sequence of MFMAs in all FP64 kernels
    // and a problem cut between them, or run on other tiles, gives the same
    // bits (but for the sign of a sum of -0 when K leaves this kernel
    // zero-padded parts).
    // A part's fragments are read while the part before it is multiplied, the
    // first part's of stage s + 1 during the last part of stage s: the stage's
    // barrier sits before that part, when the fragments of stage s are all in
    // registers and stage s + 1 is stored.
    constexpr int H = BK / 8;
    static_assert(H % 2 == 0, "fragment set of part h: h & 1");
    double fa[2][FM][2], fb[2][FN][2];
    auto fragments = [&](const char* buf, int h) {
        staged_fragments<OA, TA>(fa[h & 1], buf, wm, lr, lg, h);
        staged_fragments<OB, !TB>(fb[h & 1], buf + OA::BYTES, wn, lr, lg, h);
    };
    auto products = [&](int h, int q) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[h & 1][j][q], fa[h & 1][i][q], acc[i][j], 0, 0, 0);
    };
    auto multiply = [&](int h, int q) {
        __builtin_amdgcn_sched_barrier(0);
        products(h, q);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int NL = OA::NL + OB::NL, NM = 2 * FM * FN;  // loads and stores of a stage, MFMAs of a part
    // Two stages a turn: s, even, in buffer 0, and s + 1; stage s + 1 waits in
    // register set (s + 1) % D.  Turns that read only whole stages of one
    // segment run without conditions.
    static_assert(D == 1 || D == 2, "the register set of an odd stage is D - 1, of an even one 0");
    char* const bufs[2] = {lds, lds + L::STAGE};
    fragments(lds, 0);
    for (int64_t s = 0; s < ns;) {
        const int64_t turns = pairs && left > 0 ? (left - last) / (2 * BK) : 0;
        auto turn = [&]() {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int nx = (u + 1) % D;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (h < H - 1) {
                        fragments(bufs[u], h + 1);
#pragma unroll
                        for (int q = h * NL / (H - 1); q < (h + 1) * NL / (H - 1); ++q) {
                            if (q < OA::NL) {
                                OA::store(bufs[u ^ 1], va[nx], q);
                                oa.read(va[nx], q);
                            } else {
                                OB::store(bufs[u ^ 1] + OA::BYTES, vb[nx], q - OA::NL);
                                ob.read(vb[nx], q - OA::NL);
                            }
                        }
                    } else {
                        oa.advance();
                        ob.advance();
                        __syncthreads();
                        __builtin_amdgcn_sched_barrier(0);
                        fragments(bufs[u ^ 1], 0);
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q) products(h, q);
                    if (h < H - 1) {
                        constexpr int R = FM + FN < NM ? FM + FN : NM;      // MFMAs that follow a fragment read
                        constexpr int W = (NL / (H - 1) + NM - 1) / NM;
#pragma unroll
                        for (int g = 0; g < R; ++g) {
                            __builtin_amdgcn_sched_group_barrier(0x100, (FM + FN) / R, 0);
                            if (R == NM) {
                                __builtin_amdgcn_sched_group_barrier(0x200, W, 0);
                                __builtin_amdgcn_sched_group_barrier(0x020, W, 0);
                            }
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        }
                        constexpr int X = NM > R ? (NL / (H - 1) + NM - R - 1) / (NM - R) : 1;
#pragma unroll
                        for (int g = R; g < NM; ++g) {
                            __builtin_amdgcn_sched_group_barrier(0x200, X, 0);
                            __builtin_amdgcn_sched_group_barrier(0x020, X, 0);
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        }
                    } else {
#pragma unroll
                        for (int g = 0; g < FM + FN; ++g) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        // the first turn apart: its waits are for whatever loads came before,
        // those of the loop for its own
        if (turns > 0) turn();
        for (int64_t i = 1; i < turns; ++i) turn();
        s += 2 * turns;
        left -= 2 * BK * turns;
        if (turns > 0 && left == 0 && sg < sg_last) {
            ++sg;
            enter();
        }
#pragma unroll
        for (int u = 0; u < 2; ++u, ++s) {
            if (s >= ns) break;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                if (h < H - 1) {
                    fragments(bufs[u], h + 1);
                } else if (s + 1 < ns) {
                    __syncthreads();
                    fragments(bufs[u ^ 1], 0);
                }
                multiply(h, 0);
                if (h == H - 2 && s + 1 < ns) {
                    store(bufs[u ^ 1], (u + 1) % D);
                    read((u + 1) % D);
                }
                multiply(h, 1);
            }
        }
    }

    // Epilogue.  Register v of lane group lg holds MFMA result row lg + 4v
    // (the f64 16x16x4 result layout), i.e.
    // acc[i][j][v] = sum for C(m0 + wm + 16i + lr, n0 + wn + 16j + lg + 4v).
    // The old values of a column block are all requested, at clamped
    // addresses, before the first is used.
    const double alpha = P.alpha, beta = P.beta;
    typedef __attribute__((address_space(1))) double gd;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        double old[FM][4];
        if (beta != 0.0) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int64_t m = m0 + wm + 16 * i + lr, n = n0 + wn + 16 * j + lg + 4 * v;
                    old[i][v] = *(gd*)(P.c + (m < P.m ? m : P.m - 1) + (n < P.n ? n : P.n - 1) * P.ldc);
                }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t m = m0 + wm + 16 * i + lr, n = n0 + wn + 16 * j + lg + 4 * v;
                double val = alpha * acc[i][j][v];
                if (beta != 0.0) val = fma(beta, old[i][v], val);
                if (m < P.m && n < P.n) *(gd*)(P.c + m + n * P.ldc) = val;
            }
    }
}

// Tiles of this workgroup when each XCD takes one contiguous range: the
// workgroups of XCD x walk its range side by side (one tile each when the grid
// has them all).
template <class F>
__device__ __forceinline__ void walk_xcd(int total_tiles, const F& run) {
    constexpr int X = 8;
    const int x = blockIdx.x % X, slot = blockIdx.x / X;
    const int q = total_tiles / X, r = total_tiles % X;
    const int first = x * q + min(x, r), count = q + (x < r ? 1 : 0);
    const int slots = gridDim.x / X + (x < (int)(gridDim.x % X) ? 1 : 0);
    for (int t = slot; t < count; t += slots) {
        run(first + t);
        __syncthreads();  // the next tile's first stage goes where this one's last may still be read
    }
}

// MODE 0: one workgroup per tile, tile = blockIdx.x (round-robin over XCDs);
// MODE 1: XCD-contiguous tile ranges (walk_xcd), a workgroup per tile or
//         fewer that walk several (xcd_grid);
// MODE 2: persistent: every workgroup takes tiles from `counter` (zeroed
//         before the launch) until the tile space is exhausted.
template <class C, bool TA, bool TB, int MODE>
__global__ __launch_bounds__(C::NTH, C::OCC) void gemm_f64_kernel(const Prob* __restrict__ probs, int nprob,
                                                                  const Seg* __restrict__ segs, int total_tiles,
                                                                  int* __restrict__ counter) {
    __shared__ __attribute__((aligned(16))) char lds[2 * TileLds<C, TA, TB>::STAGE];
    auto run = [&](int tile) {
        // Problem owning this tile: last problem with tile0 <= tile.
        int lo = 0, hi = nprob - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (probs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
        }
        const Prob P = probs[lo];
        gemm_tile<C, TA, TB>(P, segs, tile - P.tile0, lds);
    };
    if (MODE == 0) {
        const int64_t bid = blockIdx.x + (int64_t)blockIdx.y * gridDim.x;
        if (bid < total_tiles) run((int)bid);
    } else if (MODE == 1) {
        walk_xcd(total_tiles, run);
    } else {
        __shared__ int next;
        while (true) {
            __syncthreads();  // previous tile's LDS reads and `next` reads are complete
            if (threadIdx.x == 0) next = atomicAdd(counter, 1);
            __syncthreads();
            const int tile = next;
            if (tile >= total_tiles) break;
            run(tile);
        }
    }
}

// One problem of one segment, passed by value: nothing is uploaded on the
// first call with new buffers, and a workgroup's first loads wait on no table
// reads (512^3: 9.3 -> 8.4 us a call, 7.9 of them on the GPU).  One workgroup
// per tile, XCD-contiguous ranges; problems whose tiles are walked several per
// workgroup (xcd_grid) stay with the tables.
template <class C, bool TA, bool TB>
__global__ __launch_bounds__(C::NTH, C::OCC) void gemm_f64_one_kernel(Prob P, Seg S) {
    __shared__ __attribute__((aligned(16))) char lds[2 * TileLds<C, TA, TB>::STAGE];
    P.seg0 = 0;
    P.nseg = 1;
    gemm_tile<C, TA, TB>(P, &S, xcd_remap(blockIdx.x, gridDim.x), lds);
}

// ---------------------------------------------------------------------------
// Direct-to-LDS form of the same GEMM for batches whose tiles are all
// interior (m, n multiples of 128, every segment's K a multiple of 8 and an
// even number of k-steps per problem, 16-byte aligned operands with even
// leading dimensions).  128x128 tiles, 4 waves of
// 64x64, two workgroups per CU, k-steps of 8 in a 3-stage LDS ring filled by
// global_load_lds_dwordx4 (no register staging).  Each operand is staged in
// the layout its memory order gives:
//  * contiguous along the tile's rows (A for opA = N, B for opB = T): one load
//    of a wave moves one k-row of 128 rows (1 KB); LDS [k][row] with a
//    1088-byte row stride, so the 64-bit fragment reads of four k-rows that
//    one MFMA needs fall in different bank halves;
//  * contiguous along k (A for opA = T, B for opB = N): one load moves 16
//    rows x 8 k (64 B each); LDS [row][k] with 16-byte chunk c of row r at
//    position c ^ ((r >> 1) & 3), the placement at which a wave's 128-bit
//    reads of 16 rows x 4 chunks run at the full LDS rate.
// Lane l of an MFMA supplies k = 2*(l/16) + s for sub-step s of a k-step:
// A and B use the same k assignment.  The fragments of step k+1 are read while
// the MFMAs of step k run, and the barrier runs one step ahead: after 24 of
// the 32 MFMAs of step k each wave waits for its own loads of step k+2, one
// barrier publishes them and frees the stage of step k (read completely during
// step k-1), which then receives step k+3.  Measured on a 16384^3 DGEMM: three
// stages beat four (fewer loads in flight) and a barrier inside the MFMA run
// beats one after it, together +2.2 %; five stages (unpadded, swizzled) lose 2 %.
namespace dmak {
constexpr int DBM = 128, DBN = 128, DBK = 8, DSTG = 3;
constexpr int RS = 1088;                   // k-row stride of a row-contiguous operand (bytes)
constexpr int RPART = DBK * RS;             // 8704 bytes
constexpr int KPART = 128 * DBK * 8;        // 8192 bytes
template <bool KC> constexpr int part() { return KC ? KPART : RPART; }
template <bool AK, bool BKC> constexpr int stage() { return part<AK>() + part<BKC>(); }
constexpr size_t lds_bytes(bool ak, bool bkc) { return (size_t)DSTG * ((ak ? KPART : RPART) + (bkc ? KPART : RPART)); }

__host__ __device__ constexpr int swz(int r) { return (r >> 1) & 3; }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    // gfx9 s_waitcnt: vmcnt in bits 3:0 and 15:14; expcnt and lgkmcnt left at their maxima
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void gvoid_t;

// Zeros for the loads of k past a segment's end and of the padding step
// that makes a tile's step count even (never written).
__device__ __align__(256) double g_dma_zero[128];

// Per-lane source of one operand's loads within a segment: `p` points at
// this lane's first element of the current k-step, `second` is the offset of
// the wave's second load and `step` the advance per k-step (all in doubles).
struct OperandCursor {
    const double* p;
    int64_t second, step;
};

// Cursor at k = 0 of a segment: `base` is the segment's operand pointer,
// `r0` the tile's first row, `ld` the leading dimension, `rows` the
// operand's row count.
//  * k-contiguous operand: rows past the end are read from the last row
//    (their products land in rows or columns of C that are never stored).
//  * row-contiguous operand: a lane loads the 16-byte aligned row pair
//    (2i, 2i+1) of a grid that starts `shift` (0 or 1) rows before `base`;
//    rows past the end read the last pair.  Every such pair holds at least
//    one element of the operand, and a 16-byte aligned access never crosses
//    a page, so the load stays inside mapped memory; the row before the
//    first (shift 1) and the row after the last (odd row count) only feed
//    rows or columns of C that are never stored.
// EDGE = false: the tile is interior and shift is 0 (no clamping).
template <bool KC, bool EDGE>
__device__ __forceinline__ OperandCursor operand_cursor(const double* base, int64_t ld, int64_t r0, int64_t rows,
                                                        int shift, int wave, int lane) {
    if constexpr (KC) {
        // rows 32w .. 32w+31 in two loads of 16 rows; lane -> row lane/4, position lane%4
        const int row = lane >> 2;
        const int chunk = (lane & 3) ^ swz(row);
        const int64_t ra = EDGE ? min(r0 + 32 * wave + row, rows - 1) : r0 + 32 * wave + row;
        const int64_t rb = EDGE ? min(r0 + 32 * wave + row + 16, rows - 1) : ra + 16;
        return OperandCursor{base + ra * ld + 2 * chunk, (rb - ra) * ld, DBK};
    } else {
        // k-rows 2w, 2w+1 of 128 rows; lane -> rows 2*lane, 2*lane+1 of the pair grid
        if constexpr (!EDGE) return OperandCursor{base + r0 + 2 * lane + (int64_t)(2 * wave) * ld, ld, DBK * ld};
        const int64_t last = (rows + shift - 1) & ~(int64_t)1;  // first row of the last pair
        const int64_t r = min(r0 + 2 * lane, last);
        return OperandCursor{base - shift + r + (int64_t)(2 * wave) * ld, ld, DBK * ld};
    }
}

// Cursor past the last segment: every load reads zeros.
__device__ __forceinline__ OperandCursor zero_cursor(int lane) { return OperandCursor{g_dma_zero + 2 * lane, 0, 0}; }

// One k-step of one operand into `dst` (its part of a stage), then advance.
// With tail != 0 the step is a segment's last and only its first `tail`
// (even for k-contiguous operands) k are real: the lanes past them load zeros.
template <bool KC>
__device__ __forceinline__ void issue_operand(char* dst, OperandCursor& c, int wave, int lane, int tail) {
    char* d0 = KC ? dst + (32 * wave) * 64 : dst + (2 * wave) * RS;
    char* d1 = KC ? d0 + 16 * 64 : d0 + RS;
    const double* p0 = c.p;
    const double* p1 = c.p + c.second;
    if (tail) {
        const double* z = g_dma_zero + 2 * lane;
        if constexpr (KC) {
            // this lane's k pair is 2 * chunk, 2 * chunk + 1 of the step
            const int k2 = 2 * ((lane & 3) ^ swz(lane >> 2));
            if (k2 >= tail) { p0 = z; p1 = z; }
        } else {
            // load 0 carries k-row 2w, load 1 k-row 2w + 1
            if (2 * wave >= tail) p0 = z;
            if (2 * wave + 1 >= tail) p1 = z;
        }
    }
    __builtin_amdgcn_global_load_lds((gvoid_t*)p0, (lds_void_t*)d0, 16, 0, 0);
    __builtin_amdgcn_global_load_lds((gvoid_t*)p1, (lds_void_t*)d1, 16, 0, 0);
    c.p += c.step;
}

// Fragments of one operand for one k-step: f[i][s] = X(row w0 + 16i + lr, k = 2lg + s).
template <bool KC>
__device__ __forceinline__ void read_operand(double (&f)[4][2], const char* part, int w0, int lr, int lg) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (KC) {
            const dv2 v = *reinterpret_cast<const dv2*>(part + (w0 + 16 * i + lr) * 64 + 16 * (lg ^ swz(lr)));
            f[i][0] = v.x;
            f[i][1] = v.y;
        } else {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                f[i][s] = *reinterpret_cast<const double*>(part + (2 * lg + s) * RS + (w0 + 16 * i + lr) * 8);
        }
    }
}
}  // namespace dmak

// EDGE = false: every tile interior, no row shift, every segment's K a
// multiple of 8 and an even step count (the same arithmetic without the
// edge paths).
template <bool AK, bool BKC, bool EDGE>
__device__ __forceinline__ void dma_tile(const Prob* __restrict__ probs, int nprob, const Seg* __restrict__ segs,
                                         int tile, char* lds) {
    using dmak::DBM; using dmak::DBN; using dmak::DBK; using dmak::DSTG;
    using dmak::read_operand; using dmak::wait_vmcnt;
    constexpr int SSZ = dmak::stage<AK, BKC>(), APART = dmak::part<AK>();
    int lo = 0, hi = nprob - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (probs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    const Prob P = probs[lo];
    const int local = tile - P.tile0;
    const int tiles_m = (int)((P.m + (P.shift & 1) + DBM - 1) / DBM);
    const int tiles_n = (int)((P.n + ((P.shift >> 1) & 1) + DBN - 1) / DBN);
    const int per_group = GROUP_M * tiles_n;
    const int group = local / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = local - group * per_group;
    const int64_t m0 = (int64_t)(first_m + in_group % gsize) * DBM;
    const int64_t n0 = (int64_t)(in_group / gsize) * DBN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int lr = lane & 15, lg = lane >> 4;

    // issue cursor over the problem's segments, one k-step (8) at a time; a
    // segment's last step may be partial, and past the last segment the
    // cursors read zeros (the padding step of an odd step count)
    const int sa = EDGE ? P.shift & 1 : 0, sb = EDGE ? (P.shift >> 1) & 1 : 0;  // row shifts of a row-contiguous A / B
    int iseg = P.seg0;
    Seg is = segs[iseg];
    int64_t left = (is.klen + DBK - 1) / DBK;  // k-steps left in the current segment
    int tail = (int)(is.klen % DBK);
    dmak::OperandCursor ca = dmak::operand_cursor<AK, EDGE>(is.a, is.lda, m0, P.m, sa, wave, lane);
    dmak::OperandCursor cb = dmak::operand_cursor<BKC, EDGE>(is.b, is.ldb, n0, P.n, sb, wave, lane);
    int ist = 0;
    auto issue_next = [&]() {
        char* st = lds + ist * SSZ;
        if (EDGE && left == 1 && tail) {
            dmak::issue_operand<AK>(st, ca, wave, lane, tail);
            dmak::issue_operand<BKC>(st + APART, cb, wave, lane, tail);
        } else {
            dmak::issue_operand<AK>(st, ca, wave, lane, 0);
            dmak::issue_operand<BKC>(st + APART, cb, wave, lane, 0);
        }
        ist = ist + 1 == DSTG ? 0 : ist + 1;
        if (--left == 0) {
            if (++iseg < P.seg0 + P.nseg) {
                is = segs[iseg];
                left = (is.klen + DBK - 1) / DBK;
                tail = (int)(is.klen % DBK);
                ca = dmak::operand_cursor<AK, EDGE>(is.a, is.lda, m0, P.m, sa, wave, lane);
                cb = dmak::operand_cursor<BKC, EDGE>(is.b, is.ldb, n0, P.n, sb, wave, lane);
            } else {
                left = INT64_MAX;
                tail = 0;
                ca = dmak::zero_cursor(lane);
                cb = dmak::zero_cursor(lane);
            }
        }
    };
    int64_t nk = 0;  // k-steps over all segments, rounded up to even (>= 2)
    for (int sg = P.seg0; sg < P.seg0 + P.nseg; ++sg) nk += (segs[sg].klen + DBK - 1) / DBK;
    nk += nk & 1;

    dv4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = dv4{0.0, 0.0, 0.0, 0.0};

    static_assert(DSTG == 3, "the waits below assume a 3-stage ring");
    for (int64_t s = 0; s < DSTG && s < nk; ++s) issue_next();
    // steps 0 and 1 published (4 loads per wave and step; step 2 may be in flight)
    if (nk >= 3) wait_vmcnt<4>(); else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    int rst = 1;  // stage of step kt + 1
    double fa0[4][2], fb0[4][2], fa1[4][2], fb1[4][2];
    read_operand<AK>(fa0, lds, wm, lr, lg);
    read_operand<BKC>(fb0, lds + APART, wn, lr, lg);
    int64_t kt = 0;
    // one step on (CA, CB) while the next step's fragments are read into (NA, NB):
    // MFMAs f = 16q + 4i + j in order, the barrier after f = 23
#define DMA_MFMAS(CA, CB, F0, F1)                                                                   \
    _Pragma("unroll") for (int f_ = F0; f_ < F1; ++f_) {                                            \
        const int q_ = f_ >> 4, i_ = (f_ >> 2) & 3, j_ = f_ & 3;                                    \
        acc[i_][j_] = __builtin_amdgcn_mfma_f64_16x16x4f64(CB[j_][q_], CA[i_][q_], acc[i_][j_], 0, 0, 0); \
    }
// FULL: kt + 3 < nk is known (the barrier and the issue of step kt+3 both run)
#define DMA_STEP(FULL, CA, CB, NA, NB)                                                                    \
    {                                                                                               \
        const char* nst = lds + rst * SSZ; /* harmless past the last step */                        \
        read_operand<AK>(NA, nst, wm, lr, lg);                                                      \
        DMA_MFMAS(CA, CB, 0, 24)                                                                    \
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                          \
        _Pragma("unroll") for (int g_ = 0; g_ < 4; ++g_) {                                          \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                      \
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                      \
        }                                                                                           \
        __builtin_amdgcn_sched_group_barrier(0x008, 14, 0);                                         \
        rst = rst + 1 == DSTG ? 0 : rst + 1;                                                        \
        if (FULL || kt + 2 < nk) {                                                                          \
            /* the stage of step kt was read during step kt-1; LDS reads retire in order, so once  \
               at most the 4 reads just issued are pending, none of it is still being read */       \
            __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (4 << 8));                  \
            wait_vmcnt<0>(); /* step kt+2, the only loads in flight */                              \
            __builtin_amdgcn_s_barrier();                                                           \
            if (FULL || kt + DSTG < nk) issue_next();                                                        \
        }                                                                                           \
        read_operand<BKC>(NB, nst + APART, wn, lr, lg);                                             \
        DMA_MFMAS(CA, CB, 24, 32)                                                                   \
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                          \
        _Pragma("unroll") for (int g_ = 0; g_ < 3; ++g_) {                                          \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                      \
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                      \
        }                                                                                           \
        ++kt;                                                                                       \
    }
    // Steady turns of twelve steps without conditions, then the last steps
    // two at a time.  The compiler drains every load at a loop head (it
    // cannot count across the direct-to-LDS loads there), which with a
    // two-step loop was a wait for step kt+2's loads every other step:
    // twelve-step turns run 5.5 % faster at 16384^3.
    while (kt + 15 <= nk) {
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
        DMA_STEP(true, fa0, fb0, fa1, fb1);
        DMA_STEP(true, fa1, fb1, fa0, fb0);
    }
    while (kt < nk) {
        DMA_STEP(false, fa0, fb0, fa1, fb1);
        DMA_STEP(false, fa1, fb1, fa0, fb0);
    }
#undef DMA_STEP
#undef DMA_MFMAS

    // acc[i][j][v] = sum for C(m0 + wm + 16i + lr - sa, n0 + wn + 16j + lg + 4v - sb)
    const double alpha = P.alpha, beta = P.beta;
    const bool interior = !EDGE || (sa == 0 && sb == 0 && m0 + DBM <= P.m && n0 + DBN <= P.n);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + wm + 16 * i + lr - sa;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t n = n0 + wn + 16 * j + lg + 4 * v - sb;
                if (!interior && (m < 0 || m >= P.m || n < 0 || n >= P.n)) continue;
                __attribute__((address_space(1))) double* cp =
                    (__attribute__((address_space(1))) double*)(P.c + m + n * P.ldc);
                double val = alpha * acc[i][j][v];
                if (beta != 0.0) val = fma(beta, *cp, val);
                *cp = val;
            }
        }
    }
}

// MODE as gemm_f64_kernel: 0 tile = blockIdx.x, 1 XCD-contiguous ranges,
// 2 persistent (tiles taken from `counter`, zeroed before the launch).
template <bool AK, bool BKC, bool EDGE, int MODE>
__global__ __launch_bounds__(256, 2) void gemm_f64_dma_kernel(const Prob* __restrict__ probs, int nprob,
                                                               const Seg* __restrict__ segs, int total_tiles,
                                                               int* __restrict__ counter) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    if (MODE == 0) {
        dma_tile<AK, BKC, EDGE>(probs, nprob, segs, blockIdx.x, lds);
    } else if (MODE == 1) {
        dma_tile<AK, BKC, EDGE>(probs, nprob, segs, xcd_remap(blockIdx.x, total_tiles), lds);
    } else {
        __shared__ int next;
        while (true) {
            __syncthreads();  // the previous tile's LDS reads and `next` reads are complete
            if (threadIdx.x == 0) next = atomicAdd(counter, 1);
            __syncthreads();
            const int tile = next;
            if (tile >= total_tiles) break;
            dma_tile<AK, BKC, EDGE>(probs, nprob, segs, tile, lds);
        }
    }
}

// A in registers (interior batches): each wave owns 32 rows of the 128x128
// tile and all 128 columns (2 x 8 MFMA tiles of 16x16), so no two waves use
// the same element of A, and A needs neither LDS nor a barrier.  Lane
// (lr, lg) holds rows 2lr, 2lr+1 of its wave's 32 at k = 2lg + q (q = 0, 1):
// MFMA tile i = 0 takes the even rows, i = 1 the odd ones.  Two 16-byte
// global loads per k-step: with A row-contiguous (opA = N) one per k (the
// row pair), with A k-contiguous (opA = T) one per row (the k pair).  A runs three k-steps ahead in a ring of registers
// (loaded after the last MFMA that reads the slot); B goes through the
// 3-stage direct-to-LDS ring of dma_tile, whose fragments of step k+1 are read
// in two halves around the barrier.  Loads in issue order: B(k+3) at the
// barrier of step k, A(k+3) after its MFMAs, so the barrier's wait for B(k+2)
// leaves the two loads of A(k+2) in flight.
template <bool AK, bool BKC>
__device__ __forceinline__ void dma_tile_ar(const Prob* __restrict__ probs, int nprob, const Seg* __restrict__ segs,
                                            int tile, char* lds) {
    using dmak::DBM; using dmak::DBN; using dmak::DBK; using dmak::DSTG;
    using dmak::read_operand; using dmak::wait_vmcnt;
    constexpr int SSZ = dmak::part<BKC>();
    int lo = 0, hi = nprob - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (probs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    const Prob P = probs[lo];
    const int local = tile - P.tile0;
    const int tiles_m = (int)((P.m + (P.shift & 1) + DBM - 1) / DBM);
    const int tiles_n = (int)((P.n + ((P.shift >> 1) & 1) + DBN - 1) / DBN);
    const int per_group = GROUP_M * tiles_n;
    const int group = local / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = local - group * per_group;
    const int64_t m0 = (int64_t)(first_m + in_group % gsize) * DBM;
    const int64_t n0 = (int64_t)(in_group / gsize) * DBN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int64_t arow = m0 + 32 * wave + 2 * lr;

    // issue cursors: every segment a whole number of k-steps, none past the end
    int iseg = P.seg0;
    Seg is = segs[iseg];
    int64_t left = is.klen / DBK;
    // A at (arow, k = 2lg) of the next step to issue; the second load is one ld away
    auto a_origin = [&](const Seg& g) { return AK ? g.a + arow * g.lda + 2 * lg : g.a + arow + (int64_t)(2 * lg) * g.lda; };
    const double* ap = a_origin(is);
    int64_t alda = is.lda;
    dmak::OperandCursor cb = dmak::operand_cursor<BKC, false>(is.b, is.ldb, n0, P.n, 0, wave, lane);
    const double* apend = ap;  // A of the step issued last
    int64_t apld = alda;
    int ist = 0;
    auto issue_next = [&]() {
        dmak::issue_operand<BKC>(lds + ist * SSZ, cb, wave, lane, 0);
        ist = ist + 1 == DSTG ? 0 : ist + 1;
        apend = ap;
        apld = alda;
        ap += AK ? DBK : DBK * alda;
        if (--left == 0 && ++iseg < P.seg0 + P.nseg) {
            is = segs[iseg];
            left = is.klen / DBK;
            ap = a_origin(is);
            alda = is.lda;
            cb = dmak::operand_cursor<BKC, false>(is.b, is.ldb, n0, P.n, 0, wave, lane);
        }
    };
    // ra[slot][h] of the slot's step: opA = N, h = q: A(rows 2lr, 2lr + 1; k = 2lg + q);
    // opA = T, h = i: A(row 2lr + i; k = 2lg, 2lg + 1)
    dv2 ra[3][2];
    auto load_a = [&](dv2 (&r)[2]) {
        r[0] = gld2(apend);
        r[1] = gld2(apend + apld);
    };
    int64_t nk = 0;  // even (an interior batch)
    for (int sg = P.seg0; sg < P.seg0 + P.nseg; ++sg) nk += segs[sg].klen / DBK;

    dv4 acc[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = dv4{0.0, 0.0, 0.0, 0.0};

    static_assert(DSTG == 3, "the waits below assume a 3-stage ring");
    issue_next();
    load_a(ra[0]);
    issue_next();
    load_a(ra[1]);
    if (nk > 2) {
        issue_next();
        load_a(ra[2]);
        wait_vmcnt<6>();  // B of steps 0 and 1 landed; A(1), B(2), A(2) may be in flight
    } else {
        wait_vmcnt<0>();
    }
    __builtin_amdgcn_s_barrier();
    int rst = 1;  // stage of step kt + 1
    double fb0[2][4][2], fb1[2][4][2];  // f[h][jj][q] = B(row 64h + 16jj + lr, k = 2lg + q)
    read_operand<BKC>(fb0[0], lds, 0, lr, lg);
    read_operand<BKC>(fb0[1], lds, 64, lr, lg);
    int64_t kt = 0;
    // MFMAs f = 16q + 8i + j in order, the barrier after f = 23
#define AR_MFMAS(SLOT, CB, F0, F1)                                                                  \
    _Pragma("unroll") for (int f_ = F0; f_ < F1; ++f_) {                                            \
        const int q_ = f_ >> 4, i_ = (f_ >> 3) & 1, j_ = f_ & 7;                                    \
        acc[i_][j_] = __builtin_amdgcn_mfma_f64_16x16x4f64(CB[j_ >> 2][j_ & 3][q_],                \
                                                           AK ? ra[SLOT][i_][q_] : ra[SLOT][q_][i_], acc[i_][j_], 0, 0, 0); \
    }
// FULL: kt + 3 < nk is known (the barrier, the issue of B(kt+3) and the load of A(kt+3) all run)
#define AR_STEP(FULL, SLOT, CB, NB)                                                                 \
    {                                                                                               \
        const char* nst = lds + rst * SSZ; /* harmless past the last step */                        \
        read_operand<BKC>(NB[0], nst, 0, lr, lg);                                                   \
        AR_MFMAS(SLOT, CB, 0, 24)                                                                   \
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                          \
        _Pragma("unroll") for (int g_ = 0; g_ < 4; ++g_) {                                          \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                      \
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                      \
        }                                                                                           \
        __builtin_amdgcn_sched_group_barrier(0x008, 14, 0);                                         \
        rst = rst + 1 == DSTG ? 0 : rst + 1;                                                        \
        if (FULL || kt + 2 < nk) {                                                                  \
            /* the stage of step kt was read during step kt-1: once at most the 4 reads just        \
               issued are pending, none of it is still being read */                                \
            __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (4 << 8));                  \
            wait_vmcnt<2>(); /* B(kt+2); A(kt+2), issued after it, may be in flight */              \
            __builtin_amdgcn_s_barrier();                                                           \
            if (FULL || kt + DSTG < nk) issue_next();                                                \
        }                                                                                           \
        read_operand<BKC>(NB[1], nst, 64, lr, lg);                                                  \
        AR_MFMAS(SLOT, CB, 24, 32)                                                                  \
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                          \
        _Pragma("unroll") for (int g_ = 0; g_ < 3; ++g_) {                                          \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                      \
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                                      \
        }                                                                                           \
        if (FULL || kt + DSTG < nk) load_a(ra[SLOT]);                                               \
        ++kt;                                                                                       \
    }
    // A slot = step % 3, B fragments alternate: six steps make a cycle, and a
    // steady turn runs four of them.  The steady turns have no conditions (so
    // the waits the compiler derives inside them stay partial); the compiler
    // drains every load at the loop head, once per turn (at 16384^3 twelve-step
    // turns beat six-step ones by 0.3 % on NN and 2 % on TN, 24-step turns
    // twelve-step ones by 0.2 %); the last 2 to 26 steps, nk even, follow.
    while (kt + 27 <= nk) {
        AR_STEP(true, 0, fb0, fb1);
        AR_STEP(true, 1, fb1, fb0);
        AR_STEP(true, 2, fb0, fb1);
        AR_STEP(true, 0, fb1, fb0);
        AR_STEP(true, 1, fb0, fb1);
        AR_STEP(true, 2, fb1, fb0);
        AR_STEP(true, 0, fb0, fb1);
        AR_STEP(true, 1, fb1, fb0);
        AR_STEP(true, 2, fb0, fb1);
        AR_STEP(true, 0, fb1, fb0);
        AR_STEP(true, 1, fb0, fb1);
        AR_STEP(true, 2, fb1, fb0);
        AR_STEP(true, 0, fb0, fb1);
        AR_STEP(true, 1, fb1, fb0);
        AR_STEP(true, 2, fb0, fb1);
        AR_STEP(true, 0, fb1, fb0);
        AR_STEP(true, 1, fb0, fb1);
        AR_STEP(true, 2, fb1, fb0);
        AR_STEP(true, 0, fb0, fb1);
        AR_STEP(true, 1, fb1, fb0);
        AR_STEP(true, 2, fb0, fb1);
        AR_STEP(true, 0, fb1, fb0);
        AR_STEP(true, 1, fb0, fb1);
        AR_STEP(true, 2, fb1, fb0);
    }
    while (true) {
        AR_STEP(false, 0, fb0, fb1);
        AR_STEP(false, 1, fb1, fb0);
        if (kt >= nk) break;
        AR_STEP(false, 2, fb0, fb1);
        AR_STEP(false, 0, fb1, fb0);
        if (kt >= nk) break;
        AR_STEP(false, 1, fb0, fb1);
        AR_STEP(false, 2, fb1, fb0);
        if (kt >= nk) break;
    }
#undef AR_STEP
#undef AR_MFMAS

    // acc[i][j][v] = sum for C(arow + i, n0 + 16j + lg + 4v)
    const double alpha = P.alpha, beta = P.beta;
    typedef __attribute__((address_space(1))) double gd;
    typedef __attribute__((address_space(1))) dv2 gd2;
    const bool vec = ((reinterpret_cast<uintptr_t>(P.c) & 15) == 0) && !(P.ldc & 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t n = n0 + 16 * j + lg + 4 * v;
            double* cp = P.c + arow + n * P.ldc;
            dv2 val = dv2{alpha * acc[0][j][v], alpha * acc[1][j][v]};
            if (vec) {
                if (beta != 0.0) {
                    const dv2 c = *(gd2*)cp;
                    val = dv2{fma(beta, c.x, val.x), fma(beta, c.y, val.y)};
                }
                *(gd2*)cp = val;
            } else {
                if (beta != 0.0) val = dv2{fma(beta, ((gd*)cp)[0], val.x), fma(beta, ((gd*)cp)[1], val.y)};
                ((gd*)cp)[0] = val.x;
                ((gd*)cp)[1] = val.y;
            }
        }
    }
}

template <bool AK, bool BKC, int MODE>
__global__ __launch_bounds__(256, 2) void gemm_f64_dma_ar_kernel(const Prob* __restrict__ probs, int nprob,
                                                                  const Seg* __restrict__ segs, int total_tiles,
                                                                  int* __restrict__ counter) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    if (MODE == 0) {
        dma_tile_ar<AK, BKC>(probs, nprob, segs, blockIdx.x, lds);
    } else if (MODE == 1) {
        dma_tile_ar<AK, BKC>(probs, nprob, segs, xcd_remap(blockIdx.x, total_tiles), lds);
    } else {
        __shared__ int next;
        while (true) {
            __syncthreads();  // the previous tile's LDS reads and `next` reads are complete
            if (threadIdx.x == 0) next = atomicAdd(counter, 1);
            __syncthreads();
            const int tile = next;
            if (tile >= total_tiles) break;
            dma_tile_ar<AK, BKC>(probs, nprob, segs, tile, lds);
        }
    }
}

template <bool AK, bool BKC>
void launch_dma_ar(int mode, const Prob* dp, int np, const Seg* ds, int tiles, int grid, int* counter, hipStream_t st) {
    const size_t lb = (size_t)dmak::DSTG * dmak::part<BKC>();
    if (mode == DG_GEMM_MODE_ROUND_ROBIN)
        hipLaunchKernelGGL((gemm_f64_dma_ar_kernel<AK, BKC, 0>), dim3(tiles), dim3(256), lb, st, dp, np, ds, tiles, counter);
    else if (mode == DG_GEMM_MODE_XCD)
        hipLaunchKernelGGL((gemm_f64_dma_ar_kernel<AK, BKC, 1>), dim3(tiles), dim3(256), lb, st, dp, np, ds, tiles, counter);
    else
        hipLaunchKernelGGL((gemm_f64_dma_ar_kernel<AK, BKC, 2>), dim3(grid), dim3(256), lb, st, dp, np, ds, tiles, counter);
}

template <bool AK, bool BKC, bool EDGE>
void launch_dma_e(int mode, const Prob* dp, int np, const Seg* ds, int tiles, int grid, int* counter, hipStream_t st) {
    const size_t lb = dmak::lds_bytes(AK, BKC);
    if (mode == DG_GEMM_MODE_ROUND_ROBIN)
        hipLaunchKernelGGL((gemm_f64_dma_kernel<AK, BKC, EDGE, 0>), dim3(tiles), dim3(256), lb, st, dp, np, ds, tiles, counter);
    else if (mode == DG_GEMM_MODE_XCD)
        hipLaunchKernelGGL((gemm_f64_dma_kernel<AK, BKC, EDGE, 1>), dim3(tiles), dim3(256), lb, st, dp, np, ds, tiles, counter);
    else
        hipLaunchKernelGGL((gemm_f64_dma_kernel<AK, BKC, EDGE, 2>), dim3(grid), dim3(256), lb, st, dp, np, ds, tiles, counter);
}
template <bool AK, bool BKC>
void launch_dma(bool edge, int mode, const Prob* dp, int np, const Seg* ds, int tiles, int grid, int* counter,
                hipStream_t st) {
    static const bool no_areg = getenv("DG_GEMM_NO_AREG") != nullptr;
    if (!edge && !no_areg) return launch_dma_ar<AK, BKC>(mode, dp, np, ds, tiles, grid, counter, st);
    if (edge) launch_dma_e<AK, BKC, true>(mode, dp, np, ds, tiles, grid, counter, st);
    else launch_dma_e<AK, BKC, false>(mode, dp, np, ds, tiles, grid, counter, st);
}

__global__ void zero_counter_kernel(int* counter) { *counter = 0; }

__global__ void scale_kernel(int64_t m, int64_t n, double beta, double* __restrict__ C, int64_t ldc) {
    const int64_t total = m * n;
    for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < total;
         x += (int64_t)gridDim.x * blockDim.x) {
        const int64_t col = x / m, row = x - col * m;
        double* p = C + row + col * ldc;
        *p = (beta == 0.0) ? 0.0 : beta * *p;
    }
}

template <class C, bool TA, bool TB>
void launch_mode(int mode, const Prob* dp, int np, const Seg* ds, int tiles, int grid, int* counter,
                 hipStream_t st) {
    if (mode == DG_GEMM_MODE_ROUND_ROBIN)
        hipLaunchKernelGGL((gemm_f64_kernel<C, TA, TB, 0>), tile_grid(tiles), dim3(C::NTH), 0, st, dp, np, ds, tiles, counter);
    else if (mode == DG_GEMM_MODE_XCD)
        hipLaunchKernelGGL((gemm_f64_kernel<C, TA, TB, 1>), dim3(std::min(grid, 1 << 22)), dim3(C::NTH), 0, st, dp, np, ds, tiles, counter);
    else
        hipLaunchKernelGGL((gemm_f64_kernel<C, TA, TB, 2>), dim3(grid), dim3(C::NTH), 0, st, dp, np, ds, tiles, counter);
}

template <class C>
void launch_one(char opA, char opB, const Prob& p, const Seg& s, int tiles, hipStream_t st) {
    const bool ta = opA == 'T', tb = opB == 'T';
    const auto kernel = !ta && !tb ? gemm_f64_one_kernel<C, false, false> : !ta ? gemm_f64_one_kernel<C, false, true>
                      : !tb        ? gemm_f64_one_kernel<C, true, false>  : gemm_f64_one_kernel<C, true, true>;
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(C::NTH), 0, st, p, s);
}

template <class C>
void launch_cfg(char opA, char opB, int mode, const Prob* dp, int np, const Seg* ds, int tiles, int grid, int* counter,
                hipStream_t st) {
    const bool ta = opA == 'T', tb = opB == 'T';
    if (!ta && !tb) launch_mode<C, false, false>(mode, dp, np, ds, tiles, grid, counter, st);
    else if (!ta && tb) launch_mode<C, false, true>(mode, dp, np, ds, tiles, grid, counter, st);
    else if (ta && !tb) launch_mode<C, true, false>(mode, dp, np, ds, tiles, grid, counter, st);
    else launch_mode<C, true, true>(mode, dp, np, ds, tiles, grid, counter, st);
}

}  // namespace

int launch_scale(int64_t m, int64_t n, double beta, double* C, int64_t ldc, hipStream_t stream) {
    if (m <= 0 || n <= 0) return DG_OK;
    int64_t total = m * n;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, m, n, beta, C, ldc);
    DG_LAUNCH_CHECK();
    return DG_OK;
}

// What the routing needs to know of a problem, from one pass over its segments.
struct Route {
    int64_t depth = 0;      // k of all segments
    int64_t staged[3];      // of several: k of the register-staged tiles' stages, each segment's last one whole
    bool direct = true;     // the direct-to-LDS kernels take it; then
    int sa = 0, sb = 0;     // whether its A (B) starts 8 bytes past a 16-byte boundary (k-contiguous: -1), and
    bool k_ok = false;      // its k is an even number of whole k-steps
    bool elements[3] = {};  // the register-staged kernel's tiles (gen[w]) load it by single elements
};

// Whether tiles of shape C load a problem's runs whole (`bits`: all its bases).
template <class C>
static bool takes(bool ak, bool bkc, uintptr_t bits, int64_t lda, int64_t ldb) {
    using KC = Staged<double, true, C::BM, C::BK>;
    using RC = Staged<double, false, C::BM, C::BK>;
    const double* x = reinterpret_cast<const double*>(bits);
    return (ak ? KC::takes(x, lda) : RC::takes(x, lda)) && (bkc ? KC::takes(x, ldb) : RC::takes(x, ldb));
}

static Route route_of(const Prob& p, const std::vector<Seg>& segs, bool ak, bool bkc) {
    Route r;
    uintptr_t bits = 0;
    int64_t lda = 1, ldb = 1;  // the longest
    int64_t s16 = 0, s32 = 0;  // stages 16 and 32 deep
    static_assert(Cfg128::BK == 16 && Cfg64::BK == 16 && Cfg32::BK == 32, "stages counted below");
    int off_a = -1, off_b = -1;  // byte offset within 16 of a row-contiguous A / B
    int64_t steps = 0;
    bool whole = true;  // every segment a whole number of k-steps
    for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) {
        const Seg& g = segs[s];
        r.depth += g.klen;
        steps += (g.klen + dmak::DBK - 1) / dmak::DBK;
        s16 += (g.klen + 15) / 16;
        s32 += (g.klen + 31) / 32;
        if (g.klen % dmak::DBK) whole = false;
        bits |= reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b);
        lda = std::max(lda, g.lda);
        ldb = std::max(ldb, g.ldb);
        const int oa = (int)(reinterpret_cast<uintptr_t>(g.a) & 15), ob = (int)(reinterpret_cast<uintptr_t>(g.b) & 15);
        if ((g.lda & 1) || (g.ldb & 1) || g.klen <= 0) r.direct = false;
        if (ak) { if (oa || (g.klen & 1)) r.direct = false; }   // k pairs, 16-byte aligned
        else { if ((oa & 7) || (off_a >= 0 && oa != off_a)) r.direct = false; off_a = oa; }
        if (bkc) { if (ob || (g.klen & 1)) r.direct = false; }
        else { if ((ob & 7) || (off_b >= 0 && ob != off_b)) r.direct = false; off_b = ob; }
    }
    r.sa = ak ? -1 : off_a == 8;
    r.sb = bkc ? -1 : off_b == 8;
    r.k_ok = whole && !(steps & 1);
    r.staged[0] = r.staged[1] = p.nseg > 1 ? 16 * s16 : r.depth;
    r.staged[2] = p.nseg > 1 ? 32 * s32 : r.depth;
    r.elements[0] = !takes<Cfg128>(ak, bkc, bits, lda, ldb);
    r.elements[1] = !takes<Cfg64>(ak, bkc, bits, lda, ldb);
    r.elements[2] = !takes<Cfg32>(ak, bkc, bits, lda, ldb);
    return r;
}

// Lists of a batch: A in registers, edge-handling direct-to-LDS, then the
// register-staged kernel's three tile edges.
enum { kListAreg, kListEdge, kListGen, kLists = kListGen + 3 };
constexpr int kTileLog2[kLists] = {7, 7, 7, 6, 5};  // of their tiles' edges
static_assert(dmak::DBM == 128 && dmak::DBN == 128 && Cfg128::BM == 128 && Cfg64::BM == 64 && Cfg32::BM == 32, "kTileLog2");

// Time (us) of one list's launch, to choose between the tiles: the fullest
// CU's c tiles at the rate that so many reach, share of 78.6 TFLOP/s, plus
// `round` us of prologue and epilogue, and `seg` us per segment after a tile's
// first, per round of `conc` resident tiles.
// Measured: A in registers 0.91 with one tile per CU, 0.95 with more (both
// operands in LDS 0.85, 0.93); register-staged 128x128 0.95 with one, 0.965 up
// to 15 (4096^3: 1816 us against 1836 with A in registers), then less, 0.89
// from 32 on: its workgroups drift apart and fetch four times as much from
// beyond the L2 (16384^3: 398 GB against 103), and with 98.5 % busy matrix cores
// it is no faster than A in registers (116.5 ms both, SUMMA too); 64x64 0.92, 0.88 from 25 tiles per CU on, 0.85 from 64 on;
// 32x32 0.67, 0.72, 0.76, 0.78 with one to four, 0.80 with more.  Loads by
// elements: kElementRate of these (TN 500 x 4096 x 4096 with 2^22 + 2 rows to a
// column, 64x64 tiles: 403 us, 257 with whole runs; NN 4096 x 4096 x 480, odd:
// 319 us against 251).
// A register-staged kernel leaves its steady turns at every segment's end,
// the direct-to-LDS kernels do not: SUMMA 2048^3 on 2 x 2 in panels of 512, 128,
// 64 and 16: direct 251, 255, 259 and 287 us, 128x128 243, 260, 282 and 380,
// 64x64 245, 255, 267 and 320, 32x32 297, 315, 346 and 963 (its stages are 32
// deep).
constexpr double kElementRate = 0.65;
struct Rate {
    int conc;
    double round, seg;
    struct { int64_t from; double eff; } at[5];  // ascending; the last whose `from` c reaches
};
constexpr Rate kRate[kLists] = {{2, 4, 0.25, {{1, 0.91}, {2, 0.95}}},
                                {2, 4, 0.25, {{1, 0.85}, {2, 0.93}}},
                                {2, 8, 1.2, {{1, 0.95}, {2, 0.965}, {16, 0.93}, {32, 0.89}}},
                                {4, 4, 0.6, {{1, 0.92}, {5, 0.91}, {25, 0.88}, {64, 0.85}}},
                                {4, 4, 0.4, {{1, 0.67}, {2, 0.72}, {3, 0.76}, {4, 0.78}, {5, 0.80}}}};

struct ListCost {
    int64_t tiles = 0, seams = 0;  // seams: segments after a tile's first, of all tiles
    double sum = 0, most = 0, least = 1e300;  // k of all tiles, the longest, the shortest
    void add(int64_t n, int64_t k, int nseg, bool elements) {
        const double x = elements ? (double)k * (1.0 / kElementRate) : (double)k;
        tiles += n;
        seams += n * (nseg - 1);
        sum += (double)n * x;
        most = std::max(most, x);
        least = std::min(least, x);
    }
    double time(const Rate& r, int64_t edge) const {
        if (!tiles) return 0;
        const int64_t c = (tiles + 255) / 256;
        double eff = 0;
        for (const auto& x : r.at)
            if (x.from > 0 && x.from <= c) eff = x.eff;
        const double load = most == least ? (double)c * most : std::max(sum / 256 + most / 2, most);
        const double us = 2.0 * (double)(edge * edge) / (78.6e6 / 256);  // per k of a tile
        return load * us / eff + (r.round + r.seg * (double)seams / (double)tiles) * std::max(1.0, (double)c / r.conc);
    }
};

// Calls part(list, first row, rows, first column, columns) for the whole of a
// problem, or for the parts it is cut into, under one tile choice.
template <class F>
static void split_problem(const Prob& p, const Route& r, int tile, bool split_edges, const F& part) {
    constexpr int64_t TM = dmak::DBM, TN = dmak::DBN;
    static const bool no_narrow = getenv("DG_GEMM_NO_NARROW") != nullptr;
    // on the register-staged kernel: the choice's own tiles, or the smaller
    // ones that a narrow part fills better
    auto staged = [&](int64_t r0, int64_t nr, int64_t c0, int64_t nc) {
        const int w = tile == DG_GEMM_TILE_32x32 ? 2 : tile == DG_GEMM_TILE_64x64 ? 1 : 0;
        const int64_t narrow = std::min(nr, nc);
        part(kListGen + std::max(w, narrow <= 32 ? 2 : narrow <= 96 ? 1 : 0), r0, nr, c0, nc);
    };
    // the strips around rows [r0, r0 + mi) x columns [c0, c0 + ni)
    auto strips = [&](int64_t r0, int64_t mi, int64_t c0, int64_t ni, bool edge) {
        auto strip = [&](int64_t r1, int64_t nr, int64_t c1, int64_t nc) {
            if (edge) part(kListEdge, r1, nr, c1, nc); else staged(r1, nr, c1, nc);
        };
        if (r0 > 0) strip(0, r0, 0, p.n);                                       // rows before it
        if (r0 + mi < p.m) strip(r0 + mi, p.m - r0 - mi, 0, p.n);               // rows after it
        if (c0 > 0) strip(r0, mi, 0, c0);                                       // columns before it
        if (c0 + ni < p.n) strip(r0, mi, c0 + ni, p.n - c0 - ni);               // columns after it
    };
    if (tile != DG_GEMM_TILE_DIRECT || !r.direct) {
        // whole, or cut into whole 128x128 tiles and strips (a strip that
        // nearly fills its tiles stays with them)
        auto inside = [](int64_t x) { return x % 128 > 96 ? x : x / 128 * 128; };
        const int64_t mi = inside(p.m), ni = inside(p.n);
        if (tile == DG_GEMM_TILE_64x64 || tile == DG_GEMM_TILE_32x32 || tile == DG_GEMM_TILE_128x128_WHOLE ||
            !split_edges || (mi == p.m && ni == p.n) || mi * ni < 8 * 128 * 128)
            return staged(0, p.m, 0, p.n);
        staged(0, mi, 0, ni);
        return strips(0, mi, 0, ni, false);
    }
    if (r.sa < 1 && r.sb < 1 && p.m % TM == 0 && p.n % TN == 0 && r.k_ok) return part(kListAreg, 0, p.m, 0, p.n);
    // A shifted row-contiguous operand is aligned from row (column) 127 on:
    // the strip before it is one tile row (column) of the shifted tiling, so
    // cutting there adds no tiles.
    const int64_t r0 = r.sa == 1 ? TM - 1 : 0, c0 = r.sb == 1 ? TN - 1 : 0;
    const int64_t mi = p.m > r0 ? (p.m - r0) / TM * TM : 0, ni = p.n > c0 ? (p.n - c0) / TN * TN : 0;
    if (!split_edges || !r.k_ok || mi * ni < 8 * TM * TN) return part(kListEdge, 0, p.m, 0, p.n);
    part(kListAreg, r0, mi, c0, ni);
    strips(r0, mi, c0, ni, no_narrow);
}

// Shift bits and tiles of a part of a problem on a list.
static int shift_of(const Route& r, int list, int64_t r0, int64_t c0) {
    if (list >= kListGen) return r.elements[list - kListGen] ? kByElements : 0;
    // k-contiguous operands have no shift, wherever their part starts
    return (r.sa >= 0 ? (int)((r.sa + r0) & 1) : 0) | (r.sb >= 0 ? (int)((r.sb + c0) & 1) : 0) << 1;
}
static int64_t tiles_of(int list, int shift, int64_t nr, int64_t nc) {
    const int e = kTileLog2[list], round = (1 << e) - 1;
    const int sa = list < kListGen ? shift & 1 : 0, sb = list < kListGen ? (shift >> 1) & 1 : 0;
    return ((nr + sa + round) >> e) * ((nc + sb + round) >> e);
}

// One tile choice of a batch: the estimated time (us) of its launches, the
// problems of each list, the segments that cut parts add, and whether it fits
// one launch per list.
struct Estimate {
    double time = 0;
    size_t probs[kLists] = {};
    int64_t segs = 0;
    bool fits = true;
};
static Estimate estimate(const std::vector<Prob>& probs, const std::vector<Route>& routes, size_t nsegs, int tile,
                         bool split_edges) {
    Estimate x;
    ListCost cost[kLists];
    for (size_t i = 0; i < probs.size(); ++i) {
        const Prob& p = probs[i];
        const Route& r = routes[i];
        if (p.m <= 0 || p.n <= 0 || p.nseg <= 0) continue;
        split_problem(p, r, tile, split_edges, [&](int list, int64_t r0, int64_t nr, int64_t c0, int64_t nc) {
            const int shift = shift_of(r, list, r0, c0);
            cost[list].add(tiles_of(list, shift, nr, nc), list < kListGen ? r.depth : r.staged[list - kListGen], p.nseg,
                           shift & kByElements);
            ++x.probs[list];
            if (nr < p.m || nc < p.n) x.segs += p.nseg;
        });
    }
    for (int l = 0; l < kLists; ++l) {
        x.time += cost[l].time(kRate[l], (int64_t)1 << kTileLog2[l]);
        x.fits = x.fits && cost[l].tiles <= INT32_MAX;
    }
    x.fits = x.fits && (int64_t)nsegs + x.segs <= INT32_MAX;
    return x;
}

// Fills the lists of one tile choice.  A part of a problem becomes a problem
// of its own, its segments re-based and appended.
static void build_lists(bool ak, bool bkc, const std::vector<Prob>& probs, const std::vector<Route>& routes,
                        std::vector<Seg>&& segs, int tile, bool split_edges, const Estimate& size, GemmBatch& out) {
    out = GemmBatch{};
    out.segs = std::move(segs);
    if (size.segs) out.segs.reserve(out.segs.size() + (size_t)size.segs);
    std::vector<Prob>* lists[kLists] = {&out.dma, &out.dmae, &out.gen[0], &out.gen[1], &out.gen[2]};
    for (int l = 0; l < kLists; ++l) lists[l]->reserve(size.probs[l]);
    int64_t tiles[kLists] = {};
    for (size_t i = 0; i < probs.size(); ++i) {
        const Prob& p = probs[i];
        const Route& r = routes[i];
        if (p.m <= 0 || p.n <= 0 || p.nseg <= 0) continue;
        split_problem(p, r, tile, split_edges, [&](int list, int64_t r0, int64_t nr, int64_t c0, int64_t nc) {
            Prob q = p;
            if (nr < p.m || nc < p.n) {
                q.m = nr;
                q.n = nc;
                q.c = p.c + r0 + c0 * p.ldc;
                q.seg0 = (int32_t)out.segs.size();
                for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) {
                    Seg g = out.segs[s];
                    g.a += ak ? r0 * g.lda : r0;
                    g.b += bkc ? c0 * g.ldb : c0;
                    out.segs.push_back(g);
                }
            }
            q.shift = shift_of(r, list, r0, c0);
            q.tile0 = (int32_t)tiles[list];
            tiles[list] += tiles_of(list, q.shift, nr, nc);
            lists[list]->push_back(q);
        });
    }
    out.tiles_dma = (int)tiles[kListAreg];
    out.tiles_dmae = (int)tiles[kListEdge];
    for (int w = 0; w < 3; ++w) out.tiles_gen[w] = (int)tiles[kListGen + w];
}

int forced_tile() {
    static const int forced = [] {
        const char* const names[DG_GEMM_TILES] = {"direct", "128x128", "128x128whole", "64x64", "32x32"};
        const char* e = getenv("DG_GEMM_TILE");
        for (int t = 0; e && t < DG_GEMM_TILES; ++t)
            if (!strcmp(e, names[t])) return t;
        return (int)DG_GEMM_TILE_AUTO;
    }();
    return forced;
}

// The batch is looked at once and built once: the choices are compared by
// their estimates.  SUMMA, both operands transposed, 8192^3 in blocks of 64
// (2.1 million segments): 13 ms of host time, 290 with a build per choice.
int prepare_gemm(char opA, char opB, const std::vector<Prob>& probs, std::vector<Seg> segs, GemmBatch& out,
                 bool split_edges, int tile) {
    // DG_GEMM_NO_DMA keeps everything on the register-staged kernel
    static const bool no_dma = getenv("DG_GEMM_NO_DMA") != nullptr;
    if (forced_tile() != DG_GEMM_TILE_AUTO) tile = forced_tile();
    if (no_dma && tile == DG_GEMM_TILE_DIRECT) tile = DG_GEMM_TILE_128x128;
    const bool ak = opA == 'T', bkc = opB != 'T';  // k-contiguous operands
    std::vector<Route> routes;
    routes.reserve(probs.size());
    bool direct = false;
    for (const Prob& p : probs) {
        routes.push_back(route_of(p, segs, ak, bkc));
        direct = direct || routes.back().direct;
    }
    const bool any = tile == DG_GEMM_TILE_AUTO;
    Estimate best;
    best.fits = false;
    // without a problem for the direct-to-LDS kernels that choice is 128x128,
    // and without one to cut the uncut choice is
    const int first = !any ? tile : no_dma || !direct ? (int)DG_GEMM_TILE_128x128 : (int)DG_GEMM_TILE_DIRECT;
    const int end = any ? (int)DG_GEMM_TILES : tile + 1;
    bool cuts = true;
    for (int c = first; c < end; ++c) {
        if (any && c == DG_GEMM_TILE_128x128_WHOLE && !cuts) continue;
        const Estimate x = estimate(probs, routes, segs.size(), c, split_edges);
        if (c == DG_GEMM_TILE_128x128) cuts = x.segs > 0;
        if (x.fits && (!best.fits || x.time < best.time)) {
            best = x;
            tile = c;
        }
    }
    if (!best.fits) return fail(DG_ERR_INVALID, "gemm: output tiles exceed one launch");
    build_lists(ak, bkc, probs, routes, std::move(segs), tile, split_edges, best, out);
    return DG_OK;
}

bool same_lists(const GemmBatch& a, const GemmBatch& b) {
    static_assert(sizeof(Prob) == 64 && sizeof(Seg) == 40, "no padding: compared as bytes");
    auto same = [](const auto& x, const auto& y) {
        return x.size() == y.size() && (x.empty() || memcmp(x.data(), y.data(), x.size() * sizeof(x[0])) == 0);
    };
    return same(a.dma, b.dma) && same(a.dmae, b.dmae) && same(a.gen[0], b.gen[0]) && same(a.gen[1], b.gen[1]) &&
           same(a.gen[2], b.gen[2]) && same(a.segs, b.segs);
}

int persistent_grid(int occ) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus * occ;
}

static constexpr int kOcc[3] = {Cfg128::OCC, Cfg64::OCC, Cfg32::OCC};

// Workgroups of a register-staged launch in XCD ranges.  Little more than one
// or two rounds of resident workgroups: the tiles left over land on the few
// CUs that drain first, several on each.  Workgroups that walk the tiles in
// fixed steps keep them apart (2050^3 on 64x64 tiles, 1.06 rounds: 354 -> 305
// us; 3072^3, 2.25: 853 -> 824).  With more left over, or more rounds, the
// order of completion balances better (4096^3: 1945 us against 1987).
static int xcd_grid(int w, int t) {
    const int slots = persistent_grid(kOcc[w]);
    return w < 2 && t > slots && t < 3 * slots && t % slots <= slots / 4 ? slots : t;
}

int launch_gemm_f64_dev(char opA, char opB, int mode, const GemmBatchDev& b, int* counter, hipStream_t stream) {
    if (mode == DG_GEMM_MODE_PERSISTENT && !counter)
        return fail(DG_ERR_INVALID, "gemm: persistent launch without a work counter");
    // grid of a list's launch: its tiles, or as many workgroups as are resident
    auto grid_of = [&](int tiles, int occ) {
        if (mode != DG_GEMM_MODE_PERSISTENT) return tiles;
        hipLaunchKernelGGL(zero_counter_kernel, dim3(1), dim3(1), 0, stream, counter);
        return std::min(tiles, persistent_grid(occ));
    };
    for (int e = 0; e < 2; ++e) {  // interior list, then edge list
        const bool edge = e == 1;
        const int t0 = edge ? b.tiles_dmae : b.tiles_dma;
        if (t0 <= 0) continue;
        const Prob* dp = edge ? b.dmae : b.dma;
        const int np = edge ? b.ndmae : b.ndma;
        const int grid = grid_of(t0, 2);
        const bool ak = opA == 'T', bkc = opB != 'T';
        if (ak && bkc) launch_dma<true, true>(edge, mode, dp, np, b.segs, t0, grid, counter, stream);
        else if (ak) launch_dma<true, false>(edge, mode, dp, np, b.segs, t0, grid, counter, stream);
        else if (bkc) launch_dma<false, true>(edge, mode, dp, np, b.segs, t0, grid, counter, stream);
        else launch_dma<false, false>(edge, mode, dp, np, b.segs, t0, grid, counter, stream);
        DG_LAUNCH_CHECK();
    }
    for (int w = 0; w < 3; ++w) {  // 128x128 tiles, 64x64, 32x32
        const int t = b.tiles_gen[w];
        if (t <= 0) continue;
        int grid = grid_of(t, kOcc[w]);
        if (mode == DG_GEMM_MODE_XCD) grid = xcd_grid(w, t);
        if (w == 0) launch_cfg<Cfg128>(opA, opB, mode, b.gen[0], b.ngen[0], b.segs, t, grid, counter, stream);
        else if (w == 1) launch_cfg<Cfg64>(opA, opB, mode, b.gen[1], b.ngen[1], b.segs, t, grid, counter, stream);
        else launch_cfg<Cfg32>(opA, opB, mode, b.gen[2], b.ngen[2], b.segs, t, grid, counter, stream);
        DG_LAUNCH_CHECK();
    }
    return DG_OK;
}

int launch_gemm_f64(char opA, char opB, const std::vector<Prob>& probs, std::vector<Seg> segs, hipStream_t stream,
                    int mode) {
    GemmBatch hb;
    int rc = prepare_gemm(opA, opB, probs, std::move(segs), hb);
    if (rc) return rc;
    if (hb.empty()) return DG_OK;
    if (mode == DG_GEMM_MODE_PERSISTENT) mode = DG_GEMM_MODE_XCD;  // needs a counter: plans only
    if (mode == DG_GEMM_MODE_XCD && hb.dma.empty() && hb.dmae.empty() &&
        hb.gen[0].size() + hb.gen[1].size() + hb.gen[2].size() == 1) {
        const int w = hb.gen[0].size() ? 0 : hb.gen[1].size() ? 1 : 2;
        const Prob& p = hb.gen[w][0];
        const int t = hb.tiles_gen[w];
        if (p.nseg == 1 && t <= (1 << 22) && xcd_grid(w, t) == t) {
            const Seg& s = hb.segs[p.seg0];
            if (w == 0) launch_one<Cfg128>(opA, opB, p, s, t, stream);
            else if (w == 1) launch_one<Cfg64>(opA, opB, p, s, t, stream);
            else launch_one<Cfg32>(opA, opB, p, s, t, stream);
            DG_LAUNCH_CHECK();
            return DG_OK;
        }
    }
    GemmBatchDev b;
    TableUseScope uses{stream};  // after the launch below returns
    auto table = [&](const auto& v, auto** dst) -> bool {
        using T = typename std::decay_t<decltype(v)>::value_type;
        *dst = nullptr;
        if (v.empty()) return true;
        *dst = static_cast<const T*>(cached_table(v.data(), v.size() * sizeof(T), stream));
        return *dst != nullptr;
    };
    if (!table(hb.dma, &b.dma) || !table(hb.dmae, &b.dmae) || !table(hb.gen[0], &b.gen[0]) ||
        !table(hb.gen[1], &b.gen[1]) || !table(hb.gen[2], &b.gen[2]) || !table(hb.segs, &b.segs))
        return DG_ERR_ALLOC;
    b.set_counts(hb);
    return launch_gemm_f64_dev(opA, opB, mode, b, nullptr, stream);
}

}  // namespace dg

extern "C" int dg_dgemm(char opA, char opB, int64_t m, int64_t n, int64_t k, double alpha, const double* A,
                        int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc,
                        void* stream) {
    using namespace dg;
    const char oa = norm_op(opA), ob = norm_op(opB);
    if (!oa) return fail(DG_ERR_INVALID, "dg_dgemm: invalid opA '%c'", opA);
    if (!ob) return fail(DG_ERR_INVALID, "dg_dgemm: invalid opB '%c'", opB);
    if (m < 0 || n < 0 || k < 0) return fail(DG_ERR_INVALID, "dg_dgemm: negative dimension");
    const int64_t rowsA = oa == 'N' ? m : k;
    const int64_t rowsB = ob == 'N' ? k : n;
    if (lda < (rowsA > 1 ? rowsA : 1)) return fail(DG_ERR_INVALID, "dg_dgemm: lda %lld < %lld", (long long)lda, (long long)rowsA);
    if (ldb < (rowsB > 1 ? rowsB : 1)) return fail(DG_ERR_INVALID, "dg_dgemm: ldb %lld < %lld", (long long)ldb, (long long)rowsB);
    if (ldc < (m > 1 ? m : 1)) return fail(DG_ERR_INVALID, "dg_dgemm: ldc %lld < %lld", (long long)ldc, (long long)m);
    if (m == 0 || n == 0) return DG_OK;
    int rc = require_device();
    if (rc != DG_OK) return rc;
    hipStream_t st = as_stream(stream);
    if (k == 0 || alpha == 0.0) return launch_scale(m, n, beta, C, ldc, st);
    if (!A || !B || !C) return fail(DG_ERR_INVALID, "dg_dgemm: null matrix pointer");
    std::vector<Seg> segs{Seg{A, B, lda, ldb, k}};
    Prob p{};
    p.m = m; p.n = n; p.c = C; p.ldc = ldc; p.alpha = alpha; p.beta = beta; p.seg0 = 0; p.nseg = 1;
    std::vector<Prob> probs{p};
    return launch_gemm_f64(oa, ob, probs, std::move(segs), st, DG_GEMM_MODE_XCD);
}
