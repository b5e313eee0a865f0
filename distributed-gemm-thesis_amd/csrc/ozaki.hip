// Ozaki split DGEMM on the low-precision matrix cores.
//
// Ozaki, Ogita, Oishi, Rump, "Error-free transformations of matrix
// multiplication by using fast routines of matrix multiplication and its
// applications", Numer. Algorithms 59 (2012); Ootomo, Ozaki, Yokota, "DGEMM on
// integer matrix multiplication unit", IJHPCA (2024).
//
//   1. e_i = frexp exponent of max_k |op(A)_ik| (max < 2^e_i), f_j likewise
//      for the columns of op(B).
//   2. r_0 = x * 2^-e, d_t = trunc(r_{t-1} * 2^b), r_t = r_{t-1} * 2^b - d_t
//      for t = 1..s, all exact in FP64: INT8 digits carry b = 7 bits
//      (|d| <= 127), BF16 digits b = 5 bits (|d| <= 31, exact in bf16).
//   3. For level l = 2..s+1 and t = 1..l-1 the exact integer product
//      A_t B_{l-t} is accumulated on the matrix cores (INT8 -> INT32,
//      BF16 -> FP32 below 2^24, both exact); the 32-bit accumulator is added
//      into an FP64 partial sum W as ldexp(acc, -b*l) whenever it could
//      overflow next (the host computes the flush points) and at the end of
//      each level.
//   4. C = alpha * ldexp(W, e_i + f_j) + beta * C, without fused multiply-add
//      so that the CPU oracle reproduces every bit.
//
// Slices are stored k-contiguous, [t][row][Kp] with rows padded to 256 and K
// padded to 128 bytes with zeros, so the product kernels have no edge cases
// until the final store.  Each run of products between two flushes (a
// group) runs as one long-K product through the scheme II pipeline
// (oz_plane_kernel: 128-byte k-steps, described with crt_gemm_kernel) into a
// 32-bit plane per group (INT32 sums, or the FP32 sums of BF16 slices), and
// oz_combine_kernel adds the planes into the FP64 partial sums W (workspace)
// in schedule order, with the operations a flush inside the product loop
// would make.
#include "dg_internal.hpp"

#include <algorithm>
#include <type_traits>

// Every FP64 operation of the recombination is rounded on its own (no fused
// multiply-add), matching the CPU oracle bit for bit.
#pragma clang fp contract(off)

namespace dg {

namespace {

typedef int iv4 __attribute__((ext_vector_type(4)));
typedef float fv4 __attribute__((ext_vector_type(4)));
typedef double dv4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef double pdv2 __attribute__((ext_vector_type(2)));
typedef pdv2 udv2 __attribute__((aligned(8)));  // a pair at any alignment
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int PAD = 256;     // row padding of the slices and residues (a multiple of BM and BN)
constexpr int KSB = 128;     // K padding granule of the slices and residues, bytes
// Product kernels: BM x BN output tiles of 8 waves of WM x WN (FM x FN
// MFMA tiles of 16x16), one workgroup per CU.
constexpr int BM = 256, BN = 256;
constexpr int WM = 128, WN = 64;
constexpr int OCC = 1;
constexpr int NW = (BM / WM) * (BN / WN);  // waves per workgroup
constexpr int CNT = NW * 64;               // threads per workgroup
constexpr int FM = WM / 16, FN = WN / 16;  // 16x16 MFMA tiles per wave
static_assert(PAD % BM == 0 && PAD % BN == 0, "slice rows are padded to whole tiles");
constexpr int NT = 256;
constexpr int GROUP_M = 4;

__device__ __forceinline__ int xcd_remap(int bid, int total) {
    constexpr int X = 8;
    const int q = total / X, r = total % X;
    const int x = bid % X, slot = bid / X;
    return x * q + min(x, r) + slot;
}

// One product of the level schedule: slices (t, u) over k range [k0, k0+klen)
// of the padded K, then optionally flush the 32-bit accumulator with weight
// 2^-(bits*level).
struct OzSeg {
    int32_t t, u;       // 0-based slice indices
    int32_t k0, klen;   // in elements, multiples of the k-step
    int32_t level;      // t + u + 2 (1-based level)
    int32_t flush;      // 0: keep accumulating; 1: add into W; 2: first flush (W = x);
                        // 3: last flush (C = alpha*ldexp(W + x, e+f) + beta*C); 4: first and last
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    // gfx9 s_waitcnt: vmcnt in bits 3:0 and 15:14; expcnt and lgkmcnt left at their maxima
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void gvoid_t;

// A pointer the caller knows to be equal across the wave, in scalar
// registers (a uniform base plus a 32-bit lane offset lets a load take the
// scalar-base address form instead of a 64-bit address per lane).
__device__ __forceinline__ const int8_t* wave_uniform(const int8_t* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const int8_t*>(((uint64_t)hi << 32) | lo);
}

// Output tile of workgroup slot `bid` among `tiles`: XCD-aware, GROUP_M tile
// rows sweep the tile columns together.  With 256x256 tiles and 32 resident
// workgroups per XCD, GROUP_M = 4 gives each XCD a 4 x 8 block of tiles (12
// distinct operand slices per k-step, as for 8 x 4) while the A panels all
// XCDs revisit stay at half the size, which keeps them in the last-level
// cache (measured on the 16384^3 CRT product: 4.8% faster than 8 x 4).
template <int TILE>
__device__ __forceinline__ void tile_origin(int bid, int tiles, int tiles_m, int tiles_n, int64_t& m0, int64_t& n0) {
    const int tile = xcd_remap(bid, tiles);
    const int per_group = GROUP_M * tiles_n;
    const int group = tile / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = tile - group * per_group;
    m0 = (int64_t)(first_m + in_group % gsize) * TILE;
    n0 = (int64_t)(in_group / gsize) * TILE;
}

// ------------------------------------------------------------ Ozaki scheme II
// Ozaki, Uchino, Imamura, "Ozaki Scheme II: A GEMM-oriented emulation of
// floating-point matrix multiplication using an integer modular technique"
// (2025).  A' = rint(op(A)_ik * 2^sigma_i) (rounded to nearest, which
// halves the RMS scaling error of truncation) and B' = rint(op(B)_kj *
// 2^tau_j) are integers; the shifts follow the paper's Cauchy-Schwarz bound
// (its fast mode): every scaled line has 2-norm <= 2^Q before rounding, with
// Q the largest such that 2^(2Q) + ceil(sqrt(k)) 2^Q + k <= P/4
// (P = prod p_t), so |V| = |A'B'| <= P/4.  The norm bound is an exact integer
// sum (crt_bound_term), so the shifts do not depend on summation order; a
// line whose norm is far below sqrt(k) times its largest entry (wide-ranging
// data) gets more bits than the per-entry bound would give it, up to 53.
// V is computed modulo N pairwise coprime moduli p_t <= 256 (one INT8 GEMM
// each, residues balanced into [-128, 127]) and rebuilt exactly by the
// Chinese remainder theorem, V = sum_t x_t (P/p_t) mod P, balanced.
// Shifts are stored as e' = Q - sigma (e'_i, f'_j), and
// C = alpha * ldexp(double(V), e'_i + f'_j - 2Q) + beta*C with double(V)
// correctly rounded.

constexpr int kMaxModuli = 16;
// Pairwise coprime: 2^8, 3*5*17, 11*23, 13*19, 7*31 and primes.
__constant__ int c_moduli[kMaxModuli] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193};


// Direct CRT: V = (sum_t x_t * M_t) mod P with M_t = P / p_t and
// x_t = r_t * (M_t^-1 mod p_t) mod p_t, then the balanced representative.
struct CrtTables {
    int32_t n;                          // moduli in use
    int32_t cinv[kMaxModuli];           // M_t^-1 mod p_t
    double mt[kMaxModuli][3];           // M_t in 40-bit limbs (as doubles), least significant first
    double Pl[3];                       // P = prod p_t in 40-bit limbs (as doubles), least significant first
    double invPd;                       // 1 / fl(P) rounded to double
};

// p_t as a constant expression, so that x % crt_modulus(t) in an unrolled
// loop compiles to a multiply-shift.
__host__ __device__ constexpr int crt_modulus(int t) {
    return t == 0 ? 256 : t == 1 ? 255 : t == 2 ? 253 : t == 3 ? 251 : t == 4 ? 247 : t == 5 ? 241 : t == 6 ? 239
         : t == 7 ? 233 : t == 8 ? 229 : t == 9 ? 227 : t == 10 ? 223 : t == 11 ? 217 : t == 12 ? 211
         : t == 13 ? 199 : t == 14 ? 197 : 193;
}

// One operand of a scheme II preparation: lines x[i*rs + k*ks].
struct CrtSide {
    const double* x;
    int64_t rows, rs, ks;
    int64_t rows_p;
    int8_t* out;        // residues, planes rows_p * Kp apart
    int32_t* e;         // line exponents, rows_p of them
    uint64_t* part;     // scan words, [chunk][rows], in the place of the residues (written after them)
    uint32_t nkt, nrt;  // k and row tiles of the residue pass
};

// Balanced residues of A' = rint(op(X)(row, k) * 2^(q - e_row)) for every
// modulus, [t][row][Kp] int8 (zeros in the padding).  A workgroup stages a
// tile of op(X) through LDS, loaded along whichever direction is contiguous
// in memory (16.5 KB, so eight workgroups share a CU and the load and store
// phases of different workgroups overlap); each thread then turns 8
// consecutive k of one row into one 8-byte store per modulus, so a wave
// writes whole 128-byte lines.  One FP64 operation and one packed 16-bit one
// per two elements make a residue (below), which leaves the pass bound by
// its memory traffic, two thirds of it stores to as many places as there are
// moduli.  8192^2 and 14 moduli (1.48 GB): contiguous lines 285 -> 273 us from
// tiles of 16 x 128 to 8 x 256 (straight from registers, without LDS: 297),
// strided lines 335 -> 285 us from nontemporal to plain stores (plain ones
// cost the contiguous form 25 us).
constexpr int RT_R = 16, RT_K = 128;  // tile of strided lines
constexpr int RC_R = 8, RC_K = 256;   // tile of lines contiguous in k

// fl(1/p) of each modulus, passed as a kernel argument so that it sits in
// scalar registers (a VOP3 FMA takes it directly; gfx9 VOP3 encodings take no
// 64-bit literals).
struct ResidueConsts {
    double inv_p[kMaxModuli];
};

// Tile order of the residue pass (workgroup -> row tile, k tile): lines
// contiguous in k walk each tile row along k; strided lines go in groups of
// RT_KG k tiles, row tiles within a group, so that the workgroups in flight
// read long runs of each column of op(X) and still write 2 KB runs of each
// residue row.
constexpr uint32_t RT_KG = 16;

template <int NMOD>
__global__ __launch_bounds__(256) void crt_residue_kernel(CrtSide A, CrtSide B, uint32_t na, int64_t K, int q,
                                                          int64_t Kp, ResidueConsts rc) {
    const bool first_side = blockIdx.x < na;
    const CrtSide o = first_side ? A : B;
    const uint32_t block = first_side ? blockIdx.x : blockIdx.x - na;
    const double* __restrict__ x = o.x;
    const int64_t rows = o.rows, rs = o.rs, ks = o.ks, slice_bytes = o.rows_p * Kp;
    const uint32_t nkt = o.nkt, nrt = o.nrt;
    __shared__ double tile[RT_R * (RT_K + 1)];
    static_assert(RC_R * (RC_K + 1) <= RT_R * (RT_K + 1), "either tile fits");
    constexpr int KPT = 8;
    const int t = threadIdx.x;
    int64_t r, k0;
    const double* row;  // the thread's eight k in the tile
    double w[KPT];
    // Eight loads per thread, all issued before the first wait: addresses
    // outside op(X) are clamped onto its last row / k (in bounds) and the
    // loaded value replaced by zero.  op(X) is read for the last time here.
    if (ks == 1) {
        const uint32_t rt = block / nkt;
        const int64_t r0 = (int64_t)rt * RC_R;
        k0 = (int64_t)(block - rt * nkt) * RC_K;
        const int64_t k = k0 + t;
        const int64_t kc = k < K ? k : K - 1;
#pragma unroll
        for (int i = 0; i < RC_R; ++i)
            w[i] = __builtin_nontemporal_load(x + (r0 + i < rows ? r0 + i : rows - 1) * rs + kc);
#pragma unroll
        for (int i = 0; i < RC_R; ++i) tile[i * (RC_K + 1) + t] = k < K ? w[i] : 0.0;
        r = r0 + t / (RC_K / KPT);
        k0 += KPT * (t % (RC_K / KPT));
        row = tile + t / (RC_K / KPT) * (RC_K + 1) + KPT * (t % (RC_K / KPT));
    } else {
        const uint32_t grp = block / (RT_KG * nrt);
        const uint32_t first = grp * RT_KG;
        const uint32_t gk = nkt - first < RT_KG ? nkt - first : RT_KG;
        const uint32_t in = block - grp * RT_KG * nrt;
        const uint32_t rt = in / gk;
        const int64_t r0 = (int64_t)rt * RT_R;
        k0 = (int64_t)(first + (in - rt * gk)) * RT_K;
        const int64_t lr = r0 + t % RT_R;
        const double* xr = x + (lr < rows ? lr : rows - 1) * rs;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const int64_t k = k0 + t / RT_R + (256 / RT_R) * i;
            w[i] = __builtin_nontemporal_load(xr + (k < K ? k : K - 1) * ks);
        }
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const int kk = t / RT_R + (256 / RT_R) * i;
            tile[t % RT_R * (RT_K + 1) + kk] = k0 + kk < K ? w[i] : 0.0;
        }
        r = r0 + t / (RT_K / KPT);
        k0 += KPT * (t % (RT_K / KPT));
        row = tile + t / (RT_K / KPT) * (RT_K + 1) + KPT * (t % (RT_K / KPT));
    }
    __syncthreads();
    if (k0 >= Kp) return;  // Kp is a multiple of 128
    // |a| <= 2^53 and |fl(1/p) - 1/p| <= 2^-61, so t = fma(a, fl(1/p), 1.5 2^52)
    // is 1.5 2^52 + q with an integer q within 1/2 + 2^-8 of a/p, and r = a - q p
    // is at most p/2 + p/256 in magnitude: at most 127 for p <= 253, for p = 255
    // too (fl(1/255) is within 2^-63), and 128 = -128 (mod 256) for p = 256.  Its
    // low byte, which is r, needs a and q modulo 256 only: a + q (256 - p) on the
    // low half words of t, two elements at a time.  Not-a-numbers and infinities
    // count as zeros.
    double a[KPT];
    u16x2 ab[KPT / 2];
    const int sh = r < rows ? q - o.e[r] : 0;
#pragma unroll
    for (int c = 0; c < KPT; ++c) {
        const double y = rint(ldexp(row[c], sh));
        a[c] = r < rows && fabs(y) <= 0x1p53 ? y : 0.0;
        const double f = a[c] * 0x1p-8;
        ab[c / 2][c % 2] = (unsigned short)(int)((f - floor(f)) * 256.0);
    }
    int8_t* dst = o.out + r * Kp + k0;
#pragma unroll
    for (int m = 0; m < NMOD; ++m) {
        uint32_t rb[KPT / 2];
#pragma unroll
        for (int c = 0; c < KPT / 2; ++c) {
            if (m == 0) {  // p = 256
                rb[c] = __builtin_bit_cast(uint32_t, ab[c]);
                continue;
            }
            const uint32_t t0 = (uint32_t)__double_as_longlong(fma(a[2 * c], rc.inv_p[m], 0x1.8p52));
            const uint32_t t1 = (uint32_t)__double_as_longlong(fma(a[2 * c + 1], rc.inv_p[m], 0x1.8p52));
            const u16x2 qw = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(t1, t0, 0x05040100u));
            const unsigned short d = (unsigned short)(256 - crt_modulus(m));
            rb[c] = __builtin_bit_cast(uint32_t, qw * u16x2{d, d} + ab[c]);
        }
        const uint32_t w0 = __builtin_amdgcn_perm(rb[1], rb[0], 0x06040200u);
        const uint32_t w1 = __builtin_amdgcn_perm(rb[3], rb[2], 0x06040200u);
        u32x2* to = reinterpret_cast<u32x2*>(dst + m * slice_bytes);
        if (ks == 1)
            __builtin_nontemporal_store(u32x2{w0, w1}, to);
        else
            *to = u32x2{w0, w1};
    }
}

struct CrtArgs {
    const int8_t* a;     // residues of A', [N][Mp][Kp]
    const int8_t* b;     // residues of B', [N][Np][Kp]
    uint8_t* res;        // CRT digits x_t of V, [N][Np][Mp] (column-major per modulus, planes res_plane apart)
    int64_t Mp, Np, Kp, res_plane;
    int64_t a_slice, b_slice;
    int32_t tiles_m, tiles_n, nmod;
    int32_t cinv[kMaxModuli];  // (P / p_t)^-1 mod p_t
};

// The scheme II product pipeline moves 128-byte k-steps: one
// global_load_lds_dwordx4 of a wave covers 8 rows x 128 bytes, so every L2
// request is a whole 128-byte line (64-byte half lines cost the same request
// slot and halve the operand stream).  A step's A rows and B rows each fill
// a 32 KB slot; five slots (160 KB) form a ring in which A_0 B_0 A_1 B_1 ...
// take consecutive slots.  Within a row, 16-byte chunk c sits at position
// c ^ (row % 8): the fragment reads (lane l: row l % 16, chunk 4h + l / 16 of
// half-step h) then run at the full LDS rate.  A step is two MFMA half-steps
// of 64 bytes; the barrier sits between them: it publishes step s+1 (A_{s+1}
// loaded two steps earlier, B_{s+1} one step earlier) and releases the slots
// of step s, whose fragments are all in registers by then, to B_{s+2} and
// A_{s+3}.  The second half-step's MFMAs run while the fragments of the
// first half of step s+1 are read, and the first half-step's while those of
// the second half are read.
constexpr int CK2 = 128;                  // bytes per scheme II k-step
constexpr int CSLOT = BM * CK2;           // one operand's rows of one step
constexpr int NSLOT = 5;
constexpr size_t kCrtLds = (size_t)NSLOT * CSLOT;
static_assert(BM == BN && BM / NW == 32, "scheme II loader: 32 rows per wave and operand");

__device__ __forceinline__ int next_slot(int x) { return x + 1 == NSLOT ? 0 : x + 1; }

// This wave's 32 rows of one operand for k-step s into `slot`; g (uniform
// across the wave) points at the wave's first row, loff is the lane's
// offset to its row and chunk, rows `ld` bytes apart.  A uniform base and a
// 32-bit lane offset let every load take the scalar-base address form.
__device__ __forceinline__ void crt_issue(int8_t* lds, int slot, int wave, const int8_t* g, uint32_t loff, int64_t s,
                                          int64_t ld) {
    int8_t* d = lds + slot * CSLOT + wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_global_load_lds((gvoid_t*)(wave_uniform(g + s * CK2 + (int64_t)(8 * i) * ld) + loff),
                                         (lds_void_t*)(d + 1024 * i), 16, 0, 0);
}

// One 64-byte MFMA of the pipeline: 16x16 INT8 products summed in INT32
// (iv4 accumulators) or BF16 products summed in FP32 (fv4 accumulators, for
// the BF16 slices of scheme I).  Either way a lane's A and B operands are 16
// bytes of one row, so the LDS layout is the same.
__device__ __forceinline__ void mfma64(iv4& acc, const iv4& a, const iv4& b) {
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ void mfma64(fv4& acc, const iv4& a, const iv4& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), acc, 0, 0, 0);
}

// One MFMA half-step on fa / cb, reading the fragments of the following
// half-step meanwhile: fa[i] right after its last use, B into nb.
template <class ACC, int M, int N>
__device__ __forceinline__ void crt_half(ACC (&acc)[M][N], iv4 (&fa)[M], const iv4 (&cb)[N], iv4 (&nb)[N],
                                         const int8_t* nas, const int8_t* nbs) {
#pragma unroll
    for (int i = 0; i < M; ++i) {
#pragma unroll
        for (int j = 0; j < N; ++j) mfma64(acc[i][j], fa[i], cb[j]);
        if (i == 0) {
#pragma unroll
            for (int j = 0; j < N; ++j) nb[j] = *reinterpret_cast<const iv4*>(nbs + 2048 * j);
        }
        fa[i] = *reinterpret_cast<const iv4*>(nas + 2048 * i);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, N, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, N + 1, 0);
#pragma unroll
    for (int g = 1; g < M; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, N, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
}

// crt_half that also issues this wave's loads of B step sb (into slot_b)
// and A step sa (into slot_a), one global_load_lds after each group of FN
// MFMAs:
// issued back to back, the eight 1 KB loads of every wave queue at the
// vector memory unit while the matrix cores wait.
template <class ACC>
__device__ __forceinline__ void crt_half_ld(ACC (&acc)[FM][FN], iv4 (&fa)[FM], const iv4 (&cb)[FN], iv4 (&nb)[FN],
                                            const int8_t* nas, const int8_t* nbs, int8_t* lds, int slot_b,
                                            int slot_a, int wave, const int8_t* gb, const int8_t* ga, uint32_t loff,
                                            int64_t sb, int64_t sa, int64_t ld) {
    static_assert(FM == 8, "one load per MFMA group: four of B, then four of A");
    int8_t* db = lds + slot_b * CSLOT + wave * 4096;
    int8_t* da = lds + slot_a * CSLOT + wave * 4096;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) mfma64(acc[i][j], fa[i], cb[j]);
        if (i == 0) {
#pragma unroll
            for (int j = 0; j < FN; ++j) nb[j] = *reinterpret_cast<const iv4*>(nbs + 2048 * j);
        }
        fa[i] = *reinterpret_cast<const iv4*>(nas + 2048 * i);
        if (i < 4)
            __builtin_amdgcn_global_load_lds((gvoid_t*)(wave_uniform(gb + sb * CK2 + (int64_t)(8 * i) * ld) + loff),
                                             (lds_void_t*)(db + 1024 * i), 16, 0, 0);
        else
            __builtin_amdgcn_global_load_lds(
                (gvoid_t*)(wave_uniform(ga + sa * CK2 + (int64_t)(8 * (i - 4)) * ld) + loff),
                (lds_void_t*)(da + 1024 * (i - 4)), 16, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, FN, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, FN + 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
#pragma unroll
    for (int g = 1; g < FM; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, FN, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
}

// The digits of a wave's sums: acc[i][j][v] = V_t(m0 + 16i + v, n0 + 16j),
// four consecutive rows of one column, stored as one 32-bit word of digits.
// x = acc * cinv is exact (|x| < 2^39) and floor(fl(x fl(1/p) + 2^-10)) is
// floor(x/p) exactly (the estimate errs by < 2^-20 and the fractional
// part of x/p lies in [0, 1 - 1/p]), so x - p floor(x/p) is the digit.
template <int M, int N>
__device__ __forceinline__ void store_digits(const iv4 (&acc)[M][N], const CrtArgs& g, int tmod, int64_t m0,
                                             int64_t n0) {
    const int p = c_moduli[tmod];
    const double pd = p, inv_p = 1.0 / p, cinv = g.cinv[tmod];
    uint8_t* out = g.res + (int64_t)tmod * g.res_plane;
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int i = 0; i < M; ++i) {
            uint32_t w = 0;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double x = (double)acc[i][j][v] * cinv;
                const double qd = floor(fma(x, inv_p, 0x1p-10));
                w |= (uint32_t)(int)fma(-qd, pd, x) << (8 * v);
            }
            *reinterpret_cast<uint32_t*>(out + (n0 + 16 * j) * g.Mp + m0 + 16 * i) = w;
        }
}

// ------------------------------------------------------------ 128 x 128 tiles
// The same pipeline for products with too few 256 x 256 tiles to fill the
// chip: four waves of 64 x 64, a ring of five whole steps (160 KB, one
// workgroup per CU).  A step's MFMAs take a quarter of the time here, so the
// loads run five steps ahead instead of two and a half.
constexpr int ST = 128, SNW = 4, SCNT = SNW * 64, SFM = 4, SFN = 4, SDEPTH = 5;
constexpr int SSTEP = 2 * ST * CK2;  // A's and B's rows of one step
static_assert(SDEPTH * SSTEP == (int)kCrtLds, "the ring fills the LDS");

// Sums of k-steps 0..last into acc; a_at(s), b_at(s): this wave's 32 rows of
// step s, `ld` bytes apart (steps past the end clamped to the last one).
template <class ACC, class At, class Bt>
__device__ __forceinline__ void small_product(ACC (&acc)[SFM][SFN], int8_t* lds, const At& a_at, const Bt& b_at,
                                              uint32_t last, int64_t ld, int wave, int lane, int wm, int wn) {
    const uint32_t loff = (uint32_t)((lane >> 3) * ld + 16 * ((lane & 7) ^ (lane >> 3)));
    const int lr = lane & 15, lg = lane >> 4;
    const int a0 = (wm + lr) * CK2 + 16 * (lg ^ (lr & 7)), a1 = (wm + lr) * CK2 + 16 * ((4 + lg) ^ (lr & 7));
    const int ab = ST * CK2 + (wn - wm) * CK2;  // from A's fragment rows to B's
    const auto load = [&](const int8_t* g, int8_t* d, int i) {
        __builtin_amdgcn_global_load_lds((gvoid_t*)(wave_uniform(g + (int64_t)(8 * i) * ld) + loff),
                                         (lds_void_t*)(d + wave * 4096 + 1024 * i), 16, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < SDEPTH; ++s) {
        const int8_t *ga = a_at(s), *gb = b_at(s);
#pragma unroll
        for (int i = 0; i < 4; ++i) load(ga, lds + s * SSTEP, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) load(gb, lds + s * SSTEP + ST * CK2, i);
    }
    wait_vmcnt<8 * (SDEPTH - 1)>();  // step 0 landed
    __builtin_amdgcn_s_barrier();
    iv4 fa[SFM], cb[SFN], nb[SFN];
#pragma unroll
    for (int j = 0; j < SFN; ++j) cb[j] = *reinterpret_cast<const iv4*>(lds + a0 + ab + 2048 * j);
#pragma unroll
    for (int i = 0; i < SFM; ++i) fa[i] = *reinterpret_cast<const iv4*>(lds + a0 + 2048 * i);
    int8_t* cur = lds;  // ring position of step s
    for (uint32_t s = 0; s < last; ++s) {
        int8_t* next = cur == lds + (SDEPTH - 1) * SSTEP ? lds : cur + SSTEP;
        crt_half(acc, fa, cb, nb, cur + a1, cur + a1 + ab);
        // this wave's reads of step s are done; its part of step s + 1 landed
        // with three steps pending
        __builtin_amdgcn_s_waitcnt((0xF) | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0)
        wait_vmcnt<8 * (SDEPTH - 2)>();
        __builtin_amdgcn_s_barrier();
        const int8_t *ga = a_at(s + SDEPTH), *gb = b_at(s + SDEPTH);
#pragma unroll
        for (int i = 0; i < SFM; ++i) {
#pragma unroll
            for (int j = 0; j < SFN; ++j) mfma64(acc[i][j], fa[i], nb[j]);
            if (i == 0) {
#pragma unroll
                for (int j = 0; j < SFN; ++j) cb[j] = *reinterpret_cast<const iv4*>(next + a0 + ab + 2048 * j);
            }
            fa[i] = *reinterpret_cast<const iv4*>(next + a0 + 2048 * i);
            load(ga, cur, i);
            load(gb, cur + ST * CK2, i);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, SFN, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, SFN + 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
#pragma unroll
        for (int i = 1; i < SFM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, SFN, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        }
        cur = next;
    }
    // last step: no loads; the reads of a following one are in bounds and unused
    int8_t* next = cur == lds + (SDEPTH - 1) * SSTEP ? lds : cur + SSTEP;
    crt_half(acc, fa, cb, nb, cur + a1, cur + a1 + ab);
    crt_half(acc, fa, nb, cb, next + a0, next + a0 + ab);
    wait_vmcnt<0>();  // the loads past the end land before the workgroup's LDS is released
}

__global__ __launch_bounds__(SCNT, 2) void crt_gemm_small_kernel(CrtArgs g) {
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
    const int tiles = g.tiles_m * g.tiles_n;
    const int tmod = blockIdx.x / tiles;
    int64_t m0, n0;
    tile_origin<ST>(blockIdx.x - tmod * tiles, tiles, g.tiles_m, g.tiles_n, m0, n0);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int8_t* ga = g.a + tmod * g.a_slice + (m0 + 32 * wave) * g.Kp;
    const int8_t* gb = g.b + tmod * g.b_slice + (n0 + 32 * wave) * g.Kp;
    const uint32_t last = (uint32_t)(g.Kp / CK2) - 1;
    iv4 acc[SFM][SFN];
#pragma unroll
    for (int i = 0; i < SFM; ++i)
#pragma unroll
        for (int j = 0; j < SFN; ++j) acc[i][j] = iv4{0, 0, 0, 0};
    small_product(
        acc, lds, [&](uint32_t s) { return ga + (int64_t)(s < last ? s : last) * CK2; },
        [&](uint32_t s) { return gb + (int64_t)(s < last ? s : last) * CK2; }, last, g.Kp, wave, lane, wm, wn);
    store_digits(acc, g, tmod, m0 + wm + 4 * (lane >> 4), n0 + wn + (lane & 15));
}

// One INT8 GEMM per modulus in one launch: workgroup b computes tile
// b % tiles of modulus b / tiles and stores the CRT digit
// x_t = ((A'_t B'_t) mod p_t) * ((P / p_t)^-1 mod p_t) mod p_t as a byte.
__global__ __launch_bounds__(CNT, OCC) void crt_gemm_kernel(CrtArgs g) {
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
    const int tiles = g.tiles_m * g.tiles_n;
    const int tmod = blockIdx.x / tiles;
    int64_t m0, n0;
    tile_origin<BM>(blockIdx.x - tmod * tiles, tiles, g.tiles_m, g.tiles_n, m0, n0);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave / (BN / WN)) * WM;
    const int wn = (wave % (BN / WN)) * WN;
    const int lr = lane & 15;
    const int lg = lane >> 4;

    // loader: lane -> row lane / 8 of an 8-row group, position lane % 8
    // holding global chunk (lane % 8) ^ (row % 8)
    const int lrow = lane >> 3;
    const int lchunk = (lane & 7) ^ lrow;
    const int8_t* ga = g.a + tmod * g.a_slice + (m0 + 32 * wave) * g.Kp;
    const int8_t* gb = g.b + tmod * g.b_slice + (n0 + 32 * wave) * g.Kp;
    const uint32_t loff = (uint32_t)(lrow * g.Kp + 16 * lchunk);
    const int roff0 = lr * CK2 + 16 * (lg ^ (lr & 7));
    const int roff1 = lr * CK2 + 16 * ((4 + lg) ^ (lr & 7));

    iv4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = iv4{0, 0, 0, 0};

    const int64_t nk = g.Kp / CK2;  // >= 1
    // Every step issues the same loads, so that every wait is the same: a
    // load of a step past the end reloads the last step into a slot that is
    // free and never read again (its data unused).
    const auto clamp = [nk](int64_t s) { return s < nk ? s : nk - 1; };
    // prologue: A_0 B_0 A_1 B_1 A_2 into slots 0..4
    crt_issue(lds, 0, wave, ga, loff, 0, g.Kp);
    crt_issue(lds, 1, wave, gb, loff, 0, g.Kp);
    crt_issue(lds, 2, wave, ga, loff, clamp(1), g.Kp);
    crt_issue(lds, 3, wave, gb, loff, clamp(1), g.Kp);
    crt_issue(lds, 4, wave, ga, loff, clamp(2), g.Kp);
    int isl = 0;
    // step 0 landed: at most A_1 B_1 A_2 (4 loads each) pending
    wait_vmcnt<12>();
    __builtin_amdgcn_s_barrier();
    int csl = 0;  // slot of A_s; B_s in the next one
    iv4 fa[FM], cb[FN], nb[FN];
    {
        const int8_t* as = lds + wm * CK2 + roff0;
        const int8_t* bs = lds + CSLOT + wn * CK2 + roff0;
#pragma unroll
        for (int j = 0; j < FN; ++j) cb[j] = *reinterpret_cast<const iv4*>(bs + 2048 * j);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const iv4*>(as + 2048 * i);
    }
    for (int64_t s = 0; s + 1 < nk; ++s) {
        const int bsl = next_slot(csl), asl1 = next_slot(bsl), bsl1 = next_slot(asl1);
        // first half of step s; fragments of its second half read meanwhile
        crt_half(acc, fa, cb, nb, lds + csl * CSLOT + wm * CK2 + roff1, lds + bsl * CSLOT + wn * CK2 + roff1);
        // every fragment of step s is in registers once this wave's LDS reads
        // are done; A_{s+1} and B_{s+1} landed with at most A_{s+2} pending
        __builtin_amdgcn_s_waitcnt((0xF) | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0)
        wait_vmcnt<4>();
        __builtin_amdgcn_s_barrier();
        // second half of step s, fragments of the first half of step s+1 read
        // meanwhile, B_{s+2} and A_{s+3} issued among its MFMAs into the slots
        // of step s
        const int sb = isl, sa = next_slot(isl);
        isl = next_slot(sa);
        crt_half_ld(acc, fa, nb, cb, lds + asl1 * CSLOT + wm * CK2 + roff0, lds + bsl1 * CSLOT + wn * CK2 + roff0,
                    lds, sb, sa, wave, gb, ga, loff, clamp(s + 2), clamp(s + 3), g.Kp);
        csl = asl1;
    }
    {
        // last step: no loads; the second half's reads of a following step
        // are in bounds and unused
        const int bsl = next_slot(csl), asl1 = next_slot(bsl), bsl1 = next_slot(asl1);
        crt_half(acc, fa, cb, nb, lds + csl * CSLOT + wm * CK2 + roff1, lds + bsl * CSLOT + wn * CK2 + roff1);
        crt_half(acc, fa, nb, cb, lds + asl1 * CSLOT + wm * CK2 + roff0, lds + bsl1 * CSLOT + wn * CK2 + roff0);
    }
    wait_vmcnt<0>();  // the reloads past the end land before the workgroup's LDS is released
    store_digits(acc, g, tmod, m0 + wm + 4 * lg, n0 + wn + lr);
}

// ---------------------------------------------- scheme I on the scheme II pipeline
// The products of scheme I between two flushes (a group: slices t0 + p of A
// against slices u0 - p of B for p < count, one level, one k range) add up
// to one long-K product, so a group's k-steps run back to back through the
// scheme II pipeline above.  Workgroup b computes tile b % tiles of the
// launch's job b / tiles (a group) and stores its 32-bit sums (INT32 for
// INT8 slices, FP32 for BF16 slices) as a plane, [Np][Mp] column-major;
// oz_combine_kernel then adds the planes into FP64 in group order.  One
// workgroup has a CU to itself, a launch has a few hundred of them and the
// groups differ up to 8-fold in length, so the jobs run longest first: in
// schedule order (counts 1, 2, ... 8) the longest tiles began last and left
// most CUs idle for their whole length (8 INT8 slices of 3000 x 2000 x 5000:
// 1115 us a call, longest first 978; 11 BF16 slices of 2048^3: 972 and 833).
struct OzGroup {
    int32_t t0, u0;   // 0-based slices of the first product
    int32_t count;    // products
    int32_t level;    // t + u + 2 (t, u 1-based) of every product
    int32_t kb;       // byte offset of the k range within a slice row
    FastDiv nks;      // 128-byte k-steps per product (nks.d), as a divisor
    int32_t plane;    // plane of its launch that takes the sums
};

struct OzPlaneArgs {
    const int8_t* a;             // A slices, [s][Mp] rows of rb bytes
    const int8_t* b;             // B slices, [s][Np] rows of rb bytes
    int32_t* planes;             // one [Np][Mp] plane per group of the launch
    const OzGroup* jobs;         // the launch's groups, longest first
    int32_t tiles_m, tiles_n;
    int64_t Mp, rb;
    int64_t a_slice, b_slice;    // bytes per slice
    int64_t plane;               // elements per plane
};

// This wave's rows of k-step s of a group (clamped to its last step, for
// the pipeline's reloads past the end): product p = s / nks, step s % nks
// within it, the product's slice `stride` bytes from the previous one's.
// Branch-free scalar arithmetic, so the loop body stays one basic block.
__device__ __forceinline__ const int8_t* group_step(const int8_t* first, int64_t stride, uint32_t s, uint32_t last,
                                                    const FastDiv& nks) {
    const uint32_t sc = s < last ? s : last;
    const uint32_t p = fdiv(sc, nks);
    return first + (int64_t)p * stride + (int64_t)(sc - p * nks.d) * CK2;
}

template <bool BF16>
__global__ __launch_bounds__(CNT, OCC) void oz_plane_kernel(OzPlaneArgs g) {
    typedef typename std::conditional<BF16, fv4, iv4>::type acc_t;
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
    const int tiles = g.tiles_m * g.tiles_n;
    const int gi = blockIdx.x / tiles;
    int64_t m0, n0;
    tile_origin<BM>(blockIdx.x - gi * tiles, tiles, g.tiles_m, g.tiles_n, m0, n0);
    const OzGroup gr = g.jobs[gi];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave / (BN / WN)) * WM;
    const int wn = (wave % (BN / WN)) * WN;
    const int lr = lane & 15;
    const int lg = lane >> 4;
    const int lrow = lane >> 3;
    const int lchunk = (lane & 7) ^ lrow;
    const uint32_t loff = (uint32_t)(lrow * g.rb + 16 * lchunk);
    const int roff0 = lr * CK2 + 16 * (lg ^ (lr & 7));
    const int roff1 = lr * CK2 + 16 * ((4 + lg) ^ (lr & 7));

    const uint32_t last = (uint32_t)gr.count * gr.nks.d - 1;  // the group's last k-step
    const int8_t* ga = g.a + gr.t0 * g.a_slice + (m0 + 32 * wave) * g.rb + gr.kb;
    const int8_t* gb = g.b + gr.u0 * g.b_slice + (n0 + 32 * wave) * g.rb + gr.kb;
    const auto a_at = [&](uint32_t s) { return group_step(ga, g.a_slice, s, last, gr.nks); };
    const auto b_at = [&](uint32_t s) { return group_step(gb, -g.b_slice, s, last, gr.nks); };

    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

    // prologue: A_0 B_0 A_1 B_1 A_2 into slots 0..4, as in crt_gemm_kernel
    crt_issue(lds, 0, wave, a_at(0), loff, 0, g.rb);
    crt_issue(lds, 1, wave, b_at(0), loff, 0, g.rb);
    crt_issue(lds, 2, wave, a_at(1), loff, 0, g.rb);
    crt_issue(lds, 3, wave, b_at(1), loff, 0, g.rb);
    crt_issue(lds, 4, wave, a_at(2), loff, 0, g.rb);
    int isl = 0;
    wait_vmcnt<12>();
    __builtin_amdgcn_s_barrier();
    int csl = 0;
    iv4 fa[FM], fb[FN], nb[FN];
    {
        const int8_t* as = lds + wm * CK2 + roff0;
        const int8_t* bs = lds + CSLOT + wn * CK2 + roff0;
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const iv4*>(bs + 2048 * j);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const iv4*>(as + 2048 * i);
    }
    for (uint32_t s = 0; s < last; ++s) {
        const int bsl = next_slot(csl), asl1 = next_slot(bsl), bsl1 = next_slot(asl1);
        crt_half(acc, fa, fb, nb, lds + csl * CSLOT + wm * CK2 + roff1, lds + bsl * CSLOT + wn * CK2 + roff1);
        __builtin_amdgcn_s_waitcnt((0xF) | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0)
        wait_vmcnt<4>();
        __builtin_amdgcn_s_barrier();
        const int sb = isl, sa = next_slot(isl);
        isl = next_slot(sa);
        crt_half_ld(acc, fa, nb, fb, lds + asl1 * CSLOT + wm * CK2 + roff0, lds + bsl1 * CSLOT + wn * CK2 + roff0,
                    lds, sb, sa, wave, b_at(s + 2), a_at(s + 3), loff, 0, 0, g.rb);
        csl = asl1;
    }
    {
        const int bsl = next_slot(csl), asl1 = next_slot(bsl), bsl1 = next_slot(asl1);
        crt_half(acc, fa, fb, nb, lds + csl * CSLOT + wm * CK2 + roff1, lds + bsl * CSLOT + wn * CK2 + roff1);
        crt_half(acc, fa, nb, fb, lds + asl1 * CSLOT + wm * CK2 + roff0, lds + bsl1 * CSLOT + wn * CK2 + roff0);
    }
    wait_vmcnt<0>();
    // acc[i][j][v] = sum at (m0 + wm + 16i + 4lg + v, n0 + wn + 16j + lr): one
    // 16-byte store each.  Written out here on purpose: the same loop in a
    // function of its own comes out with its column addresses and stores in
    // another order, and products of short K, which are bound by these stores,
    // take 7 % longer (8192 x 8192 x 64 with 8 slices: 750 us against 653 for this
    // kernel, 1205 against 1126 a call).
    int32_t* out = g.planes + (int64_t)gr.plane * g.plane;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int64_t n = n0 + wn + 16 * j + lr;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int64_t m = m0 + wm + 16 * i + 4 * lg;
            __builtin_nontemporal_store(__builtin_bit_cast(iv4, acc[i][j]), reinterpret_cast<iv4*>(out + n * g.Mp + m));
        }
    }
}

// oz_plane_kernel on 128 x 128 tiles.
template <bool BF16>
__global__ __launch_bounds__(SCNT, 2) void oz_plane_small_kernel(OzPlaneArgs g) {
    typedef typename std::conditional<BF16, fv4, iv4>::type acc_t;
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
    const int tiles = g.tiles_m * g.tiles_n;
    const int gi = blockIdx.x / tiles;
    int64_t m0, n0;
    tile_origin<ST>(blockIdx.x - gi * tiles, tiles, g.tiles_m, g.tiles_n, m0, n0);
    const OzGroup gr = g.jobs[gi];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const uint32_t last = (uint32_t)gr.count * gr.nks.d - 1;
    const int8_t* ga = g.a + gr.t0 * g.a_slice + (m0 + 32 * wave) * g.rb + gr.kb;
    const int8_t* gb = g.b + gr.u0 * g.b_slice + (n0 + 32 * wave) * g.rb + gr.kb;
    acc_t acc[SFM][SFN];
#pragma unroll
    for (int i = 0; i < SFM; ++i)
#pragma unroll
        for (int j = 0; j < SFN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    small_product(
        acc, lds, [&](uint32_t s) { return group_step(ga, g.a_slice, s, last, gr.nks); },
        [&](uint32_t s) { return group_step(gb, -g.b_slice, s, last, gr.nks); }, last, g.rb, wave, lane, wm, wn);
    int32_t* out = g.planes + (int64_t)gr.plane * g.plane + m0 + wm + 4 * (lane >> 4);
    n0 += wn + (lane & 15);
#pragma unroll
    for (int j = 0; j < SFN; ++j)
#pragma unroll
        for (int i = 0; i < SFM; ++i)
            __builtin_nontemporal_store(__builtin_bit_cast(iv4, acc[i][j]),
                                        reinterpret_cast<iv4*>(out + (n0 + 16 * j) * g.Mp + 16 * i));
}

// C = val + beta C on up to four rows of a column (`left` of them in C), in
// 32-byte accesses where C allows it (the combination of 8 planes of 3000 x
// 2000: 52 -> 44 us against single elements).
__device__ __forceinline__ void store_c(double (&val)[4], double* cp, int64_t left, double beta) {
    if (left >= 4 && (reinterpret_cast<uintptr_t>(cp) & 31) == 0) {
        dv4* c4 = reinterpret_cast<dv4*>(cp);
        if (beta != 0.0) {
            const dv4 old = __builtin_nontemporal_load(c4);
#pragma unroll
            for (int e = 0; e < 4; ++e) val[e] = __dadd_rn(val[e], __dmul_rn(beta, old[e]));
        }
        __builtin_nontemporal_store(dv4{val[0], val[1], val[2], val[3]}, c4);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e >= left) break;
            if (beta != 0.0) val[e] = __dadd_rn(val[e], __dmul_rn(beta, cp[e]));
            cp[e] = val[e];
        }
    }
}

// The FP64 recombination of scheme I from the planes of groups [gb, ge) of
// ng, for one thread's 4 rows of one column of the padded Mp x Np extent:
// each group's x = sum * 2^-(bits*level) (exact) is added in group order,
// W = x for the first group of all and W + x after (W carried in HBM from
// one launch to the next); after the last group C = alpha*ldexp(W, e_i + f_j)
// + beta*C.  Every FP64 operation is rounded on its own, in this order.
template <bool BF16>
__global__ __launch_bounds__(256) void oz_combine_kernel(const int32_t* __restrict__ planes, int64_t plane,
                                                         const OzGroup* __restrict__ groups, int gb, int ge, int ng,
                                                         int bits, double* __restrict__ W, int64_t Mp, int64_t m,
                                                         int64_t n, const int32_t* __restrict__ ea,
                                                         const int32_t* __restrict__ eb, double alpha, double beta,
                                                         double* __restrict__ C, int64_t ldc, FastDiv dqm,
                                                         uint32_t total) {
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;  // one thread per 4 rows
    if (x >= total) return;
    const uint32_t j = fdiv(x, dqm);
    const int64_t i0 = (int64_t)(x - j * dqm.d) * 4;
    const int64_t e0 = (int64_t)j * Mp + i0;
    double cur[4] = {0.0, 0.0, 0.0, 0.0};
    if (gb > 0) {
        const dv4 w = __builtin_nontemporal_load(reinterpret_cast<const dv4*>(W + e0));
#pragma unroll
        for (int e = 0; e < 4; ++e) cur[e] = w[e];
    }
    for (int gg = gb; gg < ge; ++gg) {
        const double wgt = ldexp(1.0, -bits * groups[gg].level);
        const iv4 v = __builtin_nontemporal_load(reinterpret_cast<const iv4*>(planes + (int64_t)(gg - gb) * plane + e0));
        // the FP32 sums of BF16 slices: the whole vector is bit-cast (a bit cast
        // of one vector element, v[e], read the wrong element with this compiler)
        const fv4 vf = __builtin_bit_cast(fv4, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double xv = (BF16 ? (double)vf[e] : (double)v[e]) * wgt;
            cur[e] = gg == 0 ? xv : __dadd_rn(cur[e], xv);
        }
    }
    if (ge < ng) {
        __builtin_nontemporal_store(dv4{cur[0], cur[1], cur[2], cur[3]}, reinterpret_cast<dv4*>(W + e0));
        return;
    }
    if ((int64_t)j >= n) return;
    const int jf = eb[j];
#pragma unroll
    for (int e = 0; e < 4; ++e) cur[e] = __dmul_rn(alpha, ldexp(cur[e], ea[i0 + e] + jf));  // ea is padded
    store_c(cur, C + i0 + (int64_t)j * ldc, m - i0, beta);
}

// The balanced CRT value V of one element, correctly rounded to double, from
// the limb sums L_l = sum_t x_t * limb_l(M_t) over 40-bit limbs (exact
// doubles below 2^52), S = L0 + L1 2^40 + L2 2^80 = V + jP with j in [0, 16].
// Since |V| <= P/4 (the scaling bound), S/P lies within 1/4 of the integer j
// and j = rint(fl(S) fl(1/P)) exactly (the estimate errs by ~2^-47).  Then
// in FP64, every step exact: D_l = L_l - j P_l (|D_l| < 2^52), and two carries
// bring D0, D1 into [-2^39, 2^39], so V = D2 2^80 + D1 2^40 + D0.  With
// s = fl(D2 2^80 + D1 2^40) and its exact error e, V = s + (e + D0): one
// rounding if e = 0.  Otherwise |s| >= 2^93, and s + e and every point halfway
// between two doubles there are multiples of 2^40 > |D0|, so that only D0's
// sign matters: +-2^30 in its place makes e + D0 exact (|e| <= 2^71).  About 30
// operations in all, none on 64-bit integers.
__host__ __device__ inline double crt_value(double L0, double L1, double L2, const CrtTables& tb) {
    const double Sd = fma(L2, 0x1p80, fma(L1, 0x1p40, L0));
    const double jd = rint(Sd * tb.invPd);
    double D0 = fma(-jd, tb.Pl[0], L0);
    double D1 = fma(-jd, tb.Pl[1], L1);
    double D2 = fma(-jd, tb.Pl[2], L2);
    double c = rint(D0 * 0x1p-40);
    D0 = fma(-c, 0x1p40, D0);
    D1 = D1 + c;
    c = rint(D1 * 0x1p-40);
    D1 = fma(-c, 0x1p40, D1);
    D2 = D2 + c;
    const double mid = D1 * 0x1p40;
    const double s = fma(D2, 0x1p80, mid);
    const double e = mid - fma(-D2, 0x1p80, s);
    const double low = e != 0.0 ? fmin(fmax(D0, -1.0), 1.0) * 0x1p30 : D0;
    return s + (e + low);
}

// Four consecutive rows per thread (one 32-bit load of CRT digits per modulus).
// The limb sums L_l = sum_t x_t * limb_l(M_t) over 40-bit limbs of M_t are
// exact FP64 FMAs (x_t < 256, limbs < 2^40, at most 16 terms: below 2^52);
// crt_value reduces S = sum_t x_t M_t < 16 P modulo P to the balanced V and
// rounds it to double once.
// C = alpha * ldexp(V, e_i + f_j - 2q) + beta*C, four rows per 32-byte access
// when C allows it.
// NMOD (the moduli count) is a template argument so that every digit load
// of a thread is issued before the first is used.
// Thread x (x < ceil(m/4) n < 2^32) takes rows 4 (x % qm) .. + 3 of column
// x / qm, qm = ceil(m/4), divided by multiply-shift.
template <int NMOD>
__global__ __launch_bounds__(256) void crt_reconstruct_kernel(const uint8_t* __restrict__ res, CrtTables tb, int64_t m,
                                                              int64_t n, int64_t Mp, int64_t plane,
                                                              const int32_t* __restrict__ ea,
                                                              const int32_t* __restrict__ eb, int q, double alpha,
                                                              double beta, double* __restrict__ C, int64_t ldc,
                                                              FastDiv dqm) {
    const uint32_t total = dqm.d * (uint32_t)n;
    {
        const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;  // one thread per 4 rows
        if (x >= total) return;
        const uint32_t jq = fdiv(x, dqm);
        const int64_t j = jq, i0 = (int64_t)(x - jq * dqm.d) * 4;
        const uint8_t* rp = res + j * Mp + i0;
        uint32_t w[NMOD];
#pragma unroll
        for (int t = 0; t < NMOD; ++t)  // digits and C are touched once: nontemporal accesses
            w[t] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(rp + (int64_t)t * plane));
        double L[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int l = 0; l < 3; ++l) L[e][l] = 0.0;
#pragma unroll
        for (int t = 0; t < NMOD; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double xd = (double)((w[t] >> (8 * e)) & 255u);
#pragma unroll
                for (int l = 0; l < 3; ++l) L[e][l] = fma(xd, tb.mt[t][l], L[e][l]);
            }
        }
        const int jf = eb[j];
        double val[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t i = i0 + e < m ? i0 + e : m - 1;  // rows past m are computed but never stored
            val[e] = __dmul_rn(alpha, ldexp(crt_value(L[e][0], L[e][1], L[e][2], tb), ea[i] + jf - 2 * q));
        }
        store_c(val, C + i0 + j * ldc, m - i0, beta);
    }
}


// One operand of scheme I: op(X)(row, k) at x[row*rs + k*ks].
struct OzSide {
    const double* x;
    int64_t rows, rs, ks;
    double* part;         // chunk maxima, [nchunk][rows], in the place of the slices (written after them)
    int64_t kchunk;
    uint32_t nchunk, groups;  // k-chunks and row groups of the maxima pass
    int32_t* e;           // exponents, zeros in the padding
    int8_t* out;          // slices
    int64_t rows_p, slice_bytes;
};

// Row maxima of both operands in one launch (the first `na` workgroups take
// op(A)): max |x| over a k-chunk for every row.  Rows strided in memory
// (ks != 1): a thread per row, consecutive lanes on consecutive rows, 16
// loads in flight, consecutive workgroups down the columns.  Rows
// contiguous in k: 16 lanes per row in pairs of any alignment, eight in
// flight, consecutive workgroups along the rows.  Both operands of 3000 x
// 2000 x 5000, transposed and plain: 44 us (4.6 TB/s; a launch each with 256
// k and four loads in flight per thread: 53 us), of 2048^3: 14 us (37 us).
__global__ __launch_bounds__(NT) void oz_partial_max_kernel(OzSide A, OzSide B, int64_t K, uint32_t na) {
    const bool first = blockIdx.x < na;
    const OzSide o = first ? A : B;
    const uint32_t b = first ? blockIdx.x : blockIdx.x - na;
    if (o.ks != 1) {
        const uint32_t c = b / o.groups;
        const int64_t r = (int64_t)(b - c * o.groups) * NT + threadIdx.x;
        if (r >= o.rows) return;
        const int64_t k0 = c * o.kchunk, k1 = min(K, k0 + o.kchunk);
        const double* xr = o.x + r * o.rs;
        double mx = 0.0;
        for (int64_t k = k0; k < k1; k += 16) {
            double v[16];  // past the end: the last entry again
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = xr[min(k + i, k1 - 1) * o.ks];
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmax(mx, fabs(v[i]));
        }
        o.part[c * o.rows + r] = mx;
    } else {
        const uint32_t grp = b / o.nchunk, c = b - grp * o.nchunk;
        const int l16 = threadIdx.x & 15;
        const int64_t r = (int64_t)grp * (NT / 16) + (threadIdx.x >> 4);
        if (r >= o.rows) return;  // whole 16-lane groups leave together
        const int64_t k0 = c * o.kchunk, k1 = min(K, k0 + o.kchunk);
        const double* xr = o.x + r * o.rs;
        double mx = 0.0;
        for (int64_t k = k0; k < k1; k += 256) {
            if (k + 256 <= k1) {
                udv2 v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const udv2*>(xr + k + 32 * i + 2 * l16);
#pragma unroll
                for (int i = 0; i < 8; ++i) mx = fmax(mx, fmax(fabs(v[i].x), fabs(v[i].y)));
            } else {
                for (int64_t kk = k + l16; kk < k1; kk += 16) mx = fmax(mx, fabs(xr[kk]));
            }
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off));
        if (l16 == 0) o.part[c * o.rows + r] = mx;
    }
}

// Reduces the chunk maxima of both operands and writes the frexp exponents
// (0 for zero rows, and for the padding rows beyond `rows`): 64 rows per
// workgroup (rows_p is a multiple of 256), its waves splitting the chunks.
__global__ __launch_bounds__(NT) void oz_exponent_kernel(OzSide A, OzSide B) {
    __shared__ double red[NT / 64][64];
    const uint32_t na = (uint32_t)(A.rows_p / 64);
    const bool first = blockIdx.x < na;
    const OzSide o = first ? A : B;
    const int64_t r = (int64_t)(first ? blockIdx.x : blockIdx.x - na) * 64 + (threadIdx.x & 63);
    double mx = 0.0;
    if (r < o.rows) {
#pragma unroll 4
        for (uint32_t c = threadIdx.x >> 6; c < o.nchunk; c += NT / 64) mx = fmax(mx, o.part[c * o.rows + r]);
    }
    red[threadIdx.x >> 6][threadIdx.x & 63] = mx;
    __syncthreads();
    if (threadIdx.x >= 64) return;
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) mx = fmax(mx, red[w][threadIdx.x]);
    int ex = 0;
    if (mx != 0.0) frexp(mx, &ex);
    o.e[r] = ex;
}

// Ozaki scheme II scaling (Cauchy-Schwarz bound).  Entry bound: |x| = m 2^ex
// (m in [0.5, 1)) counts ceil(256 m)^2 2^(16 - 2d), d = e - ex >= 0 for the
// exponent e of the chunk's maximum, rounded up to an integer (at least 1)
// when 2d > 16: an exact integer upper bound of 2^32 (x 2^-e)^2 whose sums do
// not depend on the summation order.  Computed in FP64 without branches:
// M^2 <= 2^16 scaled by 2^-min(2d - 16, 64) and rounded up is the integer
// exactly (a zero entry gives m = 0, hence 0), and chunk sums of at most
// 64 terms of at most 2^32 stay exact.
__device__ __forceinline__ double crt_bound_term(double x, int e) {
    int ex;
    const double m = frexp(fabs(x), &ex);
    const double M = ceil(m * 256.0);
    return ceil(ldexp(M * M, -min(2 * (e - ex) - 16, 64)));
}

// The scheme II line scan, one read of op(X) per call.  Each line is cut
// into k-chunks of CRT_KC entries; chunk c gets its own max exponent e_c
// (max |x| < 2^e_c) and the exact integer bound S_c = sum crt_bound_term(x,
// e_c) (at most CRT_KC * 2^32 = 2^38), stored as one word
// ((e_c + 2048) << 48) | S_c, or 0 for an all-zero chunk.  crt_shift_kernel
// rescales the chunk bounds to the line's max exponent.  Rows strided in
// memory (ks != 1): 4 threads per line; lines contiguous in k: 16 lanes per
// line.  Either is bound by the one read of op(X): 8192^2 strided 81 us (6.6
// TB/s; a thread per line with 64 loads: 110 us), contiguous 88 us.  Every term
// and chunk sum is an integer below 2^39, so the sums are exact in any order.
constexpr int CRT_KC = 64;

__device__ __forceinline__ uint64_t crt_chunk_word(double amax, uint64_t sum) {
    if (amax == 0.0) return 0;
    int ec;
    frexp(amax, &ec);
    return ((uint64_t)(ec + 2048) << 48) | sum;
}

__device__ __forceinline__ int crt_chunk_exp(double amax) {
    int ec = 0;
    if (amax != 0.0) frexp(amax, &ec);
    return ec;
}

// Lines strided in memory (ks != 1): a workgroup takes CSL_L lines of one
// chunk, CSL_P threads a line with CRT_KC / CSL_P entries each, consecutive
// lanes on consecutive lines (a load of CSL_L lanes is contiguous when
// rs == 1), every load in flight at once.  Each entry is kept as its
// exponent ex and mantissa bound M = ceil(256 m) (|x| = m 2^ex, M in
// [128, 256], 0 for a zero entry) packed as ((ex + 2048) << 9) | M, so the
// largest packed word of the chunk carries the exponent e of its largest
// entry, and the terms of crt_bound_term follow from (M, ex).  blockIdx.x =
// line tile, blockIdx.y = chunk (the grid walks down the columns).
constexpr int CSL_P = 4, CSL_L = 256 / CSL_P, CSL_K = CRT_KC / CSL_P;

__global__ __launch_bounds__(256) void crt_scan_lines_kernel(CrtSide A, CrtSide B, uint32_t na, int64_t K) {
    const bool first = blockIdx.x < na;
    const CrtSide o = first ? A : B;
    const double* __restrict__ x = o.x;
    const int64_t rows = o.rows, rs = o.rs, ks = o.ks;
    __shared__ uint32_t tops[CSL_P][CSL_L];
    __shared__ double sums[CSL_P][CSL_L];
    const int line = threadIdx.x % CSL_L, w = threadIdx.x / CSL_L;
    const int64_t r = (int64_t)(first ? blockIdx.x : blockIdx.x - na) * CSL_L + line;
    const int64_t k0 = (int64_t)blockIdx.y * CRT_KC + w * CSL_K;
    // every load unconditional (the last entry or line again past the end),
    // so that all of them issue before the first wait
    const double* xr = x + min(r, rows - 1) * rs;
    double raw[CSL_K];
#pragma unroll
    for (int i = 0; i < CSL_K; ++i) raw[i] = __builtin_nontemporal_load(xr + min(k0 + i, K - 1) * ks);
    uint32_t wd[CSL_K];
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < CSL_K; ++i) {
        const double v = k0 + i < K ? raw[i] : 0.0;
        int ex;
        const double m = frexp(fabs(v), &ex);
        const uint32_t M = (uint32_t)ceil(m * 256.0);
        wd[i] = M ? ((uint32_t)(ex + 2048) << 9) | M : 0u;
        top = top > wd[i] ? top : wd[i];
    }
    tops[w][line] = top;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < CSL_P; ++p) top = max(top, tops[p][line]);
    const int ec = (int)(top >> 9) - 2048;
    double sum = 0.0;
    if (top) {
#pragma unroll
        for (int i = 0; i < CSL_K; ++i) {
            const double M = (double)(wd[i] & 511u);
            const int ex = (int)(wd[i] >> 9) - 2048;
            sum += wd[i] ? ceil(ldexp(M * M, -min(2 * (ec - ex) - 16, 64))) : 0.0;
        }
    }
    sums[w][line] = sum;
    __syncthreads();
    if (w != 0 || r >= rows) return;
#pragma unroll
    for (int p = 1; p < CSL_P; ++p) sum += sums[p][line];
    o.part[(int64_t)blockIdx.y * rows + r] = top ? ((uint64_t)(ec + 2048) << 48) | (uint64_t)sum : 0;
}

// Lines contiguous in k: 16 lanes per line, two pairs of any alignment each.
// Workgroup = line tile * nchunk + chunk, so the grid walks along the lines
// (consecutive workgroups read consecutive chunks of the same lines).
__global__ __launch_bounds__(256) void crt_scan_rows_kernel(CrtSide A, CrtSide B, uint32_t na, int64_t K,
                                                            uint32_t nchunk) {
    const bool first = blockIdx.x < na;
    const CrtSide o = first ? A : B;
    const uint32_t block = first ? blockIdx.x : blockIdx.x - na;
    const double* __restrict__ x = o.x;
    const int64_t rows = o.rows, rs = o.rs;
    const uint32_t tile = block / nchunk;
    const uint32_t chunk = block - tile * nchunk;
    const int64_t k0 = (int64_t)chunk * CRT_KC;
    const int l16 = threadIdx.x & 15;
    const int64_t r = (int64_t)tile * (NT / 16) + (threadIdx.x >> 4);
    if (r >= rows) return;  // whole 16-lane groups leave together
    const double* xr = x + r * rs;
    double v[4];
    if (k0 + CRT_KC <= K) {  // the whole chunk inside the line: both loads in flight together
        const pdv2 w0 = __builtin_nontemporal_load(reinterpret_cast<const udv2*>(xr + k0 + 2 * l16));
        const pdv2 w1 = __builtin_nontemporal_load(reinterpret_cast<const udv2*>(xr + k0 + 32 + 2 * l16));
        v[0] = w0.x; v[1] = w0.y; v[2] = w1.x; v[3] = w1.y;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t k = k0 + 32 * (i >> 1) + 2 * l16 + (i & 1);
            v[i] = k < K ? xr[k] : 0.0;
        }
    }
    double mx = fmax(fmax(fabs(v[0]), fabs(v[1])), fmax(fabs(v[2]), fabs(v[3])));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off));
    const int ec = crt_chunk_exp(mx);
    double sum = (crt_bound_term(v[0], ec) + crt_bound_term(v[1], ec)) +
                 (crt_bound_term(v[2], ec) + crt_bound_term(v[3], ec));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (l16 == 0) o.part[chunk * rows + r] = crt_chunk_word(mx, (uint64_t)sum);
}

// Line shifts: e = the largest chunk exponent, S = sum over the nonzero
// chunks of ceil(S_c / 4^(e - e_c)), sigma the largest shift with
// 2^(2(sigma + e)) S <= 2^(2Q + 32) (sigma = Q + 16 - e - ceil(log4 S)),
// capped at 53 - e; an all-zero line keeps sigma = 0.  Stored as
// e' = Q - sigma, the form the residue and reconstruction kernels take.
// A workgroup takes 16 lines (a 128-byte line of words); 16 lanes a line split
// the chunks, eight loads in flight, and combine through LDS.
constexpr int CS_L = 16, CS_W = 256 / CS_L;

__global__ __launch_bounds__(256) void crt_shift_kernel(CrtSide A, CrtSide B, uint32_t na, int nchunk, int Q) {
    const bool first = blockIdx.x < na;
    const CrtSide o = first ? A : B;
    const uint64_t* __restrict__ part = o.part;
    const int64_t rows = o.rows;
    __shared__ uint64_t red[CS_W][CS_L];
    const int lane = threadIdx.x % CS_L, w = threadIdx.x / CS_L;
    const int64_t r = (int64_t)(first ? blockIdx.x : blockIdx.x - na) * CS_L + lane;
    const bool valid = r < rows;
    uint64_t top = 0;
    if (valid) {
#pragma unroll 8
        for (int c = w; c < nchunk; c += CS_W) top = max(top, part[(int64_t)c * rows + r] >> 48);
    }
    red[w][lane] = top;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < CS_W; ++i) top = max(top, red[i][lane]);
    __syncthreads();
    uint64_t S = 0;
    if (valid && top != 0) {
#pragma unroll 8
        for (int c = w; c < nchunk; c += CS_W) {
            const uint64_t wd = part[(int64_t)c * rows + r];
            const uint64_t sc = wd & ((1ull << 48) - 1);
            const int d2 = 2 * (int)(top - (wd >> 48));
            const uint64_t v = d2 >= 62 ? 1 : (sc + (1ull << d2) - 1) >> d2;
            S += wd == 0 ? 0 : v;
        }
    }
    red[w][lane] = S;
    __syncthreads();
    if (w != 0) return;  // rows_p is a multiple of CS_L
    S = 0;
#pragma unroll
    for (int i = 0; i < CS_W; ++i) S += red[i][lane];
    int sig = 0;
    if (valid && top != 0) {
        const int bl = S > 1 ? 64 - __builtin_clzll(S - 1) : 0;  // bit length of S - 1
        const int j = (bl + 1) >> 1;                              // ceil(log4 S)
        const int er = (int)top - 2048;
        sig = min(53 - er, Q + 16 - er - j);
    }
    o.e[r] = Q - sig;
}

// Writes the s digits of op(X)(row, k) into slices[t][row][Kp] (zeros in the
// padding), both operands in one launch.  A workgroup takes OS_R rows by
// OS_K k, a thread four consecutive k of every 8th row: one store per row
// and slice, 128 (INT8) or 256 (BF16) contiguous bytes per row.  Rows
// contiguous in k are read straight into registers, 16 bytes at any
// alignment; rows strided in memory go through LDS, loaded along the rows
// (quads of k rotated by 2 (k / 32) places, so that the reads of four
// consecutive k per lane spread over the banks).  Bound by memory: the
// arithmetic (six operations per element and slice) takes less than half of
// the time of reading op(X) and writing the slices.  3000 x 2000 x 5000 into
// 8 INT8 slices: 74 us (5.5 TB/s; 64 x 64 tiles through LDS, one launch per
// operand: 146 us), 2048^3 into 11 BF16 slices: 41 us (56 us).
constexpr int OS_R = 32, OS_K = 128;

__device__ __forceinline__ int os_pos(int k) { return (k & ~3) | ((k + 2 * (k >> 5)) & 3); }

template <bool BF16>
__global__ __launch_bounds__(NT) void oz_slice_kernel(OzSide A, OzSide B, int64_t K, int64_t Kp, int s, int bits,
                                                      uint32_t nkt, uint32_t na, uint32_t tiles) {
    __shared__ double tile[OS_R][OS_K + 1];
    uint32_t b = blockIdx.y * gridDim.x + blockIdx.x;
    if (b >= tiles) return;
    const bool first = b < na;
    const OzSide o = first ? A : B;
    if (!first) b -= na;
    const int t = threadIdx.x;
    const int kq = 4 * (t & 31);
    int64_t r0, k0;
    double v[4][4];
    if (o.ks == 1) {  // tiles along k
        r0 = (int64_t)(b / nkt) * OS_R;
        k0 = (int64_t)(b % nkt) * OS_K;
        const int64_t k = k0 + kq;
        if (r0 + OS_R <= o.rows && k0 + OS_K <= K) {
            udv2 w[4][2];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double* xr = o.x + (r0 + (t >> 5) + 8 * i) * o.rs + k;
                w[i][0] = *reinterpret_cast<const udv2*>(xr);
                w[i][1] = *reinterpret_cast<const udv2*>(xr + 2);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) v[i][c] = w[i][c >> 1][c & 1];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = r0 + (t >> 5) + 8 * i;
#pragma unroll
                for (int c = 0; c < 4; ++c) v[i][c] = r < o.rows && k + c < K ? o.x[r * o.rs + k + c] : 0.0;
            }
        }
    } else {  // tiles down the rows
        const uint32_t nrt = (uint32_t)(o.rows_p / OS_R);
        r0 = (int64_t)(b % nrt) * OS_R;
        k0 = (int64_t)(b / nrt) * OS_K;
        const int64_t r = r0 + (t & 31);
        const double* xr = o.x + min(r, o.rows - 1) * o.rs;
        double w[16];  // past the edges: the last row or entry again
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = xr[min(k0 + (t >> 5) + 8 * i, K - 1) * o.ks];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int kk = (t >> 5) + 8 * i;
            tile[t & 31][os_pos(kk)] = r < o.rows && k0 + kk < K ? w[i] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[i][c] = tile[(t >> 5) + 8 * i][os_pos(kq + c)];
    }
    if (k0 + kq >= Kp) return;  // Kp is a multiple of 64
    const double scale = ldexp(1.0, bits);
    int8_t* dst = o.out + ((r0 + (t >> 5)) * Kp + k0 + kq) * (BF16 ? 2 : 1);
    const int64_t step = 8 * Kp * (BF16 ? 2 : 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int sh = -o.e[r0 + (t >> 5) + 8 * i];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[i][c] = ldexp(v[i][c], sh);
    }
    for (int l = 0; l < s; ++l) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t w[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v[i][c] = v[i][c] * scale;
                const double d = trunc(v[i][c]);
                v[i][c] = v[i][c] - d;
                // BF16: |d| <= 31 is exact, its low mantissa bits are zero
                w[c] = BF16 ? __float_as_uint((float)d) : (uint32_t)(int)d;
            }
            int8_t* q = dst + l * o.slice_bytes + i * step;
            if (BF16) {
                *reinterpret_cast<u32x2*>(q) = u32x2{__builtin_amdgcn_perm(w[1], w[0], 0x07060302u),
                                                     __builtin_amdgcn_perm(w[3], w[2], 0x07060302u)};
            } else {
                *reinterpret_cast<uint32_t*>(q) =
                    __builtin_amdgcn_perm(__builtin_amdgcn_perm(w[3], w[2], 0x0c0c0400u),
                                          __builtin_amdgcn_perm(w[1], w[0], 0x0c0c0400u), 0x05040100u);
            }
        }
    }
}

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

}  // namespace

// Prepared operand of the CRT form (one side of a product): the balanced
// residues of its scaled lines, [nmod][rows_p][Kp] int8 with rows_p = rows
// rounded up to the tile height and Kp = k rounded up to the k-step (zeros
// in the padding), then the lines' exponents e' = Q - sigma (rows_p int32).
int64_t crt_operand_bytes(int64_t rows, int64_t k, int nmod) {
    const int64_t rp = round_up(rows > 0 ? rows : 1, PAD), kp = round_up(k > 0 ? k : 1, KSB);
    return round_up((int64_t)nmod * rp * kp, 256) + rp * 4;
}

int64_t crt_digit_bytes(int64_t m, int64_t n, int nmod) {
    return (int64_t)nmod * round_up(m > 0 ? m : 1, PAD) * round_up(n > 0 ? n : 1, PAD);
}

namespace {

// Scheme I groups whose planes one launch holds (the combine reads them all
// per element): 8 planes of 4 bytes per output element.
constexpr int kPlaneBatch = 8;

struct Plan {
    int64_t Mp, Np, Kp, esz, a_slice, b_slice, res_plane;
    int64_t plane_batch;  // scheme I: groups per product launch
    size_t off_a, off_b, off_ea, off_eb, off_w, off_planes, total;
};

// Whether a launch of `wgs` 256 x 256 tiles, the longest of `longest` k-steps,
// `total` k-steps in all, takes 128 x 128 tiles instead: the launch lasts
// about as long as its longest tile or its work spread over the CUs (whole
// rounds of equal tiles), and a k-step of a quarter tile takes kSmallStep of
// a whole one's time (0.37 with every CU busy, 0.42 with few: the LDS bounds
// it, whose reads per MFMA grow by a third).  8 INT8 slices, 512^3: 41 us a
// call with 128 x 128 tiles, 67 with 256 x 256; 300 x 700 x 4000: 137 and
// 294; 2048^3: 411 and 319.  14 moduli, 512^3: 39 and 43; 1024^3: 74 and 61.
constexpr double kSmallStep = 0.4;

bool small_tiles(int64_t wgs, int64_t longest, int64_t total) {
    constexpr int kCus = 256;
    const auto spread = [&](int64_t n) {
        if (total == wgs * longest) return (double)((n + kCus - 1) / kCus * longest);
        return std::max((double)longest, (double)total * (double)(n / wgs) / kCus);
    };
    return kSmallStep * spread(4 * wgs) < spread(wgs);
}

// Host side of the CRT form: q and the reconstruction tables for n moduli.
int crt_setup(int64_t k, int nmod, CrtTables* tb, int* q_out) {
    unsigned __int128 P = 1;
    for (int t = 0; t < nmod; ++t) P *= (unsigned)crt_modulus(t);
    // largest Q with 2^(2Q) + ceil(sqrt(k)) 2^Q + k <= P/4: lines of 2-norm
    // <= 2^Q before rounding keep |A'B'| <= P/4 (Cauchy-Schwarz)
    const uint64_t kk = (uint64_t)(k > 0 ? k : 0);
    uint64_t rk = (uint64_t)sqrt((double)kk);
    while (rk * rk > kk) --rk;
    while ((rk + 1) * (rk + 1) <= kk) ++rk;
    if (rk * rk < kk) ++rk;  // ceil(sqrt(k))
    int q = 62;
    while (q >= 1) {
        const unsigned __int128 need = ((unsigned __int128)1 << (2 * q)) + ((unsigned __int128)rk << q) + kk;
        if (need <= (P >> 2)) break;
        --q;
    }
    if (q < 1) return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: %d moduli leave no bits for k=%lld", nmod, (long long)k);
    *q_out = q;
    tb->n = nmod;
    for (int t = 0; t < nmod; ++t) {
        const int p = crt_modulus(t);
        const unsigned __int128 M = P / (unsigned)p;
        for (int l = 0; l < 3; ++l) tb->mt[t][l] = (double)(uint64_t)((M >> (40 * l)) & (((unsigned __int128)1 << 40) - 1));
        // inverse of M mod p by extended Euclid (M and p are coprime)
        int64_t a = (int64_t)(M % (unsigned)p), b = p, x0 = 1, x1 = 0;
        while (b) {
            const int64_t qq = a / b, tmp = a - qq * b;
            a = b; b = tmp;
            const int64_t tx = x0 - qq * x1;
            x0 = x1; x1 = tx;
        }
        tb->cinv[t] = (int32_t)(((x0 % p) + p) % p);
    }
    for (int l = 0; l < 3; ++l) tb->Pl[l] = (double)(uint64_t)((P >> (40 * l)) & (l < 2 ? (((unsigned __int128)1 << 40) - 1) : ~(unsigned __int128)0));
    tb->invPd = 1.0 / (double)P;
    return DG_OK;
}

}  // namespace

int crt_moduli_for_fp64(int64_t k) {
    if (k >= ((int64_t)1 << 19)) return kMaxModuli;
    unsigned __int128 P = 1;
    const unsigned __int128 need = (unsigned __int128)(k > 0 ? k : 1) << (2 * 53 + 2);
    for (int t = 0; t < kMaxModuli; ++t) {
        P *= (unsigned)crt_modulus(t);
        if (t >= 1 && need <= P) return t + 1;
    }
    return kMaxModuli;
}

namespace {

// Workspace of one CRT call: the prepared A and B operands (crt_operand_bytes
// each), then the CRT digits of V.
Plan make_crt_plan(int64_t m, int64_t n, int64_t k, int nmod) {
    Plan p{};
    p.esz = 1;
    p.Mp = round_up(m > 0 ? m : 1, PAD);
    p.Np = round_up(n > 0 ? n : 1, PAD);
    p.Kp = round_up(k > 0 ? k : 1, KSB);
    p.a_slice = p.Mp * p.Kp;
    p.b_slice = p.Np * p.Kp;
    p.res_plane = p.Mp * p.Np;
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off = (off + bytes + 255) / 256 * 256; return o; };
    p.off_a = take((size_t)crt_operand_bytes(m, k, nmod));
    p.off_b = take((size_t)crt_operand_bytes(n, k, nmod));
    p.off_w = take((size_t)crt_digit_bytes(m, n, nmod));
    p.total = off;
    return p;
}

std::vector<OzSeg> make_schedule(int s, int bits, int64_t Kp, int64_t K, bool bf16, int* err);

Plan make_plan(int64_t m, int64_t n, int64_t k, int s, bool bf16) {
    Plan p{};
    p.esz = bf16 ? 2 : 1;
    p.Mp = round_up(m > 0 ? m : 1, PAD);
    p.Np = round_up(n > 0 ? n : 1, PAD);
    p.Kp = round_up(k > 0 ? k : 1, KSB / p.esz);
    p.a_slice = p.Mp * p.Kp * p.esz;
    p.b_slice = p.Np * p.Kp * p.esz;
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off = (off + bytes + 255) / 256 * 256; return o; };
    p.off_a = take((size_t)s * p.a_slice);
    p.off_b = take((size_t)s * p.b_slice);
    p.off_ea = take((size_t)p.Mp * 4);
    p.off_eb = take((size_t)p.Np * 4);
    p.off_w = take((size_t)p.Mp * (size_t)p.Np * 8);
    {  // group planes
        int err = 0;
        int64_t groups = 0;
        for (const OzSeg& g : make_schedule(s, bf16 ? 5 : 7, p.Kp, k, bf16, &err)) groups += g.flush != 0;
        p.plane_batch = groups < kPlaneBatch ? (groups > 0 ? groups : 1) : kPlaneBatch;
        p.off_planes = take((size_t)p.plane_batch * (size_t)p.Mp * (size_t)p.Np * 4);
    }
    p.total = off;
    return p;
}

// Product schedule in the oracle's order: level, k-chunk, t.
std::vector<OzSeg> make_schedule(int s, int bits, int64_t Kp, int64_t K, bool bf16, int* err) {
    const int64_t dmax = (1 << bits) - 1;
    const int64_t kstep = KSB / (bf16 ? 2 : 1);
    int64_t kchunk = Kp;
    int64_t flush;
    if (bf16) {
        // fp32 sums stay exact below 2^24: chunk K so that one product fits
        const int64_t cap = ((int64_t)1 << 24) / (dmax * dmax);
        if (kchunk > cap) kchunk = cap / kstep * kstep;
        const int64_t keff = K < kchunk ? K : kchunk;
        flush = ((int64_t)1 << 24) / (dmax * dmax * (keff > 0 ? keff : 1));
    } else {
        flush = (int64_t)INT32_MAX / (dmax * dmax * (K > 0 ? K : 1));
    }
    *err = (flush < 1 || kchunk < kstep) ? 1 : 0;
    std::vector<OzSeg> segs;
    for (int l = 2; l <= s + 1; ++l)
        for (int64_t k0 = 0; k0 < Kp; k0 += kchunk) {
            const int64_t kl = (Kp - k0) < kchunk ? (Kp - k0) : kchunk;
            int cnt = 0;
            for (int t = 1; t <= l - 1; ++t) {
                OzSeg g{};
                g.t = t - 1;
                g.u = l - t - 1;
                g.k0 = (int32_t)k0;
                g.klen = (int32_t)kl;
                g.level = l;
                ++cnt;
                g.flush = (cnt == flush || t == l - 1) ? 1 : 0;
                if (g.flush) cnt = 0;
                segs.push_back(g);
            }
        }
    // Mark the first and the last flush (W is written, not read, by the first;
    // the last one writes C).
    bool seen = false;
    for (auto& g : segs)
        if (g.flush) {
            if (!seen) { g.flush = 2; seen = true; }
        }
    for (auto it = segs.rbegin(); it != segs.rend(); ++it)
        if (it->flush) { it->flush = it->flush == 2 ? 4 : 3; break; }
    return segs;
}

// The schedule's products cut at its flushes: each group is consecutive
// products of one level and one k range with t rising and u falling by one.
// Returns false if the schedule does not have that form.
bool make_groups(const std::vector<OzSeg>& sched, int64_t esz, std::vector<OzGroup>& out) {
    out.clear();
    for (size_t i = 0; i < sched.size();) {
        size_t j = i;
        while (j < sched.size() && !sched[j].flush) ++j;
        if (j == sched.size()) return false;
        const OzSeg& f = sched[i];
        for (size_t q = i; q <= j; ++q) {
            const OzSeg& x = sched[q];
            if (x.level != f.level || x.k0 != f.k0 || x.klen != f.klen || x.t != f.t + (int)(q - i) ||
                x.u != f.u - (int)(q - i))
                return false;
        }
        if ((f.klen * esz) % CK2 != 0 || (f.k0 * esz) % CK2 != 0 || f.klen <= 0) return false;
        out.push_back(OzGroup{f.t, f.u, (int32_t)(j - i + 1), f.level, (int32_t)(f.k0 * esz),
                              make_fastdiv((uint32_t)(f.klen * esz / CK2)), 0});
        if ((int64_t)out.back().count * out.back().nks.d > INT32_MAX) return false;
        i = j + 1;
    }
    return !out.empty();
}

}  // namespace

// Scheme II, one or two operands of a product: line scan, shifts and residues
// into each one's `operand` (crt_operand_bytes(rows, k, nmod) bytes, 256-byte
// aligned).  The result depends only on the operand, k and nmod, so a
// prepared operand serves every product that reads it.  The scan words (8
// bytes per 64 k) lie where the residues go (at least 64 bytes per 64 k).
int crt_prepare(const CrtLines* ops, int count, int64_t k, int nmod, hipStream_t st) {
    CrtTables tables{};
    int q = 0;
    int rc = crt_setup(k, nmod, &tables, &q);
    if (rc) return rc;
    const int64_t kp = round_up(k, KSB);
    const int nchunk = (int)((k + CRT_KC - 1) / CRT_KC);
    CrtSide side[2] = {};
    int64_t scan[2] = {0, 0}, res[2] = {0, 0};
    for (int i = 0; i < count; ++i) {
        const CrtLines& l = ops[i];
        CrtSide& o = side[i];
        o.x = l.x; o.rows = l.rows; o.rs = l.rs; o.ks = l.ks;
        o.rows_p = round_up(l.rows, PAD);
        o.out = static_cast<int8_t*>(l.operand);
        o.e = reinterpret_cast<int32_t*>(static_cast<char*>(l.operand) + round_up((int64_t)nmod * o.rows_p * kp, 256));
        o.part = static_cast<uint64_t*>(l.operand);
        o.nkt = (uint32_t)(l.ks == 1 ? (kp + RC_K - 1) / RC_K : kp / RT_K);
        o.nrt = (uint32_t)(l.ks == 1 ? o.rows_p / RC_R : o.rows_p / RT_R);
        scan[i] = l.ks == 1 ? (l.rows + NT / 16 - 1) / (NT / 16) * nchunk : (l.rows + CSL_L - 1) / CSL_L;
        res[i] = (int64_t)o.nkt * o.nrt;
        if (scan[i] > INT32_MAX) return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: too many lines for one scan");
        if (res[i] > INT32_MAX) return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: too many residue tiles");
    }
    // Small operands share every launch they can (512^3, 14 moduli: 39 -> 35 us
    // a call); operands that fill the chip by themselves gain nothing from it and
    // keep their own launches (and grids below 2^32 threads).
    const auto launch_scan = [&](const CrtSide& a, const CrtSide& b, int64_t na, int64_t nb) {
        if (a.ks != 1)
            hipLaunchKernelGGL(crt_scan_lines_kernel, dim3((unsigned)(na + nb), (unsigned)nchunk), dim3(NT), 0, st, a, b,
                               (uint32_t)na, k);
        else
            hipLaunchKernelGGL(crt_scan_rows_kernel, dim3((unsigned)(na + nb)), dim3(NT), 0, st, a, b, (uint32_t)na, k,
                               (uint32_t)nchunk);
    };
    const bool together = count == 2 && res[0] + res[1] < (1 << 16);
    if (together && (side[0].ks == 1) == (side[1].ks == 1)) {
        launch_scan(side[0], side[1], scan[0], scan[1]);
    } else {
        for (int i = 0; i < count; ++i) launch_scan(side[i], side[i], scan[i], 0);
    }
    const auto shifts = [](const CrtSide& o) { return (uint32_t)(o.rows_p / CS_L); };
    if (together) {
        hipLaunchKernelGGL(crt_shift_kernel, dim3(shifts(side[0]) + shifts(side[1])), dim3(NT), 0, st, side[0], side[1],
                           shifts(side[0]), nchunk, q);
    } else {
        for (int i = 0; i < count; ++i)
            hipLaunchKernelGGL(crt_shift_kernel, dim3(shifts(side[i])), dim3(NT), 0, st, side[i], side[i],
                               shifts(side[i]), nchunk, q);
    }
    decltype(&crt_residue_kernel<16>) rsk = crt_residue_kernel<16>;
    switch (nmod) {
#define DG_CRT_CASE(N) case N: rsk = crt_residue_kernel<N>; break;
        DG_CRT_CASE(2) DG_CRT_CASE(3) DG_CRT_CASE(4) DG_CRT_CASE(5) DG_CRT_CASE(6) DG_CRT_CASE(7)
        DG_CRT_CASE(8) DG_CRT_CASE(9) DG_CRT_CASE(10) DG_CRT_CASE(11) DG_CRT_CASE(12) DG_CRT_CASE(13)
        DG_CRT_CASE(14) DG_CRT_CASE(15)
#undef DG_CRT_CASE
        default: break;
    }
    ResidueConsts rcs{};
    for (int t = 0; t < kMaxModuli; ++t) {
        rcs.inv_p[t] = 1.0 / (double)crt_modulus(t);
    }
    if (together) {
        hipLaunchKernelGGL(rsk, dim3((unsigned)(res[0] + res[1])), dim3(256), 0, st, side[0], side[1], (uint32_t)res[0],
                           k, q, kp, rcs);
    } else {
        for (int i = 0; i < count; ++i)
            hipLaunchKernelGGL(rsk, dim3((unsigned)res[i]), dim3(256), 0, st, side[i], side[i], (uint32_t)res[i], k, q,
                               kp, rcs);
    }
    DG_LAUNCH_CHECK();
    return DG_OK;
}

// Scheme II, the product of two prepared operands (m lines of op(A), n lines
// of op(B)^T, both over k with nmod moduli): the nmod INT8 GEMMs into the CRT
// digits (`digits`, crt_digit_bytes(m, n, nmod) bytes), then
// C = alpha * V * 2^(e'_i + f'_j - 2Q) + beta * C.
int crt_multiply(int64_t m, int64_t n, int64_t k, int nmod, double alpha, const void* a_op, const void* b_op,
                 double beta, double* C, int64_t ldc, void* digits, hipStream_t st) {
    CrtTables tables{};
    int q = 0;
    int rc = crt_setup(k, nmod, &tables, &q);
    if (rc) return rc;
    const int64_t mp = round_up(m, PAD), np = round_up(n, PAD), kp = round_up(k, KSB);
    CrtArgs cg{};
    cg.a = static_cast<const int8_t*>(a_op);
    cg.b = static_cast<const int8_t*>(b_op);
    cg.res = static_cast<uint8_t*>(digits);
    cg.Mp = mp; cg.Np = np; cg.Kp = kp; cg.a_slice = mp * kp; cg.b_slice = np * kp;
    cg.res_plane = mp * np;
    cg.tiles_m = (int32_t)(mp / BM); cg.tiles_n = (int32_t)(np / BN); cg.nmod = nmod;
    for (int t = 0; t < kMaxModuli; ++t) cg.cinv[t] = tables.cinv[t];
    const int32_t* ea = reinterpret_cast<const int32_t*>(static_cast<const char*>(a_op) + round_up((int64_t)nmod * mp * kp, 256));
    const int32_t* eb = reinterpret_cast<const int32_t*>(static_cast<const char*>(b_op) + round_up((int64_t)nmod * np * kp, 256));
    int64_t grid = (int64_t)cg.tiles_m * cg.tiles_n * nmod;
    const int64_t steps = kp / CK2;
    const bool small = small_tiles(grid, steps, grid * steps);
    if (small) {
        cg.tiles_m *= BM / ST;
        cg.tiles_n *= BN / ST;
        grid *= (BM / ST) * (BN / ST);
    }
    if (grid > INT32_MAX) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: too many tiles");
    const int64_t quads = ((m + 3) / 4) * n;
    if (quads > (int64_t)UINT32_MAX - 255)
        return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: too many output elements for one reconstruction");
    if (small)
        hipLaunchKernelGGL(crt_gemm_small_kernel, dim3((unsigned)grid), dim3(SCNT), kCrtLds, st, cg);
    else
        hipLaunchKernelGGL(crt_gemm_kernel, dim3((unsigned)grid), dim3(CNT), kCrtLds, st, cg);
    DG_LAUNCH_CHECK();
    decltype(&crt_reconstruct_kernel<16>) rk = crt_reconstruct_kernel<16>;
    switch (nmod) {
#define DG_CRT_CASE(N) case N: rk = crt_reconstruct_kernel<N>; break;
        DG_CRT_CASE(2) DG_CRT_CASE(3) DG_CRT_CASE(4) DG_CRT_CASE(5) DG_CRT_CASE(6) DG_CRT_CASE(7)
        DG_CRT_CASE(8) DG_CRT_CASE(9) DG_CRT_CASE(10) DG_CRT_CASE(11) DG_CRT_CASE(12) DG_CRT_CASE(13)
        DG_CRT_CASE(14) DG_CRT_CASE(15)
#undef DG_CRT_CASE
        default: break;
    }
    hipLaunchKernelGGL(rk, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, cg.res, tables, m, n, mp,
                       cg.res_plane, ea, eb, q, alpha, beta, C, ldc, make_fastdiv((uint32_t)((m + 3) / 4)));
    DG_LAUNCH_CHECK();
    return DG_OK;
}

}  // namespace dg

extern "C" {

int64_t dg_ozaki_workspace(int64_t m, int64_t n, int64_t k, int slices, int kind) {
    if (m < 0 || n < 0 || k < 0 || slices < 1 || slices > 16) return -1;
    if (kind == DG_OZAKI_INT8_CRT) {
        if (slices < 2) return -1;
        return (int64_t)dg::make_crt_plan(m, n, k, slices).total;
    }
    if (kind != DG_OZAKI_INT8 && kind != DG_OZAKI_BF16) return -1;
    return (int64_t)dg::make_plan(m, n, k, slices, kind == DG_OZAKI_BF16).total;
}

int dg_ozaki_dgemm(char opA, char opB, int64_t m, int64_t n, int64_t k, double alpha, const double* A, int64_t lda,
                   const double* B, int64_t ldb, double beta, double* C, int64_t ldc, int slices, int kind,
                   void* workspace, int64_t workspace_bytes, double* err_bound, void* stream) {
    using namespace dg;
    const char oa = norm_op(opA), ob = norm_op(opB);
    if (!oa || !ob) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: invalid op '%c%c'", opA, opB);
    if (kind != DG_OZAKI_INT8 && kind != DG_OZAKI_BF16 && kind != DG_OZAKI_INT8_CRT)
        return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: kind %d", kind);
    if (slices < 1 || slices > 16) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: slices %d (1..16)", slices);
    const bool crt = kind == DG_OZAKI_INT8_CRT;
    if (crt && slices < 2) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: the CRT form needs 2..16 moduli");
    if (m < 0 || n < 0 || k < 0) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: negative dimension");
    const int64_t rowsA = oa == 'N' ? m : k, rowsB = ob == 'N' ? k : n;
    if (lda < (rowsA > 1 ? rowsA : 1) || ldb < (rowsB > 1 ? rowsB : 1) || ldc < (m > 1 ? m : 1))
        return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: leading dimension too small");
    const bool bf16 = kind == DG_OZAKI_BF16;
    const int bits = bf16 ? 5 : 7;
    CrtTables tables{};
    int q = 0;
    if (crt) {
        if (k > 131071) return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: CRT form needs k < 131072 (exact int32 sums)");
        int rc0 = crt_setup(k, slices, &tables, &q);
        if (rc0) return rc0;
        // every line's shift reaches sigma + e >= qe = min(53, Q - ceil(log4 k)) (its
        // bound sum is at most k 2^32), so |A - 2^-sigma A'| <= 2^(e - qe - 1) per entry
        // and the product error is below k * 2^(1-qe) * 2^(e_i+f_j)
        int l4 = 0;
        while (((int64_t)1 << (2 * l4)) < k) ++l4;
        const int qe = q - l4 < 53 ? q - l4 : 53;
        if (err_bound) *err_bound = (double)k * ldexp(1.0, 1 - qe);
    } else if (err_bound) {
        *err_bound = (double)k * (slices + 3) * ldexp(1.0, -bits * slices);
    }
    if (m == 0 || n == 0) return DG_OK;
    int rc = require_device();
    if (rc) return rc;
    hipStream_t st = as_stream(stream);
    if (k == 0 || alpha == 0.0) return launch_scale(m, n, beta, C, ldc, st);
    if (!A || !B || !C) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: null pointer");
    if (k > INT32_MAX / 2) return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: k too large");
    const Plan p = crt ? make_crt_plan(m, n, k, slices) : make_plan(m, n, k, slices, bf16);
    if (p.Mp / 32 > 65535 || p.Np / 32 > 65535 || p.Kp / 64 > INT32_MAX)
        return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: matrix too large for one slicing launch");
    if (!workspace || workspace_bytes < (int64_t)p.total)
        return fail(DG_ERR_WORKSPACE, "dg_ozaki_dgemm: workspace %lld < %zu bytes", (long long)workspace_bytes, p.total);
    if (reinterpret_cast<uintptr_t>(workspace) & 255)
        return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: workspace must be 256-byte aligned");
    int serr = 0;
    std::vector<OzSeg> sched;
    if (!crt) {
        sched = make_schedule(slices, bits, p.Kp, k, bf16, &serr);
        if (serr)
            return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: k=%lld too large for exact 32-bit slice sums", (long long)k);
    }

    char* ws = static_cast<char*>(workspace);
    int8_t* sa = reinterpret_cast<int8_t*>(ws + p.off_a);
    int8_t* sb = reinterpret_cast<int8_t*>(ws + p.off_b);
    int32_t* ea = reinterpret_cast<int32_t*>(ws + p.off_ea);
    int32_t* eb = reinterpret_cast<int32_t*>(ws + p.off_eb);

    // op(A)(i, k) at A[i*rs + k*ks]; op(B) as the rows of its transpose: B^T(j, k).
    const int64_t a_rs = oa == 'N' ? 1 : lda, a_ks = oa == 'N' ? lda : 1;
    const int64_t b_rs = ob == 'N' ? ldb : 1, b_ks = ob == 'N' ? 1 : ldb;

    if (crt) {
        // op(A)'s rows and op(B)'s columns prepared in the workspace, then their product
        const CrtLines ops[2] = {{A, m, a_rs, a_ks, ws + p.off_a}, {B, n, b_rs, b_ks, ws + p.off_b}};
        rc = crt_prepare(ops, 2, k, slices, st);
        if (!rc) rc = crt_multiply(m, n, k, slices, alpha, ws + p.off_a, ws + p.off_b, beta, C, ldc, ws + p.off_w, st);
        return rc;
    }
    // Row exponents of op(A), column exponents of op(B), then the slices (the
    // padding is written as zeros by the same kernels).  The chunk maxima lie
    // where the slices go: a chunk has at least 32 k, 8 bytes of maximum
    // against 32 bytes of the smallest slice.
    const auto side = [&](const double* x, int64_t rows, int64_t rs, int64_t ks, int8_t* out, int32_t* e,
                          int64_t rows_p, int64_t slice_bytes) {
        OzSide o{x, rows, rs, ks, reinterpret_cast<double*>(out), ks == 1 ? 256 : 32, 0, 0, e, out, rows_p, slice_bytes};
        while ((k + o.kchunk - 1) / o.kchunk > 4096) o.kchunk *= 2;  // bounds the grid and the reduction
        o.nchunk = (uint32_t)((k + o.kchunk - 1) / o.kchunk);
        const int64_t per = ks == 1 ? NT / 16 : NT;
        o.groups = (uint32_t)((rows + per - 1) / per);
        return o;
    };
    const OzSide da = side(A, m, a_rs, a_ks, sa, ea, p.Mp, p.a_slice);
    const OzSide db = side(B, n, b_rs, b_ks, sb, eb, p.Np, p.b_slice);
    const int64_t max_a = (int64_t)da.groups * da.nchunk, max_b = (int64_t)db.groups * db.nchunk;
    const uint32_t nkt = (uint32_t)((p.Kp + OS_K - 1) / OS_K);
    const int64_t sl_a = p.Mp / OS_R * nkt, sl = sl_a + p.Np / OS_R * nkt;
    const int64_t sl_y = (sl >> 23) + 1;  // keeps a dimension below 2^32 threads
    if (max_a + max_b >= (int64_t)1 << 24 || sl > INT32_MAX)
        return fail(DG_ERR_UNSUPPORTED, "dg_ozaki_dgemm: matrix too large for one slicing launch");
    hipLaunchKernelGGL(oz_partial_max_kernel, dim3((unsigned)(max_a + max_b)), dim3(NT), 0, st, da, db, k,
                       (uint32_t)max_a);
    DG_LAUNCH_CHECK();
    hipLaunchKernelGGL(oz_exponent_kernel, dim3((unsigned)((p.Mp + p.Np) / 64)), dim3(NT), 0, st, da, db);
    DG_LAUNCH_CHECK();
    hipLaunchKernelGGL(bf16 ? oz_slice_kernel<true> : oz_slice_kernel<false>,
                       dim3((unsigned)((sl + sl_y - 1) / sl_y), (unsigned)sl_y), dim3(NT), 0, st, da, db, k, p.Kp,
                       slices, bits, nkt, (uint32_t)sl_a, (uint32_t)sl);
    DG_LAUNCH_CHECK();
    // INT8 products: each launch computes up to plane_batch groups into
    // planes, then the combine adds them into W (or, after the last group, C).
    std::vector<OzGroup> groups;
    if (!make_groups(sched, p.esz, groups))
        return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: internal error: product schedule without group form");
    const int ng = (int)groups.size();
    const int batch = (int)p.plane_batch;
    for (int i = 0; i < ng; ++i) groups[i].plane = i % batch;
    // entries ng.. : the same groups in launch order, each batch's longest first
    groups.reserve(2 * (size_t)ng);
    groups.insert(groups.end(), groups.begin(), groups.begin() + ng);
    for (int g0 = 0; g0 < ng; g0 += batch)
        std::stable_sort(groups.begin() + ng + g0, groups.begin() + ng + std::min(ng, g0 + batch),
                         [](const OzGroup& a, const OzGroup& b) {
                             return (int64_t)a.count * a.nks.d > (int64_t)b.count * b.nks.d;
                         });
    TableUseScope uses{st};  // after the launches below return
    const OzGroup* dgroups = static_cast<const OzGroup*>(cached_table(groups.data(), groups.size() * sizeof(OzGroup), st));
    if (!dgroups) return DG_ERR_ALLOC;
    const int64_t tiles = (p.Mp / BM) * (p.Np / BN);
    if (tiles * p.plane_batch > INT32_MAX || (p.Mp / 4) * p.Np > UINT32_MAX)
        return fail(DG_ERR_INVALID, "dg_ozaki_dgemm: too many tiles");
    OzPlaneArgs g{};
    g.a = sa; g.b = sb; g.planes = reinterpret_cast<int32_t*>(ws + p.off_planes);
    g.Mp = p.Mp; g.rb = p.Kp * p.esz; g.a_slice = p.a_slice; g.b_slice = p.b_slice; g.plane = p.Mp * p.Np;
    double* W = reinterpret_cast<double*>(ws + p.off_w);
    const uint32_t total = (uint32_t)((p.Mp / 4) * p.Np);
    const FastDiv dqm = make_fastdiv((uint32_t)(p.Mp / 4));
    for (int g0 = 0; g0 < ng; g0 += batch) {
        const int cnt = std::min(batch, ng - g0);
        g.jobs = dgroups + ng + g0;
        int64_t longest = 0, sum = 0;
        for (int i = g0; i < g0 + cnt; ++i) {
            const int64_t steps = (int64_t)groups[i].count * groups[i].nks.d;
            longest = std::max(longest, steps);
            sum += steps;
        }
        const bool small = small_tiles(tiles * cnt, longest, tiles * sum);
        const int split = small ? BM / ST : 1;
        g.tiles_m = (int32_t)(p.Mp / BM) * split; g.tiles_n = (int32_t)(p.Np / BN) * split;
        const dim3 grid((unsigned)(tiles * cnt * split * split)), wg(small ? SCNT : CNT);
        const dim3 cgrid((total + 255) / 256);
        if (bf16) {
            hipLaunchKernelGGL(small ? oz_plane_small_kernel<true> : oz_plane_kernel<true>, grid, wg, kCrtLds, st, g);
            hipLaunchKernelGGL(oz_combine_kernel<true>, cgrid, dim3(256), 0, st, g.planes, g.plane, dgroups, g0,
                               g0 + cnt, ng, bits, W, p.Mp, m, n, ea, eb, alpha, beta, C, ldc, dqm, total);
        } else {
            hipLaunchKernelGGL(small ? oz_plane_small_kernel<false> : oz_plane_kernel<false>, grid, wg, kCrtLds, st, g);
            hipLaunchKernelGGL(oz_combine_kernel<false>, cgrid, dim3(256), 0, st, g.planes, g.plane, dgroups, g0,
                               g0 + cnt, ng, bits, W, p.Mp, m, n, ea, eb, alpha, beta, C, ldc, dqm, total);
        }
        DG_LAUNCH_CHECK();
    }
    return DG_OK;
}

}  // extern "C"
