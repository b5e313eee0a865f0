// One operand of a register-staged GEMM tile (gemm_f64_kernel,
// sgemm_kernel): global memory -> registers -> LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace dg {

typedef double dv2 __attribute__((ext_vector_type(2)));
typedef float fv4 __attribute__((ext_vector_type(4)));

// 16 bytes of a matrix at whatever alignment its elements have: one load all
// the same (the hardware takes unaligned global loads).
template <typename T> struct Vec16;
template <> struct Vec16<double> {
    typedef dv2 type;
    typedef dv2 any __attribute__((aligned(8)));
};
template <> struct Vec16<float> {
    typedef fv4 type;
    typedef fv4 any __attribute__((aligned(4)));
};

// Grid of one workgroup of 256 threads per tile: a launch dimension holds
// less than 2^32 threads, so tiles past 2^22 go on a second one (the last row
// may run over `tiles`).
inline dim3 tile_grid(int tiles) {
    const unsigned x = tiles < (1 << 22) ? (unsigned)tiles : 1u << 22;
    return dim3(x, ((unsigned)tiles + x - 1) / x);
}

// BK-deep stages of ROWS rows for a workgroup of 256 threads, loaded in runs
// of E elements (16 bytes) at any alignment -- a run per load instead of
// single elements is what lets odd leading dimensions run like even ones --
// and stored to LDS in the direction memory has, so that the stores and the
// fragment reads spread over the banks (4096^3 on FP64 128x128 tiles: conflicts
// in 3 % of a CU's cycles).
//  * KC, element (row, k) at base[k + row*ld]: a thread takes the run at
//    k = E*(t % CH) of rows t/CH + RPP*q; LDS [row][k], rows padded by a run.
//  * else, element (row, k) at base[row + k*ld]: a thread takes the run at row
//    E*(t % HP) of k t/HP + KPP*q; LDS [k][row], k-rows padded by 128/E bytes
//    (the k-rows that one MFMA reads, E apart, then fall in different halves
//    of the banks).
// Rows past the end are read from the last row; they feed only outputs that
// are never stored.  In a whole stage that is not a segment's last, every run
// is inside the matrix: one that starts at the last row ends in the next k's
// first rows or in the columns' padding (ld >= E - 1).  A segment's last stage
// is read by elements (read_last), with k past the end turned into zeros,
// unless it is whole and no run can start at a last row (KC, or a full tile).
// A whole stage uses no vector instruction but the memory ones: a scalar base
// that moves and 32-bit lane offsets that stay.  An FP64 MFMA runs on the
// vector ALU's own pipes, and 1.4 to 3.7 vector instructions per MFMA cost a
// fifth of the rate.  The compiler counts loads in flight only along straight
// code, so whole stages also have no branch around their loads (with one it
// waited for all of them every stage).
template <typename T, bool KC, int ROWS, int BK>
struct Staged {
    static constexpr int E = 16 / sizeof(T), S = sizeof(T);
    static constexpr int CH = BK / E, RPP = 256 / CH;          // KC
    static constexpr int HP = ROWS / E, KPP = 256 / HP;        // else
    static constexpr int NL = ROWS * BK / (256 * E);           // loads per thread and stage
    static constexpr int LROW = KC ? (BK + E) * S : ROWS * S + 128 / E;  // bytes
    static constexpr int BYTES = KC ? ROWS * LROW : BK * LROW;
    static_assert(256 % CH == 0 && 256 % HP == 0 && NL * 256 * E == ROWS * BK, "whole loads");
    typedef typename Vec16<T>::type vec;
    typedef __attribute__((address_space(1))) const typename Vec16<T>::any gvec;
    typedef __attribute__((address_space(1))) const T gelem;

    const T* base;     // the tile's first row at the next stage's first k (uniform)
    int64_t ld;
    uint32_t off[NL];  // bytes from it to this thread's runs

    // Run q of thread t: its row within the tile, its k within the stage, and
    // its place in a whole stage, bytes from the stage's first element.
    static constexpr __host__ __device__ __forceinline__ int row(int t, int q) { return KC ? t / CH + RPP * q : E * (t % HP); }
    static constexpr __host__ __device__ __forceinline__ int kk(int t, int q) { return KC ? E * (t % CH) : t / HP + KPP * q; }
    static __host__ __device__ __forceinline__ uint32_t offset(int t, int q, int64_t ld, int rows) {
        const uint32_t r = row(t, q) < rows ? row(t, q) : rows - 1, k = kk(t, q);
        return (uint32_t)S * (KC ? r * (uint32_t)ld + k : k * (uint32_t)ld + r);
    }
    // Where element e of it is read in a stage of `left` real k, in elements.
    static __host__ __device__ __forceinline__ int64_t last_offset(int t, int q, int e, int64_t ld, int rows, int left) {
        const int r0 = row(t, q) + (KC ? 0 : e), k0 = kk(t, q) + (KC ? e : 0);
        const int64_t r = r0 < rows ? r0 : rows - 1, k = k0 < left ? k0 : left - 1;
        return KC ? r * ld + k : k * ld + r;
    }

    // At a segment's first k; the tile has `rows` rows from row0 on.
    __device__ __forceinline__ void start(const T* x, int64_t ld_, int64_t row0, int rows) {
        ld = ld_;
        base = x + row0 * (KC ? ld : 1);
#pragma unroll
        for (int q = 0; q < NL; ++q) off[q] = offset(threadIdx.x, q, ld, rows);
    }
    __device__ __forceinline__ void advance() {
        base += KC ? BK : BK * ld;
        asm volatile("" : "+s"(base));  // stays a scalar: not folded into vector address increments
    }
    // Run q of a whole stage (all of them, then advance).
    __device__ __forceinline__ void read(vec (&v)[NL], int q) {
        asm volatile("" : "+v"(off[q]));  // stays 32 bits: the load adds it to the scalar base itself
        v[q] = *(gvec*)((const char*)base + off[q]);
    }
    __device__ __forceinline__ void read(vec (&v)[NL]) {
#pragma unroll
        for (int q = 0; q < NL; ++q) read(v, q);
        advance();
    }
    // The segment's last stage, `left` <= BK of its k real (or any stage of a
    // matrix that read() does not take).
    __device__ __forceinline__ void read_last(vec (&v)[NL], int left, int rows) {
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int e = 0; e < E; ++e) v[q][e] = *(gelem*)(base + last_offset(threadIdx.x, q, e, ld, rows, left));
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int e = 0; e < E; ++e) v[q][e] = kk(threadIdx.x, q) + (KC ? e : 0) < left ? v[q][e] : T(0);
        advance();
    }
    static __device__ __forceinline__ void store(char* s, const vec (&v)[NL], int q) {
        const int r = row(threadIdx.x, q), k = kk(threadIdx.x, q);
        *reinterpret_cast<vec*>(s + (KC ? r * LROW + k * S : k * LROW + r * S)) = v[q];
    }
    static __device__ __forceinline__ void store(char* s, const vec (&v)[NL]) {
#pragma unroll
        for (int q = 0; q < NL; ++q) store(s, v, q);
    }
    // Whether read() takes a matrix: elements on their own alignment, and rows
    // (or k) neither so far apart that a lane's offset leaves 32 bits nor so
    // close that a run at the last row would pass the matrix's end.  Others are
    // read by elements throughout, at 0.65 (FP64) or 0.55 (FP32) of the rate.
    static constexpr int64_t kMaxLd =
        ((((int64_t)1 << 32) - 1) / S - ((KC ? BK : ROWS) - E)) / ((KC ? ROWS : BK) - 1);
    static bool takes(const T* x, int64_t ld) {
        return !(reinterpret_cast<uintptr_t>(x) & (S - 1)) && ld <= kMaxLd && (KC || ld >= E - 1);
    }
};

}  // namespace dg
