// Internal helpers shared by the HIP sources of libdgamd: error state,
// HIP call checking, device checks and the device table cache.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <algorithm>
#include <vector>

#include "dgamd.h"

namespace dg {

// Sets the calling thread's last-error message and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// Returns DG_OK when the current device is a gfx950 GPU.
int require_device();

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Normalises 'n','N','t','T','c','C' to 'N' or 'T'; returns 0 on a bad op.
inline char norm_op(char op) {
    switch (op) {
        case 'n': case 'N': return 'N';
        case 't': case 'T': case 'c': case 'C': return 'T';
        default: return 0;
    }
}

// Device-resident copy of a small host table (problem / segment descriptors).
// Identical tables (same bytes) share one device buffer, so repeated calls
// with the same arguments upload nothing.  Returns nullptr and sets the
// error on failure.  Uploading while `stream` is being captured into a HIP
// graph is refused: tables must be built before capture; a table looked up
// during a capture stays resident for the life of the process (the graph
// holds its address), and so do the first 128 of at most 64 KiB of a device.
// Beyond 256 others per device, a new table reuses the buffer of the least
// recently used of them whose last use has completed on the device, found by
// event queries (nothing waits, nothing is freed).
const void* cached_table(const void* host, size_t bytes, hipStream_t stream);

// Marks the kernels that read this thread's tables looked up since the last
// mark as enqueued on `stream`: records the completion event that a later
// reuse of those buffers waits for.  TableUseScope calls it when a call that
// looks up tables returns, after its launches.
void table_uses_enqueued(hipStream_t stream);
struct TableUseScope {
    hipStream_t stream;
    ~TableUseScope() { table_uses_enqueued(stream); }
};

#define DG_HIP(call)                                                            \
    do {                                                                        \
        hipError_t e_ = (call);                                                 \
        if (e_ != hipSuccess)                                                   \
            return ::dg::fail(DG_ERR_HIP, "%s:%d %s: %s", __FILE__, __LINE__,   \
                              #call, hipGetErrorString(e_));                    \
    } while (0)

#define DG_LAUNCH_CHECK()                                                       \
    do {                                                                        \
        hipError_t e_ = hipGetLastError();                                      \
        if (e_ != hipSuccess)                                                   \
            return ::dg::fail(DG_ERR_HIP, "%s:%d kernel launch: %s", __FILE__,  \
                              __LINE__, hipGetErrorString(e_));                 \
    } while (0)

// ---------------------------------------------------------------- GEMM core
// One K-segment of an output tile's reduction: op(A) rows x klen starting at
// `a` (leading dimension lda of the stored matrix) times op(B) klen x cols at
// `b`.  A problem walks its segments in order; Cannon rotations and SUMMA
// panels are segments whose pointers point into other ranks' tiles.
struct Seg {
    const double* a;
    const double* b;
    int64_t lda;
    int64_t ldb;
    int64_t klen;
};

struct Prob {
    int64_t m, n;
    double* c;
    int64_t ldc;
    double alpha, beta;
    int32_t seg0, nseg;    // segment range in the segment table
    int32_t tile0;         // first tile id of this problem in its list
    // direct-to-LDS kernel: bit 0 (bit 1) set when the row-contiguous A (B)
    // starts 8 bytes past a 16-byte boundary; its loads then start one row
    // earlier and the tile grid runs over rows + 1; register-staged kernel:
    // kByElements or 0
    int32_t shift;
};
constexpr int32_t kByElements = 4;  // load single elements instead of pairs

// Division of 32-bit unsigned integers by a launch constant d >= 1 with
// one high multiply, a subtract, an add and two shifts (Granlund and
// Montgomery, "Division by invariant integers using multiplication", PLDI
// 1994, figure 4.1): l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1,
// t = mulhi(m, n), n / d = (t + ((n - t) >> min(l, 1))) >> max(l - 1, 0).
struct FastDiv {
    uint32_t d, m, s1, s2;
};

inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f{};
    uint32_t l = 0;
    while (l < 32 && ((uint64_t)1 << l) < d) ++l;
    f.d = d;
    f.m = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - d)) / d + 1);
    f.s1 = l < 1 ? l : 1;
    f.s2 = l > 1 ? l - 1 : 0;
    return f;
}

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) {
    const uint32_t t = __umulhi(f.m, n);
    return (t + ((n - t) >> f.s1)) >> f.s2;
}

// A launch dimension holds less than 2^32 threads (a launch past that is
// refused).  Workgroups for `items` threads' work in a kernel that loops over
// what they leave:
inline unsigned looped_blocks(int64_t items, int threads) {
    const int64_t blocks = (items + threads - 1) / threads, most = (((int64_t)1 << 32) - 1) / threads;
    return (unsigned)std::max<int64_t>(1, std::min(blocks, most));
}
// Workgroups of at most 64 threads for `chunks` run chunks (x, spilling into
// z; at most 2^31) by `cols` column groups:
inline dim3 run_grid(int64_t chunks, unsigned cols) {
    const int64_t z = (chunks + (1 << 25) - 1) >> 25;
    return dim3((unsigned)((chunks + z - 1) / z), cols, (unsigned)z);
}

// `chunks` run chunks cut into eight ranges, one for each XCD (workgroups go
// to the XCDs in turn, by their number): a launch of 8 * eighth(chunks)
// workgroups in x, of which number x takes chunk eighth_chunk(x, eighth(chunks)),
// if there is one.
inline uint32_t eighth(uint32_t chunks) { return (chunks + 7) / 8; }
__host__ __device__ __forceinline__ uint32_t eighth_chunk(uint32_t x, uint32_t per) { return (x & 7) * per + (x >> 3); }

// Tile scheduling of the FP64 GEMM launch.
enum {
    DG_GEMM_MODE_ROUND_ROBIN = 0,  // tile = workgroup id (tiles dealt round-robin over XCDs)
    DG_GEMM_MODE_XCD = 1,          // each XCD gets one contiguous tile range (L2 reuse)
    DG_GEMM_MODE_PERSISTENT = 2,   // CU-count workgroups pull tiles from an atomic counter
};

// Tile choices of an FP64 GEMM batch.
enum {
    DG_GEMM_TILE_AUTO = -1,          // the one whose estimated time is least
    DG_GEMM_TILE_DIRECT = 0,         // direct-to-LDS kernels where they apply, as 128x128 elsewhere
    DG_GEMM_TILE_128x128 = 1,        // register-staged kernel, uneven problems cut into whole tiles and strips
    DG_GEMM_TILE_128x128_WHOLE = 2,  // the same, uncut
    DG_GEMM_TILE_64x64 = 3,          // register-staged kernel
    DG_GEMM_TILE_32x32 = 4,          // register-staged kernel
    DG_GEMM_TILES = 5,
};
// The choice that DG_GEMM_TILE forces, FP32 included: "direct", "128x128",
// "128x128whole", "64x64" or "32x32"; DG_GEMM_TILE_AUTO when it is unset or
// anything else.
int forced_tile();

// Whether an FP32 product of m rows on the register-staged kernels runs
// sgemm_short_kernel: K less than one 32-deep stage of sgemm_kernel, or less
// than two with few rows in tiles that are not whole.  Share of sgemm_kernel's
// time over 15 outputs in all layouts: K = 1 0.73, 8 0.81, 16 0.80, none above
// 1.04; K = 32 0.90, but 130 x 60000 1.07 and 2000 x 2001 1.04; 37 x 400000 x 48
// 0.56.
inline bool sgemm_is_short(int64_t m, int64_t k) { return k < 32 || (k < 64 && m < 128 && m % 64); }

// Launches the FP64 MFMA GEMM over `probs` (host vector; uploaded through
// the table cache).  All problems share opA/opB.
int launch_gemm_f64(char opA, char opB, const std::vector<Prob>& probs, std::vector<Seg> segs, hipStream_t stream,
                    int mode);

// A batch split by kernel.  With DG_GEMM_TILE_DIRECT, the direct-to-LDS
// kernels take a problem when every segment has K > 0 and even leading
// dimensions, its k-contiguous operand (A with opA = T, B with opB = N) has
// 16-byte aligned bases and even K, and its row-contiguous operand (A with
// opA = N, B with opB = T) has 8-byte aligned bases with the same offset
// within 16 bytes in every segment; the register-staged kernel takes the
// others, and all of them with the other choices.  DG_GEMM_TILE_AUTO estimates
// each choice's time from its tiles and takes the least: the larger the
// tiles, the less operand traffic, but the more CUs stay idle and the more of
// the work is padding (DG_GEMM_TILE forces a choice, DG_GEMM_NO_DMA routes
// everything to the register-staged kernel).  Every kernel and tile sums an
// element in the same order, so a problem gives the same bits alone, in any
// batch and on any tile, with one exception: a sum of -0 (negative products
// that all underflow) comes out +0 where zeros follow it.  Each segment's k is
// padded with them to whole stages, 8 deep in the direct-to-LDS kernels, 16 on
// 128x128 and 64x64 tiles and 32 on 32x32 ones, and the tile depends on the batch.
// Direct-to-LDS problems whose tiles are all interior (no row shift, m and n
// multiples of 128, whole k-steps, an even step count) go to `dma`, which
// the A-in-registers kernel runs; the others go to `dmae` (the edge-handling
// kernel).  With split_edges, a direct-to-LDS problem with edges and at
// least 8 interior tiles is cut into sub-problems: an interior block on
// `dma` (a row-shifted problem's interior starts at its row 127), and strips
// around it on the register-staged kernel (on `dmae` under
// DG_GEMM_NO_NARROW).  The sub-problems' segments are appended to `segs`
// (which starts with the input segments).
// Register-staged problems and strips go to gen[0] (128x128 tiles), gen[1]
// (64x64) or gen[2] (32x32): the choice's own, or a smaller one where they are
// at most 96 or 32 rows or columns.
struct GemmBatch {
    std::vector<Prob> dma, dmae, gen[3];  // tile ranges assigned per list
    int tiles_dma = 0, tiles_dmae = 0, tiles_gen[3] = {0, 0, 0};
    std::vector<Seg> segs;                // the segment table all lists index
    bool empty() const { return dma.empty() && dmae.empty() && gen[0].empty() && gen[1].empty() && gen[2].empty(); }
};
int prepare_gemm(char opA, char opB, const std::vector<Prob>& probs, std::vector<Seg> segs, GemmBatch& out,
                 bool split_edges = true, int tile = DG_GEMM_TILE_AUTO);

// Whether two tile choices of one batch came out alike: the same lists of the
// same problems.
bool same_lists(const GemmBatch& a, const GemmBatch& b);

// Times the scheduling modes of each tile choice in `choices` and keeps the
// fastest: trial(choice, mode, &ms) runs one and returns a status.  The best of
// three runs in a row counts.  A variant's first run is cold (up to 1.34 times
// its steady time: the 7 x 5 batch of 5000 with 256 products, 6.1 against 5.5 ms
// for its best variant), so only one that is half as slow again as the best so
// far, and 0.2 ms, ends there.  25 batches in four processes each: the choice is
// 0.7 % behind the best one on average (0.8 % with three runs of all); taking turns
// in rounds, with the second run of a pair or the settled run of up to eight
// counting, came out 1.3 to 1.4 % behind.
template <class F>
int fastest_variant(const std::vector<int>& choices, const F& trial, int* choice, int* mode) {
    float best = 1e30f;
    for (int c : choices)
        for (int v : {(int)DG_GEMM_MODE_XCD, (int)DG_GEMM_MODE_ROUND_ROBIN, (int)DG_GEMM_MODE_PERSISTENT}) {
            float least = 1e30f;
            for (int run = 0; run < 3; ++run) {
                float ms = 0.f;
                const int rc = trial(c, v, &ms);
                if (rc) return rc;
                least = std::min(least, ms);
                if (least > std::max(1.5f * best, best + 0.2f)) break;
            }
            if (least < best) {
                best = least;
                *choice = c;
                *mode = v;
            }
        }
    return DG_OK;
}

// The same batch with its tables resident on the device.
struct GemmBatchDev {
    const Prob *dma = nullptr, *dmae = nullptr, *gen[3] = {nullptr, nullptr, nullptr};
    int ndma = 0, ndmae = 0, ngen[3] = {0, 0, 0};
    int tiles_dma = 0, tiles_dmae = 0, tiles_gen[3] = {0, 0, 0};
    const Seg* segs = nullptr;
    void set_counts(const GemmBatch& h) {
        ndma = (int)h.dma.size();
        ndmae = (int)h.dmae.size();
        tiles_dma = h.tiles_dma;
        tiles_dmae = h.tiles_dmae;
        for (int w = 0; w < 3; ++w) {
            ngen[w] = (int)h.gen[w].size();
            tiles_gen[w] = h.tiles_gen[w];
        }
    }
};
// Device half.  The persistent mode needs a device int `counter`, which it
// zeroes with a kernel before each launch (graph safe).  `dma` runs the
// A-in-registers kernel (the lean direct-to-LDS kernel under
// DG_GEMM_NO_AREG), `dmae` the edge-handling direct-to-LDS kernel, `gen` the
// register-staged kernel; one launch per non-empty list.
int launch_gemm_f64_dev(char opA, char opB, int mode, const GemmBatchDev& b, int* counter, hipStream_t stream);

// C[x] = beta*C[x] over an m x n column-major matrix (beta == 0 writes 0).
int launch_scale(int64_t m, int64_t n, double beta, double* C, int64_t ldc, hipStream_t stream);

// Smallest CRT moduli count (2..16) whose scaling reaches q = 53 bits for
// inner dimension k (16 when none does).
int crt_moduli_for_fp64(int64_t k);

// Ozaki scheme II in two parts.  A prepared operand holds the residues and
// line exponents of `rows` lines of length k (crt_operand_bytes bytes);
// crt_prepare builds one or two from lines x[i*rs + k*ks]; crt_multiply forms C = alpha op(A) op(B) + beta C
// from prepared op(A) rows and op(B) columns with a digit buffer of
// crt_digit_bytes bytes.  Buffers 256-byte aligned.
int64_t crt_operand_bytes(int64_t rows, int64_t k, int nmod);
int64_t crt_digit_bytes(int64_t m, int64_t n, int nmod);
struct CrtLines {
    const double* x;
    int64_t rows, rs, ks;
    void* operand;  // receives the prepared operand
};
int crt_prepare(const CrtLines* ops, int count, int64_t k, int nmod, hipStream_t st);
int crt_multiply(int64_t m, int64_t n, int64_t k, int nmod, double alpha, const void* a_op, const void* b_op,
                 double beta, double* C, int64_t ldc, void* digits, hipStream_t st);

}  // namespace dg
