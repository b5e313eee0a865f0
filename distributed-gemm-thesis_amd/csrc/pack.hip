// Bit-exact layout kernels: 2D-block and block-cyclic pack/unpack, strided
// block copy and the 2.5D layer reduction.  All are HBM-bound copies.  A
// workgroup (one wave) moves one chunk of one column run (or, for short
// runs, the same chunk of several columns), one 16-byte vector per thread,
// and the grid walks row chunks fastest: every thread has exactly one load
// in flight and the workgroups resident at any moment cover a compact
// window of both buffers, which is what keeps the HBM queues full.
// Measured on MI355X for a 16384^2 column copy: 6.3 TB/s in this shape with
// 256-thread workgroups, against 5.5-5.8 TB/s for four columns or two
// vectors per thread and 4.4-4.9 TB/s for grid-stride loops; nontemporal
// accesses and one-wave workgroups then took the kernels from 73-78 % to
// 78-83 % of the 8 TB/s peak (a plain 2 GiB copy: 79 -> 83.5 %).  Runs off
// 16-byte alignment: 5003 x 7001 at 4.9-6.2 TB/s (element by element
// 3.8-5.2 TB/s).
#include "dg_internal.hpp"

#include <algorithm>

namespace dg {

namespace {

constexpr int kThreads = 64;  // one wave per workgroup
constexpr int kMaxParts = 256;

typedef __attribute__((address_space(1))) const double gcdouble;
typedef __attribute__((address_space(1))) double gdouble;
typedef double dv2 __attribute__((ext_vector_type(2)));

// Every byte these kernels move is read once and written once.
template <typename G>
__device__ __forceinline__ void move_nt(const G* src, G* dst) {
    __builtin_nontemporal_store(__builtin_nontemporal_load(src), dst);
}

// Copies one chunk of `len` <= lanes*E elements (E = 16/sizeof(T)) with the
// calling thread's `lane` of `lanes`: the first elements up to a 16-byte
// boundary of the destination singly, then one 16-byte vector per lane, then
// the tail elements.  The vector loads take any element's alignment, so only
// the stores have to be aligned.  LINES: every run starts and ends on a
// 128-byte line of both buffers; only then does a load carry the nontemporal
// hint (16384^2: 1-3 % faster), because two workgroups read a line that two
// runs share (5003 x 7001, runs of 112-715 rows, with the hint 113-140 us,
// without 90-119 us; element by element, nontemporal, 107-146 us).
template <bool LINES, typename T>
__device__ __forceinline__ void copy_chunk(const T* src, T* dst, int64_t len, int lane, int lanes) {
    typedef __attribute__((address_space(1))) const T gcT;
    typedef __attribute__((address_space(1))) T gT;
    typedef T vT __attribute__((ext_vector_type(16 / sizeof(T))));
    typedef vT uT __attribute__((aligned(sizeof(T))));
    typedef __attribute__((address_space(1))) const uT gcV;
    typedef __attribute__((address_space(1))) vT gV;
    constexpr int E = 16 / sizeof(T);
    int64_t p = (int64_t)(((16 - (reinterpret_cast<uintptr_t>(dst) & 15)) & 15) / sizeof(T));
    if (p > len) p = len;
    const int64_t nv = (len - p) / E;
    const int64_t t0 = p + nv * E;
    if (lane < nv) {
        gcV* x = (gcV*)(src + p) + lane;
        const vT v = LINES ? __builtin_nontemporal_load(x) : *x;
        __builtin_nontemporal_store(v, (gV*)(dst + p) + lane);
    }
    if (lane < p) move_nt((gcT*)src + lane, (gT*)dst + lane);
    if (lane < len - t0) move_nt((gcT*)src + t0 + lane, (gT*)dst + t0 + lane);
}

// Workgroup shape for runs of `run` elements: `lanes` threads (a power of
// two, 16..kThreads) per column chunk of lanes*E elements, kThreads/lanes
// columns per workgroup.
struct RunShape {
    int lanes_log2;
    int64_t chunk;    // elements per column chunk
    int64_t chunks;   // chunks per run
    int cols_per_wg;
};

RunShape run_shape(int64_t run, int E) {
    RunShape r{};
    const int64_t vecs = (run + E - 1) / E;
    int l2 = 4;
    while ((1 << l2) < vecs && (1 << l2) < kThreads) ++l2;
    r.lanes_log2 = l2;
    r.chunk = (int64_t)(1 << l2) * E;
    r.chunks = run > 0 ? (run + r.chunk - 1) / r.chunk : 1;
    r.cols_per_wg = kThreads >> l2;
    return r;
}

unsigned col_groups(int64_t cols, int cols_per_wg) {
    int64_t g = (cols + cols_per_wg - 1) / cols_per_wg;
    if (g > 65535) g = 65535;  // the kernels loop over the remaining column groups
    return (unsigned)(g < 1 ? 1 : g);
}

// Whether two addresses and a length in bytes are whole lines (or parts of
// `unit` bytes).
bool whole_lines(const void* a, const void* b, int64_t bytes, int unit = 128) {
    return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)bytes) & (unit - 1)) == 0;
}

struct Bands {
    int64_t off[kMaxParts + 1];
    int32_t cpre[kMaxParts + 1];  // first chunk of each band (prefix of its chunk counts)
    int n;
};

// Row band b (rows [off[b], off[b+1])) of every column: the packed index of
// global (r, c) in band b is off[b]*cols + (r - off[b]) + c*rows_b (tiles of
// one band are contiguous in rank order and share ld = rows_b).  The grid
// walks global columns top to bottom (blockIdx.x, blockIdx.z = chunk of the
// column across the bands, blockIdx.y = column group), so that the two bands
// that share a line of the global matrix are in flight together: unpacking
// band by band took 129 us for 5003 x 7001 in 7 bands, this order 111 us
// (5000 x 7000 in 5: 120 -> 88 us).  Where no line is shared (LINES),
// unpacking reads each band's packed region front to back (blockIdx.x = chunk
// of the band's column run, blockIdx.z = band; 16384^2 in 4: 667 us, global
// order 684 us).
template <bool PACK, bool LINES>
__global__ __launch_bounds__(kThreads) void block2d_kernel(const double* __restrict__ src, double* __restrict__ dst,
                                                           int64_t ldg, int64_t cols, Bands bands, int lanes_log2) {
    int b;
    int64_t q0;  // first row of the chunk within its band
    const int64_t chunk = (int64_t)2 << lanes_log2;
    if (PACK || !LINES) {
        const int64_t x = (int64_t)blockIdx.z * gridDim.x + blockIdx.x;
        int lo = 0, hi = bands.n - 1;  // band b with cpre[b] <= x < cpre[b+1]
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (bands.cpre[mid] <= x) lo = mid; else hi = mid - 1;
        }
        b = lo;
        q0 = (x - bands.cpre[b]) * chunk;
    } else {
        b = blockIdx.z;
        q0 = (int64_t)blockIdx.x * chunk;
    }
    const int64_t r0 = bands.off[b];
    const int64_t rb = bands.off[b + 1] - r0;
    const int64_t len = rb - q0 < chunk ? rb - q0 : chunk;
    if (len <= 0) return;
    const int lane = threadIdx.x & ((1 << lanes_log2) - 1);
    const int cpw = kThreads >> lanes_log2;
    const int64_t band_base = r0 * cols;
    for (int64_t c = (int64_t)blockIdx.y * cpw + (threadIdx.x >> lanes_log2); c < cols; c += (int64_t)gridDim.y * cpw) {
        const int64_t g = r0 + q0 + c * ldg;
        const int64_t p = band_base + q0 + c * rb;
        copy_chunk<LINES>(PACK ? src + g : src + p, PACK ? dst + p : dst + g, len, lane, 1 << lanes_log2);
    }
}

// numroc(n, b, p, 0, procs) = base*b + (b if p < extra, rem if p == extra,
// else 0) with full = n / b, rem = n % b, base = full / procs, extra = full
// % procs, and its prefix over the processes before p.
struct Numroc {
    uint32_t b, rem, base, extra;
};

Numroc make_numroc(uint32_t n, uint32_t b, uint32_t procs) {
    const uint32_t full = n / b;
    return Numroc{b, n - full * b, full / procs, full % procs};
}

__device__ __forceinline__ uint32_t local_extent(const Numroc& r, uint32_t p) {
    return r.base * r.b + (p < r.extra ? r.b : (p == r.extra ? r.rem : 0u));
}
__device__ __forceinline__ uint32_t local_prefix(const Numroc& r, uint32_t p) {
    return p * r.base * r.b + (p < r.extra ? p : r.extra) * r.b + (p > r.extra ? r.rem : 0u);
}

// Block-cyclic geometry (rows, cols, mb, nb < 2^31; source process 0), all
// in kernel arguments, so that a thread's first load waits on no table read.
struct Cyclic {
    int64_t ldg;
    uint32_t rows, cols, mb, nb, P, Q;
    Numroc nr, nc;            // row and column distributions
    FastDiv dP, dQ, dnb, dchunks;
};

// Row block ib (rows [ib*mb, ...)) of column c belongs to process row
// ib % P at local row (ib / P)*mb; column c to process column (c/nb) % Q at
// local column ((c/nb)/Q)*nb + c % nb.  The local matrix of rank (pr, pc)
// (column-major, ld = its local rows) starts at rowpre(pr)*cols +
// lrows(pr)*colpre(pc) in the packed buffer.  Both directions walk the global
// columns top to bottom (blockIdx.x, blockIdx.z = row block * chunks + chunk,
// blockIdx.y = column group).  Unpacking in this order, against each rank's
// local matrix front to back: 5003 x 7001 on 3 x 2 in blocks of 128 x 96
// 110 -> 106 us, 16384^2 on 4 x 4 in 512 x 512 649 -> 651 us.
// Unpacking row blocks of 16 to 32, of which most lines hold parts of two,
// each XCD takes an eighth of the column (per_xcd, of eighth()), so that both
// parts of a line meet in one L2: written from two XCDs a little apart they
// cost more than far apart, as in the packed order.  12288 x 7168 on 2 x 2 in
// 16 x 64, ldg 12291: 512 us (block by block over the XCDs 810, packed order
// 590); over 1368 unpackings of such blocks 0.86 of the time on average, 0.66 of
// the packed order's.  Blocks of 48 and more gain nothing, those of 8 lose 2 %,
// and those that share no half line 3 to 5 %.
template <bool PACK, bool LINES>
__global__ __launch_bounds__(kThreads) void cyclic_kernel(const double* __restrict__ src, double* __restrict__ dst,
                                                          Cyclic g, int lanes_log2, uint32_t per_xcd) {
    const uint32_t chunk = 2u << lanes_log2;
    const uint32_t x = !PACK && !LINES && per_xcd ? eighth_chunk(blockIdx.x, per_xcd) : blockIdx.z * gridDim.x + blockIdx.x;
    const uint32_t blk = fdiv(x, g.dchunks);
    const uint32_t q0 = (x - blk * g.dchunks.d) * chunk;  // first row of the chunk within its row block
    const int lane = threadIdx.x & ((1 << lanes_log2) - 1);
    const uint32_t cpw = kThreads >> lanes_log2;
    if ((uint64_t)blk * g.mb + q0 >= g.rows || q0 >= g.mb) return;
    const uint32_t row0 = blk * g.mb + q0;
    uint32_t len = g.mb - q0 < chunk ? g.mb - q0 : chunk;
    if (g.rows - row0 < len) len = g.rows - row0;
    const uint32_t bq = fdiv(blk, g.dP), pr = blk - bq * g.P;
    const uint32_t lrows = local_extent(g.nr, pr);
    const int64_t rbase = (int64_t)local_prefix(g.nr, pr) * g.cols + bq * g.mb + q0;
    for (uint32_t c = blockIdx.y * cpw + (threadIdx.x >> lanes_log2); c < g.cols; c += gridDim.y * cpw) {
        const uint32_t jb = fdiv(c, g.dnb);
        const uint32_t jq = fdiv(jb, g.dQ), pc = jb - jq * g.Q;
        const uint32_t lcol = jq * g.nb + (c - jb * g.nb);
        const int64_t p = rbase + (int64_t)lrows * (local_prefix(g.nc, pc) + lcol);
        const int64_t at = row0 + c * g.ldg;
        copy_chunk<LINES>(PACK ? src + at : src + p, PACK ? dst + p : dst + at, len, lane, 1 << lanes_log2);
    }
}

// blockIdx.x, blockIdx.z = chunk of a column, blockIdx.y = column group.
template <bool LINES, typename T>
__global__ __launch_bounds__(kThreads) void copy_block_kernel(int64_t rows, int64_t cols, const T* __restrict__ src,
                                                              int64_t lds, T* __restrict__ dst, int64_t ldd,
                                                              int lanes_log2) {
    constexpr int E = 16 / sizeof(T);
    const int64_t chunk = (int64_t)E << lanes_log2;
    const int64_t r0 = ((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * chunk;
    const int64_t len = rows - r0 < chunk ? rows - r0 : chunk;
    if (len <= 0) return;
    const int lane = threadIdx.x & ((1 << lanes_log2) - 1);
    const int cpw = kThreads >> lanes_log2;
    for (int64_t c = (int64_t)blockIdx.y * cpw + (threadIdx.x >> lanes_log2); c < cols; c += (int64_t)gridDim.y * cpw)
        copy_chunk<LINES>(src + r0 + c * lds, dst + r0 + c * ldd, len, lane, 1 << lanes_log2);
}

// C[x] += partial[0*n + x] + partial[1*n + x] + ... in layer order, one pair
// per thread, the grid covering n (past 2^33 the kernel loops).  With n odd
// every second layer starts off 16-byte alignment: the pair accesses take any
// element's alignment, and the layers' loads (ODD) are plain ones, since a line
// may then serve two workgroups: 35026003 elements and one layer 119 us, with
// the nontemporal hint 125 us.  With n even the hint stays (70052006 elements,
// one layer: 249 us, without 253 us).
template <bool ODD>
__global__ __launch_bounds__(kThreads) void layer_reduce_kernel(double* __restrict__ C,
                                                                const double* __restrict__ partial, int64_t n,
                                                                int nlayers) {
    typedef dv2 uv2 __attribute__((aligned(8)));
    typedef __attribute__((address_space(1))) uv2 guv2;
    typedef __attribute__((address_space(1))) const uv2 gcuv2;
    gdouble* c = (gdouble*)C;
    gcdouble* p = (gcdouble*)partial;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t nv = n / 2;
    for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < nv + (n & 1); x += stride) {
        if (x < nv) {
            dv2 acc = __builtin_nontemporal_load((guv2*)(c + 2 * x));
            for (int l = 0; l < nlayers; ++l) {
                gcuv2* y = (gcuv2*)(p + (int64_t)l * n + 2 * x);
                acc += ODD ? *y : __builtin_nontemporal_load(y);
            }
            __builtin_nontemporal_store(acc, (guv2*)(c + 2 * x));
        } else {
            double acc = __builtin_nontemporal_load(c + n - 1);
            for (int l = 0; l < nlayers; ++l) acc += __builtin_nontemporal_load(p + (int64_t)l * n + n - 1);
            __builtin_nontemporal_store(acc, c + n - 1);
        }
    }
}

// The same with one element per thread.  Up to three odd layers that do not
// stay in the caches run faster so, by all loads being nontemporal: 70000001
// elements and 1, 2, 3 or 4 layers 243, 345, 446 and 555 us, in pairs 256, 357,
// 457 and 555; 20000001 elements 72, 101, 130 and 160, in pairs 69, 95, 128 and
// 157.
__global__ __launch_bounds__(kThreads) void layer_reduce_single_kernel(double* __restrict__ C,
                                                                       const double* __restrict__ partial, int64_t n,
                                                                       int nlayers) {
    gdouble* c = (gdouble*)C;
    gcdouble* p = (gcdouble*)partial;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < n; x += stride) {
        double acc = __builtin_nontemporal_load(c + x);
        for (int l = 0; l < nlayers; ++l) acc += __builtin_nontemporal_load(p + (int64_t)l * n + x);
        __builtin_nontemporal_store(acc, c + x);
    }
}
constexpr double kSingleBytes = 600e6;  // of C and the layers; the two cross there (25000001 elements, two layers)

int check_offsets(const char* who, const int64_t* off, int parts, int64_t total) {
    if (!off) return fail(DG_ERR_INVALID, "%s: null offsets", who);
    if (parts < 1 || parts > kMaxParts) return fail(DG_ERR_INVALID, "%s: %d parts (1..%d)", who, parts, kMaxParts);
    if (off[0] != 0 || off[parts] != total)
        return fail(DG_ERR_INVALID, "%s: offsets must run from 0 to %lld", who, (long long)total);
    for (int i = 0; i < parts; ++i)
        if (off[i + 1] < off[i]) return fail(DG_ERR_INVALID, "%s: offsets decrease at %d", who, i);
    return DG_OK;
}

template <bool PACK>
int block2d(const char* who, const double* src, double* dst, int64_t ldg, int64_t rows, int64_t cols,
            const int64_t* row_off, int nrb, const int64_t* col_off, int ncb, void* stream) {
    if (rows < 0 || cols < 0) return fail(DG_ERR_INVALID, "%s: negative size", who);
    if (ldg < (rows > 1 ? rows : 1)) return fail(DG_ERR_INVALID, "%s: ldg %lld < rows %lld", who, (long long)ldg, (long long)rows);
    int rc = check_offsets(who, row_off, nrb, rows);
    if (rc) return rc;
    rc = check_offsets(who, col_off, ncb, cols);
    if (rc) return rc;
    if (rows == 0 || cols == 0) return DG_OK;
    if (!src || !dst) return fail(DG_ERR_INVALID, "%s: null pointer", who);
    rc = require_device();
    if (rc) return rc;
    Bands b;
    b.n = nrb;
    int64_t tallest = 0;
    for (int i = 0; i <= nrb; ++i) b.off[i] = row_off[i];
    for (int i = 0; i < nrb; ++i) tallest = std::max<int64_t>(tallest, row_off[i + 1] - row_off[i]);
    const RunShape rs = run_shape(tallest, 2);
    int64_t chunks = 0;
    for (int i = 0; i < nrb; ++i) {
        b.cpre[i] = (int32_t)chunks;
        chunks += (row_off[i + 1] - row_off[i] + rs.chunk - 1) / rs.chunk;
        if (chunks > INT32_MAX) return fail(DG_ERR_INVALID, "%s: too many row chunks", who);
    }
    b.cpre[nrb] = (int32_t)chunks;
    bool lines = whole_lines(src, dst, 8 * ldg);
    for (int i = 1; i <= nrb; ++i) lines = lines && row_off[i] % 16 == 0;
    const int64_t tallest_chunks = (tallest + rs.chunk - 1) / rs.chunk;
    lines = lines && (PACK || tallest_chunks <= 1 << 25);  // the band's own order has its chunks on x alone
    dim3 grid = run_grid(chunks, col_groups(cols, rs.cols_per_wg));
    if (!PACK && lines) grid = dim3((unsigned)tallest_chunks, grid.y, (unsigned)nrb);
    const auto kernel = lines ? block2d_kernel<PACK, true> : block2d_kernel<PACK, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, as_stream(stream), src, dst, ldg, cols, b, rs.lanes_log2);
    DG_LAUNCH_CHECK();
    return DG_OK;
}

template <bool PACK>
int cyclic(const char* who, const double* src, double* dst, int64_t ldg, int64_t rows, int64_t cols, int64_t mb,
           int64_t nb, int P, int Q, void* stream) {
    if (rows < 0 || cols < 0) return fail(DG_ERR_INVALID, "%s: negative size", who);
    if (mb <= 0 || nb <= 0) return fail(DG_ERR_INVALID, "%s: block size must be positive", who);
    if (P < 1 || Q < 1 || P > kMaxParts || Q > kMaxParts)
        return fail(DG_ERR_INVALID, "%s: process grid %dx%d (1..%d per side)", who, P, Q, kMaxParts);
    if (ldg < (rows > 1 ? rows : 1)) return fail(DG_ERR_INVALID, "%s: ldg %lld < rows %lld", who, (long long)ldg, (long long)rows);
    if (rows == 0 || cols == 0) return DG_OK;
    if (!src || !dst) return fail(DG_ERR_INVALID, "%s: null pointer", who);
    int rc = require_device();
    if (rc) return rc;
    if (rows > INT32_MAX || cols > INT32_MAX || mb > INT32_MAX || nb > INT32_MAX)
        return fail(DG_ERR_UNSUPPORTED, "%s: rows, cols and block sizes must be below 2^31", who);
    Cyclic g{};
    g.ldg = ldg;
    g.rows = (uint32_t)rows; g.cols = (uint32_t)cols; g.mb = (uint32_t)mb; g.nb = (uint32_t)nb;
    g.P = (uint32_t)P; g.Q = (uint32_t)Q;
    g.nr = make_numroc(g.rows, g.mb, g.P);
    g.nc = make_numroc(g.cols, g.nb, g.Q);
    const RunShape rs = run_shape(mb < rows ? mb : rows, 2);
    g.dP = make_fastdiv(g.P); g.dQ = make_fastdiv(g.Q); g.dnb = make_fastdiv(g.nb);
    g.dchunks = make_fastdiv((uint32_t)rs.chunks);
    const int64_t row_blocks = (rows + mb - 1) / mb;
    if (row_blocks > INT32_MAX / rs.chunks) return fail(DG_ERR_INVALID, "%s: too many row chunks", who);
    dim3 grid = run_grid(row_blocks * rs.chunks, col_groups(cols, rs.cols_per_wg));
    bool lines = whole_lines(src, dst, 8 * (ldg | rows | std::min(mb, rows)));
    // packed runs of half a line each want the hint too (12288 x 7168 in 8 x 64:
    // 618 us without, 594 with it; runs of three halves lose 8 % with it)
    if (PACK && mb == 8) lines = whole_lines(src, dst, 8 * (ldg | rows), 64);
    const bool halves = whole_lines(dst, dst, 8 * (ldg | mb), 64);
    const uint32_t per_xcd = !PACK && !halves && mb >= 16 && mb <= 32 && grid.z == 1 ? eighth(grid.x) : 0;
    if (per_xcd) grid.x = 8 * per_xcd;
    const auto kernel = lines ? cyclic_kernel<PACK, true> : cyclic_kernel<PACK, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, as_stream(stream), src, dst, g, rs.lanes_log2, per_xcd);
    DG_LAUNCH_CHECK();
    return DG_OK;
}

}  // namespace

}  // namespace dg

extern "C" {

int dg_block_splits(int64_t n, int parts, int64_t* offsets) {
    using namespace dg;
    if (n < 0 || parts < 1 || !offsets) return fail(DG_ERR_INVALID, "dg_block_splits: n=%lld parts=%d", (long long)n, parts);
    const int64_t base = n / parts;
    for (int i = 0; i < parts; ++i) offsets[i] = (int64_t)i * base;
    offsets[parts] = n;
    return DG_OK;
}

int dg_virtual_grid(int size, int* drow, int* dcol) {
    using namespace dg;
    if (size < 1 || !drow || !dcol) return fail(DG_ERR_INVALID, "dg_virtual_grid: size %d", size);
    int px = 1;
    while ((int64_t)(px + 1) * (px + 1) <= size) ++px;  // floor(sqrt(size)) in integers
    int d = px;
    while (d > 1 && size % d != 0) --d;
    *dcol = d;
    *drow = size / d;
    return DG_OK;
}

int64_t dg_numroc(int64_t n, int64_t nb, int iproc, int isrcproc, int nprocs) {
    if (n <= 0 || nb <= 0 || nprocs <= 0) return 0;
    const int64_t dist = ((int64_t)nprocs + iproc - isrcproc) % nprocs;
    const int64_t nblocks = n / nb;
    int64_t r = (nblocks / nprocs) * nb;
    const int64_t extra = nblocks % nprocs;
    if (dist < extra) r += nb;
    else if (dist == extra) r += n % nb;
    return r;
}

int64_t dg_block_cyclic_size(int64_t rows, int64_t cols, int64_t mb, int64_t nb, int P, int Q) {
    int64_t total = 0;
    for (int pr = 0; pr < P; ++pr)
        for (int pc = 0; pc < Q; ++pc) total += dg_numroc(rows, mb, pr, 0, P) * dg_numroc(cols, nb, pc, 0, Q);
    return total;
}

int dg_pack_block2d(const double* G, int64_t ldg, int64_t rows, int64_t cols, const int64_t* row_off, int nrb,
                    const int64_t* col_off, int ncb, double* packed, void* stream) {
    return dg::block2d<true>("dg_pack_block2d", G, packed, ldg, rows, cols, row_off, nrb, col_off, ncb, stream);
}

int dg_unpack_block2d(const double* packed, const int64_t* row_off, int nrb, const int64_t* col_off, int ncb,
                      double* G, int64_t ldg, int64_t rows, int64_t cols, void* stream) {
    return dg::block2d<false>("dg_unpack_block2d", packed, G, ldg, rows, cols, row_off, nrb, col_off, ncb, stream);
}

int dg_pack_block_cyclic(const double* G, int64_t ldg, int64_t rows, int64_t cols, int64_t mb, int64_t nb, int P,
                         int Q, double* packed, void* stream) {
    return dg::cyclic<true>("dg_pack_block_cyclic", G, packed, ldg, rows, cols, mb, nb, P, Q, stream);
}

int dg_unpack_block_cyclic(const double* packed, int64_t mb, int64_t nb, int P, int Q, double* G, int64_t ldg,
                           int64_t rows, int64_t cols, void* stream) {
    return dg::cyclic<false>("dg_unpack_block_cyclic", packed, G, ldg, rows, cols, mb, nb, P, Q, stream);
}

}  // extern "C"

namespace dg {
namespace {
template <typename T>
int copy_block(const char* name, int64_t rows, int64_t cols, const T* src, int64_t lds, T* dst, int64_t ldd,
               void* stream) {
    if (rows < 0 || cols < 0) return fail(DG_ERR_INVALID, "%s: negative size", name);
    if (lds < rows || ldd < rows) return fail(DG_ERR_INVALID, "%s: leading dimension < rows", name);
    if (rows == 0 || cols == 0) return DG_OK;
    if (!src || !dst) return fail(DG_ERR_INVALID, "%s: null pointer", name);
    int rc = require_device();
    if (rc) return rc;
    const RunShape rs = run_shape(rows, 16 / (int)sizeof(T));
    if (rs.chunks > INT32_MAX) return fail(DG_ERR_INVALID, "%s: too many rows", name);
    const bool lines = whole_lines(src, dst, (lds | ldd | rows) * (int64_t)sizeof(T));
    const auto kernel = lines ? copy_block_kernel<true, T> : copy_block_kernel<false, T>;
    hipLaunchKernelGGL(kernel, run_grid(rs.chunks, col_groups(cols, rs.cols_per_wg)), dim3(kThreads), 0,
                       as_stream(stream), rows, cols, src, lds, dst, ldd, rs.lanes_log2);
    DG_LAUNCH_CHECK();
    return DG_OK;
}
}  // namespace
}  // namespace dg

extern "C" {

int dg_copy_block(int64_t rows, int64_t cols, const double* src, int64_t lds, double* dst, int64_t ldd,
                  void* stream) {
    return dg::copy_block("dg_copy_block", rows, cols, src, lds, dst, ldd, stream);
}

int dg_copy_block_f32(int64_t rows, int64_t cols, const float* src, int64_t lds, float* dst, int64_t ldd,
                      void* stream) {
    return dg::copy_block("dg_copy_block_f32", rows, cols, src, lds, dst, ldd, stream);
}

int dg_layer_reduce(double* C, const double* partial, int64_t n, int nlayers, void* stream) {
    using namespace dg;
    if (n < 0 || nlayers < 0) return fail(DG_ERR_INVALID, "dg_layer_reduce: negative size");
    if (n == 0 || nlayers == 0) return DG_OK;
    if (!C || !partial) return fail(DG_ERR_INVALID, "dg_layer_reduce: null pointer");
    if ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(partial)) & 15)
        return fail(DG_ERR_INVALID, "dg_layer_reduce: buffers must be 16-byte aligned");
    int rc = require_device();
    if (rc) return rc;
    const bool single = (n & 1) && nlayers <= 3 && 8.0 * (double)n * (nlayers + 1) > kSingleBytes;
    const auto kernel = single ? layer_reduce_single_kernel : (n & 1) ? layer_reduce_kernel<true> : layer_reduce_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(looped_blocks(single ? n : (n + 1) / 2, kThreads)), dim3(kThreads), 0,
                       as_stream(stream), C, partial, n, nlayers);
    DG_LAUNCH_CHECK();
    return DG_OK;
}

}  // extern "C"
