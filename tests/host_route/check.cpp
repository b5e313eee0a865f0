// CPU-only checks of the FP64 GEMM's routing (prepare_gemm of libdgamd.so),
// built and run by tests/test_host_route.py.  No GPU call is made and no
// operand is read: the matrices are addresses only.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <random>
#include <string>

static inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)((uint64_t)a * b >> 32); }  // no device pass here
#include "dg_internal.hpp"

static size_t allocated = 0;  // bytes asked of operator new so far, the library's included
void* operator new(size_t n) {
    allocated += n;
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

using dg::Prob;
using dg::Seg;

static int failures = 0;
#define CHECK(c)                                                                                        \
    do {                                                                                                \
        if (!(c)) { std::fprintf(stderr, "FAILED: %s (line %d)\n", #c, __LINE__); ++failures; }         \
    } while (0)

static double* at(uintptr_t x) { return reinterpret_cast<double*>(x); }

// The host cost of a batch of many segments: its tables are copied once.
static void check_bytes() {
    std::vector<Prob> probs;
    std::vector<Seg> segs;
    for (int i = 0; i < 1024; ++i) {
        Prob p{};
        p.m = p.n = 64;
        p.c = at(0x100000000 + 32768 * (uintptr_t)i);
        p.ldc = 64;
        p.alpha = 1.0;
        p.seg0 = (int32_t)segs.size();
        p.nseg = 64;
        for (int s = 0; s < 64; ++s) segs.push_back(Seg{at(0x200000000), at(0x300000000), 2048, 2048, 64});
        probs.push_back(p);
    }
    for (char oa : {'N', 'T'}) {
        dg::GemmBatch b;
        const size_t before = allocated;
        CHECK(dg::prepare_gemm(oa, 'T', probs, segs, b) == DG_OK);
        const size_t spent = allocated - before, tables = segs.size() * sizeof(Seg) + probs.size() * sizeof(Prob);
        std::printf("prepared %zu bytes of tables with %zu bytes\n", tables, spent);
        CHECK(spent <= tables + tables / 2);
    }
    // many problems of one segment: their lists are made in their final size
    segs.assign(1000, Seg{at(0x200000000), at(0x300000000), 33, 17, 17});
    probs.resize(1000);
    for (int i = 0; i < 1000; ++i) {
        probs[i].m = probs[i].ldc = 33;
        probs[i].n = 65;
        probs[i].seg0 = i;
        probs[i].nseg = 1;
    }
    dg::GemmBatch b;
    const size_t before = allocated;
    CHECK(dg::prepare_gemm('N', 'N', probs, segs, b) == DG_OK);
    const size_t spent = allocated - before, tables = segs.size() * sizeof(Seg) + probs.size() * sizeof(Prob);
    std::printf("prepared %zu bytes of tables with %zu bytes\n", tables, spent);
    CHECK(spent <= 2 * tables);
}

// Every choice covers each element of each problem once, each part at the
// operands' right places, with tile numbers that follow one another.
static void check_parts() {
    std::mt19937_64 rng(7);
    auto pick = [&](int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); };
    const int64_t edges[5] = {128, 128, 128, 64, 32};
    for (int trial = 0; trial < 60; ++trial) {
        const char oa = "NT"[trial & 1], ob = "NT"[(trial >> 1) & 1];
        const bool ak = oa == 'T', bkc = ob == 'N', even = trial % 3 != 0;
        std::vector<Prob> probs;
        std::vector<Seg> segs;
        const int count = (int)pick(1, 3);
        for (int i = 0; i < count; ++i) {
            Prob p{};
            p.m = pick(1, trial % 5 ? 3000 : 300);
            p.n = pick(1, trial % 5 ? 3000 : 300);
            if (trial % 7 == 0) { p.m = (p.m + 127) / 128 * 128; p.n = (p.n + 127) / 128 * 128; }
            p.ldc = p.m + pick(0, 5);
            p.c = at(0x1000000000 * (uintptr_t)(i + 1));
            p.alpha = 1.0;
            p.seg0 = (int32_t)segs.size();
            p.nseg = (int32_t)pick(1, 4);
            const uintptr_t sa = even ? 8 * pick(0, 1) : 0, sb = even ? 8 * pick(0, 1) : 0;
            for (int s = 0; s < p.nseg; ++s) {
                const int64_t k = even ? 16 * pick(1, 20) : pick(1, 300);
                Seg g{at(0x20000000000 + sa * !ak), at(0x30000000000 + sb * !bkc), (ak ? k : p.m) + pick(0, 9), (bkc ? k : p.n) + pick(0, 9), k};
                if (even) { g.lda += g.lda & 1; g.ldb += g.ldb & 1; }
                segs.push_back(g);
            }
            probs.push_back(p);
        }
        for (int tile = dg::DG_GEMM_TILE_AUTO; tile < dg::DG_GEMM_TILES; ++tile)
            for (bool split : {true, false}) {
                dg::GemmBatch b;
                CHECK(dg::prepare_gemm(oa, ob, probs, segs, b, split, tile) == DG_OK);
                CHECK(b.segs.size() >= segs.size() && !memcmp(b.segs.data(), segs.data(), segs.size() * sizeof(Seg)));
                const std::vector<Prob>* lists[5] = {&b.dma, &b.dmae, &b.gen[0], &b.gen[1], &b.gen[2]};
                const int tiles[5] = {b.tiles_dma, b.tiles_dmae, b.tiles_gen[0], b.tiles_gen[1], b.tiles_gen[2]};
                std::vector<std::vector<unsigned char>> seen(count);
                for (int i = 0; i < count; ++i) seen[i].assign((size_t)(probs[i].m * probs[i].n), 0);
                for (int l = 0; l < 5; ++l) {
                    int64_t next = 0;
                    for (const Prob& q : *lists[l]) {
                        const int i = (int)(reinterpret_cast<uintptr_t>(q.c) / 0x1000000000) - 1;
                        CHECK(i >= 0 && i < count);
                        const Prob& p = probs[i];
                        const int64_t off = q.c - p.c, r0 = off % p.ldc, c0 = off / p.ldc;
                        CHECK(q.ldc == p.ldc && q.nseg == p.nseg && r0 + q.m <= p.m && c0 + q.n <= p.n);
                        CHECK(q.tile0 == next);
                        int sa = 0, sb = 0;
                        for (int s = 0; s < q.nseg; ++s) {
                            const Seg &g = b.segs[q.seg0 + s], &h = segs[p.seg0 + s];
                            CHECK(g.lda == h.lda && g.ldb == h.ldb && g.klen == h.klen);
                            CHECK(g.a == h.a + (ak ? r0 * h.lda : r0) && g.b == h.b + (bkc ? c0 * h.ldb : c0));
                            sa = !ak && (reinterpret_cast<uintptr_t>(g.a) & 15);
                            sb = !bkc && (reinterpret_cast<uintptr_t>(g.b) & 15);
                            if (l < 2) CHECK(!(g.lda & 1) && !(g.ldb & 1) && (!ak || !(reinterpret_cast<uintptr_t>(g.a) & 15)));
                            if (l == 0) CHECK(g.klen % 8 == 0 && !sa && !sb);
                        }
                        if (l == 0) CHECK(q.m % 128 == 0 && q.n % 128 == 0);
                        if (l < 2) CHECK(q.shift == (sa | sb << 1)); else { CHECK(q.shift == 0); sa = sb = 0; }
                        next += ((q.m + sa + edges[l] - 1) / edges[l]) * ((q.n + sb + edges[l] - 1) / edges[l]);
                        for (int64_t c = c0; c < c0 + q.n; ++c)
                            for (int64_t r = r0; r < r0 + q.m; ++r) ++seen[i][(size_t)(r + c * p.m)];
                    }
                    CHECK(tiles[l] == next);
                }
                for (int i = 0; i < count; ++i) {
                    bool once = true;
                    for (unsigned char x : seen[i]) once = once && x == 1;
                    CHECK(once);
                }
                if (failures) {
                    std::fprintf(stderr, "trial %d, choice %d, split %d\n", trial, tile, (int)split);
                    return;
                }
            }
    }
}

// Leading dimensions of millions: the direct-to-LDS kernels keep the problems
// that they take, and the register-staged ones load by elements only where a
// lane's offset would leave 32 bits.
static void check_long() {
    struct { char oa, ob; int64_t m, n, k, lda, ldb; int direct, elements; } cases[] = {
        {'T', 'N', 2048, 2048, 5000000, 5000000, 5000000, -1, 0},
        {'T', 'N', 4096, 4096, 5000000, 5000000, 5000000, -1, 0},
        {'N', 'N', 4096, 4096, 4096, 8000000, 4096, -1, 0},
        {'N', 'N', 4096, 4096, 4096, 8000001, 4096, 0, 0},
        {'T', 'N', 2048, 2048, 4096, 4227000, 4096, -1, 0},
        {'T', 'N', 2048, 2048, 4096, 8000001, 4096, 0, 0},   // 128x128 tiles past their limit, 64x64 within it
        {'T', 'N', 2048, 2048, 4096, 18000000, 4096, 1, 0},  // past every tile's
        {'T', 'T', 4096, 4096, 4096, 18000000, 4096, 1, 0},
        {'T', 'N', 2048, 2048, 4096, 18000001, 4096, 0, 1},
        {'N', 'T', 2048, 2048, 512, 35000000, 2048, -1, 0},
        {'N', 'T', 2048, 2048, 512, 36000000, 2048, 1, 0},
        {'N', 'T', 2048, 2048, 512, 36000001, 2048, 0, 1},
    };
    const int64_t edges[3] = {128, 64, 32}, depths[3] = {16, 16, 32};
    for (const auto& c : cases) {
        const bool ak = c.oa == 'T', bkc = c.ob == 'N';
        std::vector<Seg> segs{Seg{at(0x10000), at(0x20000), c.lda, c.ldb, c.k}};
        Prob p{};
        p.m = c.m; p.n = c.n; p.ldc = c.m; p.c = at(0x30000); p.alpha = 1.0; p.nseg = 1;
        dg::GemmBatch b;
        CHECK(dg::prepare_gemm(c.oa, c.ob, {p}, segs, b) == DG_OK);
        const bool direct = !b.dma.empty() || !b.dmae.empty();
        bool any = false;
        for (int w = 0; w < 3; ++w)
            for (const Prob& q : b.gen[w]) {
                const bool elements = q.shift & dg::kByElements;
                auto most = [&](bool kc, int64_t ld) { return 8 * (kc ? (edges[w] - 1) * ld : (depths[w] - 1) * ld + edges[w]); };
                const bool leaves = std::max(most(ak, c.lda), most(bkc, c.ldb)) >= (int64_t)1 << 32;
                CHECK(elements == leaves);
                any = any || elements;
            }
        CHECK(any == (c.elements != 0));
        CHECK(c.direct < 0 || direct == (c.direct != 0));
        if (failures) {
            std::fprintf(stderr, "%c%c %lld %lld %lld lda %lld\n", c.oa, c.ob, (long long)c.m, (long long)c.n, (long long)c.k, (long long)c.lda);
            return;
        }
    }
}

// Short segments: the direct-to-LDS kernels, which run through them, keep the
// products whose register-staged tiles would start anew every few stages.
static void check_short() {
    struct { int64_t M; int nb, direct; } cases[] = {{2048, 16, 1}, {2048, 32, 1}, {2048, 64, 1}, {2048, 512, 0},
                                                     {4096, 16, 1}, {4096, 64, 1}, {4096, 512, 0}, {1024, 64, 0}};
    for (const auto& c : cases) {  // SUMMA of M^3 on 2 x 2 in panels of nb
        std::vector<Prob> probs;
        std::vector<Seg> segs;
        for (int r = 0; r < 4; ++r) {
            Prob p{};
            p.m = p.n = p.ldc = c.M / 2;
            p.c = at(0x100000000); p.alpha = 1.0;
            p.seg0 = (int32_t)segs.size();
            p.nseg = (int32_t)(c.M / c.nb);
            for (int s = 0; s < p.nseg; ++s) segs.push_back(Seg{at(0x200000000), at(0x300000000), c.M / 2, c.M / 2, c.nb});
            probs.push_back(p);
        }
        dg::GemmBatch b;
        CHECK(dg::prepare_gemm('N', 'N', probs, segs, b) == DG_OK);
        CHECK(b.dma.empty() == !c.direct);
        // half-empty stages of the 32x32 tiles are no bargain
        if (c.nb == 16) CHECK(b.gen[2].empty());
        if (failures) { std::fprintf(stderr, "%lld in panels of %d\n", (long long)c.M, c.nb); return; }
    }
}

// An autotuned plan's first use: choices that come out alike are timed once,
// and slow variants once.
static void check_trials() {
    auto distinct = [](char oa, char ob, int64_t m, int64_t n, int64_t k) {
        std::vector<Seg> segs{Seg{at(0x10000), at(0x20000), oa == 'T' ? k : m, ob == 'N' ? k : n, k}};
        Prob p{};
        p.m = m; p.n = n; p.ldc = m; p.c = at(0x30000); p.alpha = 1.0; p.nseg = 1;
        std::vector<dg::GemmBatch> b(dg::DG_GEMM_TILES);
        std::vector<int> out;
        for (int t = 0; t < dg::DG_GEMM_TILES; ++t) {
            CHECK(dg::prepare_gemm(oa, ob, {p}, segs, b[t], true, t) == DG_OK);
            bool seen = false;
            for (int u : out) seen = seen || dg::same_lists(b[t], b[u]);
            if (!seen) out.push_back(t);
        }
        return out;
    };
    CHECK((distinct('N', 'N', 2048, 2048, 2048) == std::vector<int>{0, 1, 3, 4}));     // nothing to cut
    CHECK((distinct('N', 'N', 2047, 2049, 2049) == std::vector<int>{0, 2, 3, 4}));     // odd: not direct
    CHECK((distinct('T', 'N', 5000, 5000, 5000) == std::vector<int>{0, 1, 2, 3, 4}));
    CHECK((distinct('T', 'T', 90, 2000, 333) == std::vector<int>{0, 4}));              // narrow: 64x64 at most
    // the fastest, found with one run of what is half as slow again as the best before it and three of the others
    const std::vector<int> choices{0, 1, 3, 4};
    const float ms[4][3] = {{6.0f, 6.1f, 9.2f}, {5.5f, 5.4f, 5.6f}, {0, 0, 0}, {8.2f, 6.6f, 8.5f}};
    int runs = 0, choice = -1, mode = -1;
    auto trial = [&](int c, int v, float* t) {
        ++runs;
        const int row = c == 0 ? 0 : c == 1 ? 1 : 3;
        *t = c == 3 ? 5.45f : ms[row][v == dg::DG_GEMM_MODE_XCD ? 0 : v == dg::DG_GEMM_MODE_ROUND_ROBIN ? 1 : 2];
        return DG_OK;
    };
    CHECK(dg::fastest_variant(choices, trial, &choice, &mode) == DG_OK);
    CHECK(choice == 1 && mode == dg::DG_GEMM_MODE_ROUND_ROBIN);
    CHECK(runs == 3 + 3 + 1 + 9 + 9 + 1 + 3 + 1);
    // runs so short that a launch's gap decides keep all three
    runs = 0;
    CHECK(dg::fastest_variant(choices, [&](int c, int v, float* t) { trial(c, v, t); *t *= 0.01f; return DG_OK; }, &choice, &mode) == DG_OK);
    CHECK(choice == 1 && runs == 36);
    // a first run that is cold (code, tables, clocks) does not lose: measured first and steady
    // times of the 7 x 5 batch of 5000 with 256 products, choices 0 to 4, modes 0 to 2
    const float cold[5][3] = {{6.673f, 14.713f, 5.887f}, {6.676f, 17.454f, 6.094f}, {6.917f, 18.615f, 6.198f},
                              {7.060f, 18.292f, 6.539f}, {9.676f, 20.202f, 10.147f}};
    const float warm[5][3] = {{5.767f, 11.612f, 5.718f}, {5.574f, 17.592f, 5.584f}, {5.547f, 18.527f, 5.511f},
                              {5.948f, 17.663f, 6.163f}, {9.517f, 18.957f, 10.201f}};
    int run[5][3] = {};
    CHECK(dg::fastest_variant({0, 1, 2, 3, 4}, [&](int c, int v, float* t) { *t = run[c][v]++ ? warm[c][v] : cold[c][v]; return DG_OK; },
                              &choice, &mode) == DG_OK);
    CHECK(choice == 2 && mode == dg::DG_GEMM_MODE_PERSISTENT);
    // nor does one that is timed while the clock is low: a batch of 3265 in 35 tiles with 5 products, whose runs
    // from 23 to 32 ms after the first took an eighth longer
    const float steady[5][3] = {{1.653f, 1.656f, 1.657f}, {1.537f, 1.535f, 1.540f}, {1.460f, 1.460f, 1.472f},
                                {1.302f, 1.306f, 1.347f}, {1.974f, 1.394f, 1.825f}};
    float now = 0;
    CHECK(dg::fastest_variant({0, 1, 2, 3, 4}, [&](int c, int v, float* t) {
        *t = steady[c][v] * (now > 23 && now < 32 ? 1.12f : 1.0f);
        now += *t;
        return DG_OK;
    }, &choice, &mode) == DG_OK);
    CHECK(choice == 3 && mode != dg::DG_GEMM_MODE_PERSISTENT);
    // a failing trial ends it
    CHECK(dg::fastest_variant(choices, [&](int, int, float*) { return DG_ERR_HIP; }, &choice, &mode) == DG_ERR_HIP);
}

// Launch dimensions stay below 2^32 threads and cover the work, or leave the
// rest to the kernel's loop.
static void check_grids() {
    for (int64_t items : {(int64_t)0, (int64_t)1, (int64_t)64, (int64_t)65, ((int64_t)1 << 32) - 1, (int64_t)1 << 32, ((int64_t)1 << 32) + 1, (int64_t)1 << 40})
        for (int threads : {64, 256}) {
            const int64_t blocks = dg::looped_blocks(items, threads);
            CHECK(blocks >= 1 && blocks * threads < (int64_t)1 << 32);
            CHECK(blocks * threads >= items || (blocks + 1) * threads >= (int64_t)1 << 32);
        }
    for (int64_t chunks : {(int64_t)1, (int64_t)1000, (int64_t)1 << 25, ((int64_t)1 << 25) + 1, (int64_t)1 << 26, ((int64_t)1 << 26) + 12345, ((int64_t)1 << 31) - 1}) {
        const dim3 g = dg::run_grid(chunks, 7);
        CHECK((int64_t)g.x * 64 < (int64_t)1 << 32 && g.y == 7 && g.z < 65536);
        CHECK((int64_t)g.x * g.z >= chunks && (int64_t)g.x * (g.z - 1) < chunks);
    }
    // eight ranges: every chunk once, neighbours on one XCD (workgroup number modulo 8) but at the seams
    for (uint32_t chunks : {1u, 2u, 7u, 8u, 9u, 15u, 64u, 313u, 768u, 100001u}) {
        const uint32_t per = dg::eighth(chunks);
        CHECK(8 * per >= chunks && 8 * per < chunks + 8);
        std::vector<int> xcd(8 * per, -1);
        for (uint32_t x = 0; x < 8 * per; ++x) {
            const uint32_t c = dg::eighth_chunk(x, per);
            CHECK(c < 8 * per && xcd[c] < 0);
            xcd[c] = x % 8;
        }
        int seams = 0;
        for (uint32_t c = 1; c < 8 * per; ++c) seams += xcd[c] != xcd[c - 1];
        CHECK(seams == 7);
    }
}

// Where FP32 products of short K take their own kernel: below one whole
// 32-deep stage, and with few rows in tiles that are not whole below two.
static void check_sgemm_short() {
    for (int64_t m : {1, 37, 64, 103, 128, 4096, 100000})
        for (int64_t k : {1, 4, 8, 16, 31}) CHECK(dg::sgemm_is_short(m, k));
    for (int64_t k : {32, 33, 48, 63}) {
        CHECK(dg::sgemm_is_short(37, k) && dg::sgemm_is_short(103, k));
        CHECK(!dg::sgemm_is_short(64, k) && !dg::sgemm_is_short(128, k) && !dg::sgemm_is_short(130, k) && !dg::sgemm_is_short(2000, k));
    }
    for (int64_t m : {1, 37, 64, 4096})
        for (int64_t k : {64, 65, 1024}) CHECK(!dg::sgemm_is_short(m, k));
}

// The lists of one FP64 problem under DG_GEMM_TILE: sizes of the five.
static void print_lists(char** v) {
    const char oa = v[0][0], ob = v[1][0];
    int64_t x[7];
    for (int i = 0; i < 7; ++i) x[i] = std::atoll(v[2 + i]);  // m n k lda ldb, elements off a 16-byte boundary of A and B
    std::vector<Seg> segs{Seg{at(0x10000) + x[5], at(0x20000) + x[6], x[3], x[4], x[2]}};
    Prob p{};
    p.m = x[0]; p.n = x[1]; p.ldc = x[0]; p.c = at(0x30000); p.alpha = 1.0; p.nseg = 1;
    dg::GemmBatch b;
    CHECK(dg::prepare_gemm(oa, ob, {p}, segs, b) == DG_OK);
    std::printf("%zu %zu %zu %zu %zu\n", b.dma.size(), b.dmae.size(), b.gen[0].size(), b.gen[1].size(), b.gen[2].size());
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "bytes") check_bytes();
    else if (what == "parts") check_parts();
    else if (what == "long") check_long();
    else if (what == "short") check_short();
    else if (what == "sgemm_short") check_sgemm_short();
    else if (what == "trials") check_trials();
    else if (what == "grids") check_grids();
    else if (what == "forced") std::printf("%d\n", dg::forced_tile());
    else if (what == "lists" && argc == 11) print_lists(argv + 2);
    else { std::fprintf(stderr, "unknown check '%s'\n", what.c_str()); return 2; }
    if (!failures) std::printf("%s: ok\n", what.c_str());
    return failures ? 1 : 0;
}
