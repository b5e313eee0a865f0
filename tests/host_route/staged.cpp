// CPU-only checks of the addresses in csrc/staged.hpp (Staged), compiled for
// the host by tests/test_host_route.py.  No GPU call is made.
#include <cstdio>
#include <vector>

#include "staged.hpp"

static int failures = 0;
#define CHECK(c)                                                                                \
    do {                                                                                        \
        if (!(c)) { std::fprintf(stderr, "FAILED: %s (line %d)\n", #c, __LINE__); ++failures; } \
    } while (0)

template <typename T, bool KC, int ROWS, int BK>
void check() {
    using O = dg::Staged<T, KC, ROWS, BK>;
    constexpr int E = O::E, S = O::S;
    // the longest leading dimension and the next: offsets in 32 bits are the true ones
    const int64_t big = O::kMaxLd;
    CHECK(O::takes(nullptr, big) && !O::takes(nullptr, big + 1));
    CHECK(O::takes(nullptr, E - 1) && O::takes(nullptr, 1) == (KC || E <= 2));
    CHECK(!O::takes(reinterpret_cast<const T*>(S / 2), 64));
    int64_t most = 0;
    for (int t = 0; t < 256; ++t)
        for (int q = 0; q < O::NL; ++q) {
            const int64_t r = O::row(t, q), k = O::kk(t, q);
            CHECK(r >= 0 && r < ROWS && k >= 0 && k < BK);
            CHECK((int64_t)O::offset(t, q, big, ROWS) == S * (KC ? r * big + k : k * big + r));
            most = std::max(most, S * (KC ? r * (big + 1) + k : k * (big + 1) + r));
        }
    CHECK(most >= (int64_t)1 << 32);  // the bound gives nothing away
    // ragged operands: every element loaded lies between the operand's first
    // and last, each of a stage arrives once, with zeros past the last k
    for (int rows : {1, 2, 3, 31, 32, 33, 65, 127, 128, 129, 200})
        for (int klen : {1, 2, 3, 15, 16, 17, 31, 32, 33, 50, 64, 65, 130})
            for (int64_t ld : {KC ? klen : rows, (KC ? klen : rows) + 1}) {
                const bool runs = O::takes(nullptr, ld);
                const int64_t end = KC ? (rows - 1) * ld + klen : rows + (klen - 1) * ld;
                for (int64_t row0 = 0; row0 < rows; row0 += ROWS) {
                    const int inside = (int)std::min<int64_t>(ROWS, rows - row0);
                    const int last = KC || inside == ROWS ? 0 : 1;
                    for (int k0 = 0; k0 < klen; k0 += BK) {
                        const int64_t base = row0 * (KC ? ld : 1) + k0 * (KC ? 1 : ld);
                        const int left = klen - k0;
                        std::vector<int64_t> got(ROWS * BK, -2);
                        for (int t = 0; t < 256; ++t)
                            for (int q = 0; q < O::NL; ++q)
                                for (int e = 0; e < E; ++e) {
                                    const int r = O::row(t, q) + (KC ? 0 : e), k = O::kk(t, q) + (KC ? e : 0);
                                    const bool whole = runs && left >= BK + last;
                                    const int64_t at = base + (whole ? O::offset(t, q, ld, inside) / S + e
                                                                     : O::last_offset(t, q, e, ld, inside, std::min(left, BK)));
                                    CHECK(at >= 0 && at < end);
                                    CHECK(got[r * BK + k] == -2);
                                    got[r * BK + k] = whole || k < left ? at : -1;
                                }
                        for (int r = 0; r < inside; ++r)
                            for (int k = 0; k < BK; ++k) {
                                const int64_t want = k0 + k < klen ? (KC ? (row0 + r) * ld + k0 + k : row0 + r + (k0 + k) * ld) : -1;
                                CHECK(got[r * BK + k] == want);
                            }
                    }
                }
            }
}

int main() {
    check<double, true, 128, 16>();
    check<double, false, 128, 16>();
    check<double, true, 64, 16>();
    check<double, false, 64, 16>();
    check<double, true, 32, 32>();
    check<double, false, 32, 32>();
    check<float, true, 64, 32>();
    check<float, false, 64, 32>();
    check<float, true, 32, 64>();
    check<float, false, 32, 64>();
    if (!failures) std::printf("staged: ok\n");
    return failures ? 1 : 0;
}
