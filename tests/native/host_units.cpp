// Checks of the engine's host arithmetic that no call on a CPU reaches (built by
// tests/native/Makefile with AddressSanitizer and UndefinedBehaviorSanitizer, the host side
// only): exact reciprocals, launch sizes at the largest counts that the interface takes, where
// a call counts its candidates.  Exit status 0 = all checks passed.
#include <cstdio>

#include "lj_candidates.h"
#include "lj_rows.h"
#include "lj_stencil27.h"

static int failures = 0;
#define CHECK(c)                                                           \
    do {                                                                   \
        if (!(c)) {                                                        \
            std::fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
            ++failures;                                                    \
        }                                                                  \
    } while (0)

// Every workgroup has a place, no dimension holds 2^32 threads, and less than one row's
// number of places is left over.
static void check_launch(uint64_t blocks, uint64_t threads) {
    const dim3 g = lj::grid_of_blocks(blocks);
    const uint64_t places = (uint64_t)g.x * g.y;
    CHECK(g.z == 1 && places >= blocks && places < 0xffffffffull);
    CHECK(g.x * threads < (1ull << 32) && g.y < 65536);
    CHECK(places - blocks < g.y || blocks == 0);
}

// The quotients of cell indices by reciprocal multiplication, at every place where the
// quotient changes near the ends of its range and at its powers of two.
static void check_division(uint32_t v) {
    lj::GridGeom g{};
    g.g[0] = g.g[1] = (int32_t)v;
    lj::set_divisors(&g);
    const uint32_t most = 0x7fffffffu, top = most / v;
    bool ok = true;
    auto at = [&](uint64_t q) {
        for (uint64_t n = q * v > 0 ? q * v - 1 : 0; n <= q * v + 1 && n <= most; ++n)
            ok = ok && lj::div_axis(g, 0, (uint32_t)n) == n / v && lj::div_axis(g, 1, (uint32_t)n) == n / v;
    };
    for (uint64_t q = 0; q <= 16 && q <= top; ++q) at(q), at(top - q);
    for (uint64_t q = 1; q <= top; q <<= 1) at(q), at(q - 1), at(q + 1 <= top ? q + 1 : top);
    ok = ok && lj::div_axis(g, 0, most) == most / v;
    CHECK(ok);
}

int main() {
    // axes of a grid: up to 2^24 cells
    for (uint32_t v = 1; v <= 30000; ++v) check_division(v);
    for (uint32_t v = 30001; v < (1u << 24); v += 997) check_division(v);
    for (uint32_t b = 2; b <= 24; ++b)
        for (uint32_t v = (1u << b) - 2; v <= (1u << b) + 2 && v <= (1u << 24); ++v) check_division(v);
    const uint64_t most = 0x7fffffffull;  // particles of a call
    for (uint64_t n : {(uint64_t)0, (uint64_t)1, (uint64_t)1 << 20, ((uint64_t)1 << 28) - 1, (uint64_t)1 << 28,
                       (uint64_t)1 << 30, most - 1, most}) {
        // row sort, 4 lanes a row and a thread a row
        check_launch((n + lj::kBlockRows - 1) / lj::kBlockRows, lj::kSortThreads);
        check_launch((n + lj::kSortThreads - 1) / lj::kSortThreads, lj::kSortThreads);
        // neighbour lists, 16 slots a wave of 64
        check_launch((n + 63) / 64, 256);
        // batched forces, two lanes a particle, with as many further waves as there can be
        for (uint64_t block : {64, 128, 256}) {
            const uint64_t extra = n;  // one for every system of a particle
            check_launch((n * lj::kPairLanes + block - 1) / block + (extra * lj::kWaveSize + block - 1) / block, block);
        }
    }
    // one workgroup is not left with the cells of a large system, however few there are
    CHECK(lj::count_in_reduction(96 * 650, 650));
    CHECK(!lj::count_in_reduction(195112, 195112));
    CHECK(!lj::count_in_reduction(1000375, 1000000));
    CHECK(!lj::count_in_reduction(4096ull * 3125, 8000));
    // nor a large grid with the few waves of a small system's force launch
    CHECK(lj::count_beside_forces(1000, 4096) && lj::count_beside_forces(500000, 640u * 640 * 640));
    CHECK(!lj::count_beside_forces(1000, 640u * 640 * 640) && !lj::count_beside_forces(100000, 400u * 400 * 400));
    for (uint64_t blocks = 1; blocks < (1u << 27); blocks += 1 + blocks / 3) check_launch(blocks, 256);
    if (failures) {
        std::fprintf(stderr, "%d checks failed\n", failures);
        return 1;
    }
    std::printf("all checks passed\n");
    return 0;
}
