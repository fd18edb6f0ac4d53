// sz3d_lane_check.cpp -- host checks of the lane kernels' work split (3-D,
// block side 4) through the functions of zccl_sz3d.h that the kernels use.
//
//   routes   volumes with too few rows or columns to fill the chip are left to
//            the tiled decoder, larger ones take the lane decoder
//   rows     the lane compress takes rows of any length in 32-bit offsets
//
// Built and run by tests/test_sz3d_lane.py with g++; prints "ok <cases>" or the
// first violation.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "zccl_sz3d.h"

using namespace zk;

static long g_cases = 0;

#define REQUIRE(cond, ...)                                                                         \
    do {                                                                                           \
        if (!(cond)) {                                                                             \
            std::printf("FAIL %s:%d: %s | ", __FILE__, __LINE__, #cond);                           \
            std::printf(__VA_ARGS__);                                                              \
            std::printf("\n");                                                                     \
            std::exit(1);                                                                          \
        }                                                                                          \
    } while (0)

// Volumes timed by both decoders (lanes: the faster one), and those that the
// lane decoder's GPU tests take.
static void routes()
{
    struct {
        uint32_t d1, d2, d3;
        int T;
        bool lanes;
    } v[] = {{118, 27, 194, 4, false}, {77, 38, 138, 1, false}, {172, 27, 321, 8, false}, {290, 61, 367, 16, false},
        {86, 165, 127, 1, false}, {167, 342, 264, 1, false}, {64, 336, 320, 2, false}, {160, 464, 320, 2, false},
        {256, 256, 256, 16, true}, {300, 300, 300, 16, true}, {384, 384, 384, 8, true}, {448, 320, 176, 1, true},
        {512, 512, 512, 16, true}, {512, 512, 512, 1, true}, {510, 510, 510, 16, true},
        {256, 192, 256, 16, true}, {250, 190, 250, 16, true}, {200, 350, 250, 9, true}, {260, 192, 260, 4, true},
        {131, 195, 515, 2, true}, {67, 257, 1021, 1, true}, {66, 256, 1024, 1, true}};
    for (const auto& x : v) {
        Geom3 g;
        std::vector<Part3> parts(x.T);
        REQUIRE(make_geom3(x.d1, x.d2, x.d3, 4, x.T, &g, parts.data()), "geometry");
        REQUIRE((g.nruns > 0) == x.lanes, "%ux%ux%u T %d: runs %u", x.d1, x.d2, x.d3, x.T, g.nruns);
        g_cases++;
    }
}

// Every volume of block side 4 takes the lane compress, also those with rows of
// 2^27 values and more (the generic kernels' launch of a wave per block is too
// large for some of them); row offsets and block numbers fit 32 signed bits.
static void long_rows()
{
    const uint32_t v[][4] = {{1, 1, (1u << 27) - 1, 1}, {1, 1, 1u << 27, 1}, {2, 2, 1u << 27, 4}, {1, 3, (1u << 27) + 1001, 1},
        {1, 4, (1u << 29) - 1, 1}, {1, 2, (1u << 30) - 1, 1}, {1, 1, 0x7FFFFFFFu, 1}, {3, 1, 715827882u, 3}};
    for (const auto& x : v) {
        Geom3 g;
        std::vector<Part3> parts(x[3]);
        REQUIRE(make_geom3(x[0], x[1], x[2], 4, (int) x[3], &g, parts.data()), "geometry");
        REQUIRE(g.nlane > 0 && g.nlane <= g.nblocks, "%ux%ux%u: %u tiles", x[0], x[1], x[2], g.nlane);
        REQUIRE((uint64_t) g.nlane * g.wlane * 64 < (1ull << 32), "threads of the launch");
        const uint64_t rows = g.d2 < 4 ? g.d2 : 4;  // rows -1 .. 3 of a block, those there are
        REQUIRE((rows - 1) * g.d3 < (1ull << 31) && g.d3 < (1ull << 31), "row offsets");
        for (const Part3& p : parts)
            REQUIRE((uint64_t) p.b1 * p.b2 * p.b3 + 64 * g.wlane < (1ull << 31), "block numbers");
        g_cases++;
    }
}

int main()
{
    routes();
    long_rows();
    std::printf("ok %ld\n", g_cases);
    return 0;
}
