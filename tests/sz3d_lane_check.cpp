// sz3d_lane_check.cpp -- host checks of the lane kernels' work split (3-D,
// block side 4) through the functions of zccl_sz3d.h that the kernels use.
//
//   routes   volumes with too few rows or columns to fill the chip are left to
//            the tiled decoder, larger ones take the lane decoder
//   rows     the lane compress takes rows of any length in 32-bit offsets
//   split    the table a lane per sub-volume fills; the lane compress's tiles,
//            the decoder's runs, rows of blocks, kept planes and y columns: all
//            blocks and values covered once, what is stored within the workspace
//   carries  (1-D, 36-value blocks) a carry in the index for every lane tile
//
// Built and run by tests/test_sz3d_lane.py with g++; prints "ok <cases>" or the
// first violation.
#include <cstdio>
#include <cstdlib>
#include <cstring>
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

static void split(uint32_t d1, uint32_t d2, uint32_t d3, int T)
{
    Geom3 g;
    std::vector<Part3> parts(T);
    if (!make_geom3(d1, d2, d3, 4, T, &g, parts.data()))
        return;
    // the table as the kernel fills it: each entry from its number, sums before it
    const Split3 sp = split3(g);
    Sums3 run = {};
    for (int t = 0; t < T; t++) {
        Part3 p;
        const Sums3 c = part3(g, sp, (uint32_t) t, p);
        place3(p, run);
        for (uint32_t i = 0; i < kSums3; i++)
            run.v[i] += c.v[i];
        const Part3& q = parts[t];
        REQUIRE(std::memcmp(&p, &q, sizeof(p)) == 0, "entry %d", t);
        REQUIRE(q.ox + q.sx <= d1 && q.oy + q.sy <= d2 && q.oz + q.sz <= d3 && q.sx && q.sy && q.sz, "part %d", t);
        if (t + 1 < T) {
            const Part3& n = parts[t + 1];
            REQUIRE(n.oz == q.oz + q.sz || (n.oz == 0 && (n.oy == q.oy + q.sy || (n.oy == 0 && n.ox == q.ox + q.sx))), "next");
        }
    }
    // lane compress: lanes 1..63 of a wave hold its run, tiles do not cross sub-volumes
    std::vector<int> seen(g.nblocks, 0);
    REQUIRE(g.nlane <= g.nblocks, "the tiles' words lie where the block offsets do");
    for (uint32_t t = 0; t < g.nlane; t++) {
        const Part3& p = parts[part_of_lane_tile(parts.data(), g.T, t)];
        const uint32_t nbp = p.b1 * p.b2 * p.b3;
        for (uint32_t wv = 0; wv < g.wlane; wv++)
            for (uint32_t lane = 1; lane < 64; lane++) {
                const uint32_t lb = kLaneRun3 * (g.wlane * (t - p.l0) + wv) + lane - 1;
                if (lb < nbp)
                    seen[p.g0 + lb]++;
            }
    }
    for (uint32_t b = 0; b < g.nblocks; b++)
        REQUIRE(seen[b] == 1, "block %u in %d tiles", b, seen[b]);
    g_cases++;
    if (!g.nruns)
        return;
    // decoder: runs as k3l_sizes reads them, rows as k3l_decode takes them
    const Ws3 ws = ws3_layout(g.nblocks, g.T);
    REQUIRE(4ull * g.nruns <= ws.offs - ws.words, "the runs' words");
    REQUIRE(8ull * (ceil_div(g.nruns, 256) + 1) <= ws.parts - ws.sums, "the run groups' sums and the total");
    REQUIRE(4ull * g.ntail <= ws.sums - ws.offs, "the kept planes");
    std::vector<int> runs(g.nblocks, 0), rows(g.nblocks, 0);
    std::vector<uint32_t> run_of(g.nblocks, 0);
    for (uint32_t u = 0; u < g.nruns; u++) {
        uint32_t t = 0;
        while (t + 1 < g.T && parts[t + 1].v0 <= u)
            t++;
        const Part3& p = parts[t];
        const uint32_t nz = (p.b3 + 63) / 64, rel = u - p.v0, row = rel / nz, z0 = 64 * (rel - row * nz);
        REQUIRE(row < p.b1 * p.b2, "row of run %u", u);
        for (uint32_t i = 0; i < 64 && z0 + i < p.b3; i++) {
            runs[p.g0 + row * p.b3 + z0 + i]++;
            run_of[p.g0 + row * p.b3 + z0 + i] = u;
        }
    }
    std::vector<char> tail(g.ntail, 0);
    uint64_t kept = 0;
    for (uint32_t b = 0; b < g.nrows; b++) {
        uint32_t t = 0;
        while (t + 1 < g.T && parts[t + 1].d0 <= b)
            t++;
        const Part3& p = parts[t];
        const uint32_t nseg = (p.b1 + kLaneSeg3 - 1) / kLaneSeg3, nz = (p.b3 + 63) / 64;
        const uint32_t by = (b - p.d0) / nseg, seg = b - p.d0 - by * nseg, ey = p.sy - 4 * by < 4 ? p.sy - 4 * by : 4;
        REQUIRE(by < p.b2 && nz <= g.wruns && g.wruns <= kLaneRuns3, "row %u", b);
        for (uint32_t bx = kLaneSeg3 * seg; bx < kLaneSeg3 * (seg + 1) && bx < p.b1; bx++)
            for (uint32_t bz = 0; bz < p.b3; bz++) {
                const uint32_t row = bx * p.b2 + by, i = p.g0 + row * p.b3 + bz;
                rows[i]++;
                REQUIRE(run_of[i] == p.v0 + row * nz + bz / 64, "run of a block");
            }
        if (seg + 1 < nseg)
            for (uint32_t j = 0; j < ey; j++)
                for (uint32_t z = 0; z < p.sz; z++) {
                    const uint64_t at = p.t0 + ((uint64_t) seg * p.sy + 4 * by + j) * p.sz + z;
                    REQUIRE(at < g.ntail && !tail[at], "kept value %llu", (unsigned long long) at);
                    tail[at] = 1;
                    kept++;
                }
    }
    for (uint32_t b = 0; b < g.nblocks; b++)
        REQUIRE(runs[b] == 1 && rows[b] == 1, "block %u: %d runs, %d rows", b, runs[b], rows[b]);
    REQUIRE(kept == g.ntail, "kept planes");
    uint64_t cols = 0;
    for (const Part3& p : parts) {
        REQUIRE(p.h0 == cols, "y columns");
        cols += (uint64_t) p.b1 * p.sz;
    }
    REQUIRE(cols == g.nhcol, "y columns");
}

static void carries()
{
    for (uint64_t n : {1ull, 2ull, 37ull, 38ull, 2305ull, 2306ull, 99991ull, 1000003ull, 16777216ull, 2147483647ull})
        for (uint32_t T : {1u, 2u, 7u, 16u, 64u, 1000u}) {
            Geom g;
            if (!make_geom(n, kLaneL, T, &g))
                continue;
            REQUIRE(lane_layout_ok(g), "36-value blocks");
            const Tiling tl = make_lane_tiling(g);
            REQUIRE(g.ncarry == tl.ntiles && g.cT == tl.tilesT && g.cR == tl.tilesR, "n %llu T %u", (unsigned long long) n, T);
            REQUIRE(g.ix_carry >= g.ix_meta + 32 && g.ix_carry % 4 == 0, "carries behind the meta words");
            REQUIRE((uint64_t) g.ix_carry + 4ull * g.ncarry <= g.ix_bytes, "carries inside the index");
            g_cases++;
        }
}

int main()
{
    routes();
    long_rows();
    carries();
    const uint32_t sides[] = {1, 3, 4, 5, 29, 64, 67, 130, 257};
    for (uint32_t a : sides)
        for (uint32_t b : sides)
            for (uint32_t c : {1u, 4u, 61u, 128u, 259u})
                for (int T : {1, 2, 6, 16, 65})
                    split(a, b, c, T);
    for (const auto& v : {std::vector<uint32_t>{256, 192, 256, 16}, {250, 190, 250, 16}, {200, 350, 250, 9}, {260, 192, 260, 4},
             {131, 195, 515, 2}, {67, 257, 1021, 1}, {66, 256, 1024, 1}, {300, 300, 300, 16}, {33, 800, 1024, 1}})
        split(v[0], v[1], v[2], (int) v[3]);
    std::printf("ok %ld\n", g_cases);
    return 0;
}
