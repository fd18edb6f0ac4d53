// zccl_sz3d.h -- geometry of the 3-D SZp codec shared by the host launchers
// and the kernels (zccl_sz3d.hip).
//
// Stream (reference: SZp_compress3D_fast_openmp, ZCCL/src/ZCCL_float.c:
// 1862-2048, and its decoder ZCCL/src/ZCCLd_float.c:2873-3040):
//   [T x u64 payload offsets, relative to the end of this header]
//   [payload of sub-volume 0] ... [payload of sub-volume T-1]
//   payload = one width byte per block (all blocks of the sub-volume, x, y, z
//   order), then for each block of nonzero width w: the MSB-first sign bitmap
//   of its values and their fixed-length bits (w >> 3 little-endian high bytes
//   per value, then the low w & 7 bits MSB-first), values in (i, j, k) order.
// The volume d1 x d2 x d3 (d3 fastest) is cut into T sub-volumes by the
// factorisation of T into three dims (My_Dims_create), every sub-volume into
// cubic blocks of side Bs (smaller at its far edges).  A value's residual is
// the 3-D difference dx dy dz q of q = floor(x * (0.5 / eb) + 0.5) with q = 0
// outside its sub-volume; the decoder is the 3-D prefix sum.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "zccl_internal.h"

namespace zk {

constexpr int kMaxParts3 = 4096;     // sub-volumes (the reference's OpenMP team size)
constexpr uint32_t kMaxBs3 = 64;     // block side: a payload (< 2^26 bytes) and its width share a word

struct Part3 {
    uint32_t ox, oy, oz;   // first plane along each axis
    uint32_t sx, sy, sz;   // planes along each axis
    uint32_t b1, b2, b3;   // blocks along each axis
    uint32_t g0;           // global index of the sub-volume's first block
    uint32_t nbc;          // blocks of the sub-volumes before it
    uint32_t zr0;          // first z-row (x, y pair) of the sub-volume in the z pass
    uint32_t yc0;          // first y-column (x, z pair) in the y pass
    uint32_t xc0;          // first x-column (y, z pair) in the x pass
    uint32_t u0;           // first chunk of the tiled compress (block side 8)
    uint32_t c0;           // first block column (bx, by) of the tiled decoder
    uint32_t l0;           // first workgroup tile of the lane compress (block side 4)
    uint32_t v0;           // lane decoder: first run of 64 blocks along z
    uint32_t d0;           // its first workgroup (a row of blocks along z, kLaneSeg3 of them along x)
    uint32_t t0;           // first of its segments' last planes
    uint32_t h0;           // first column (bx, z) of its y pass
};

struct Geom3 {
    uint32_t d1, d2, d3;
    uint32_t Bs, T;
    uint32_t nblocks;      // all blocks of all sub-volumes
    uint32_t zrows, ycols, xcols;
    uint32_t nunits;       // chunks of the tiled compress (0: no tiled path)
    uint32_t ncols;        // block columns of the tiled decoder
    uint32_t nlane;        // workgroup tiles of the lane compress (0: not that path)
    uint32_t wlane;        // waves of such a tile
    uint32_t nruns;        // runs of the lane decoder (0: not that path)
    uint32_t nrows;        // its workgroups
    uint32_t ntail;        // values of its segments' last planes
    uint32_t nhcol;        // columns of its y pass
    uint32_t wruns;        // runs (waves) to a row
    uint32_t edges;        // some sub-volume has blocks of fewer values
};

// Blocks per chunk along z of the tiled kernels: a chunk is one (bx, by)
// column of blocks cut to tile_nz3 blocks, whose quantized values with a
// one-value halo fit in LDS.  0 where the tiled path has no instance.
ZK_HD constexpr uint32_t tile_nz3(uint32_t Bs) { return Bs == 4 ? 64u : Bs == 8 ? 8u : 0u; }

// Lane compress (block side 4): one lane per block, a wave per run of
// kLaneRun3 blocks of a sub-volume in stream order (lane 0 holds the block
// before the run), kLaneWide3 waves per workgroup tile, or kLaneSlim3 below
// kLaneFew3 values, where wide tiles leave compute units idle.  A block's rows
// are addressed by 32-bit offsets: at most 3 d3 with four of them, which is below
// the volume's values (kMaxN).
constexpr uint32_t kLaneRun3 = 63;
constexpr uint32_t kLaneSlim3 = 4, kLaneWide3 = 12;
constexpr uint64_t kLaneFew3 = 64ull * kLaneRun3 * kLaneWide3 * 256;

// Lane decoder (block side 4): one lane per block, a wave per run of 64 blocks
// along z (kLaneRuns3 to a row at most), a workgroup per row of blocks and
// kLaneSeg3 blocks along x.  Rows shorter than kLaneMinB3 blocks leave most
// lanes idle and take the tiled kernels.  So do volumes that give the decoder
// fewer than three waves for each of 256 compute units, or its y pass (a thread
// per four columns, serial along y) less than one: what one wave waits for
// then sets the pace, and the tiled kernels have four times the threads.  us by
// lanes / tiled: 118 x 27 x 194 in 4 sub-volumes, 56 waves: 79 / 42; 64 x 336 x 320
// in 2, 336 waves: 150 / 86; 167 x 342 x 264, 1032 waves and 173 in the y pass: 175 /
// 131; 448 x 320 x 176, 1120 and 308: 156 / 179; 256^3 in 16, 1024 and 512: 100 / 117;
// 512^3: 387 / 757.  (Of 270 volumes of 24 to 512 a side the line leaves a few with
// long x and short y to the slower one: 502 x 40 x 130, 160 waves: 86 / 106.)  The last
// plane of every segment but a sub-volume's last is kept for the y pass: at most
// 8 bytes per block.
constexpr uint32_t kLaneSeg3 = 8, kLaneMinB3 = 32, kLaneRuns3 = 4;
constexpr uint32_t kLaneWaves3 = 3 * 256, kLaneCols3 = 64 * 256;

// Factorise T over three dims as My_Dims_create (ZCCL/src/ZCCL_multidim.c:
// 100-140): prime factors of T, largest first, each multiplied into the
// currently smallest dim (the first on ties); dims sorted descending.
ZK_HD void dims_create3(int T, int d[3])
{
    d[0] = d[1] = d[2] = 1;
    int f[32], nf = 0, rem = T;
    for (int i = 2; i <= rem && nf < 32; i++)
        while (rem % i == 0 && nf < 32) {
            f[nf++] = i;
            rem /= i;
        }
    for (int a = 0; a < nf; a++)
        for (int b = a + 1; b < nf; b++)
            if (f[b] > f[a]) {
                int t = f[a];
                f[a] = f[b];
                f[b] = t;
            }
    for (int i = 0; i < nf; i++) {
        int m = 0;
        for (int j = 1; j < 3; j++)
            if (d[j] < d[m])
                m = j;
        d[m] *= f[i];
    }
    for (int a = 0; a < 3; a++)
        for (int b = a + 1; b < 3; b++)
            if (d[b] > d[a]) {
                int t = d[a];
                d[a] = d[b];
                d[b] = t;
            }
}

ZK_HD uint32_t nblk3(uint32_t s, uint32_t Bs) { return (s - 1) / Bs + 1; }

// The cut of a volume along each dim: td parts of b values, the first r of them
// of one more.
struct Split3 {
    uint32_t td[3], b[3], r[3];
};

ZK_HD Split3 split3(const Geom3& g)
{
    int td[3];
    dims_create3((int) g.T, td);
    const uint32_t d[3] = {g.d1, g.d2, g.d3};
    Split3 s;
    for (int i = 0; i < 3; i++) {
        s.td[i] = (uint32_t) td[i];
        s.b[i] = d[i] / s.td[i];
        s.r[i] = d[i] % s.td[i];
    }
    return s;
}

// What one sub-volume adds to the table's running sums.
constexpr uint32_t kSums3 = 11;
struct Sums3 {
    uint32_t v[kSums3];  // blocks, zr, yc, xc, u, c, l, v, d, t, h
};

// Sub-volume t's place and extents, and its share of the sums.
ZK_HD Sums3 part3(const Geom3& g, const Split3& s, uint32_t t, Part3& p)
{
    const uint32_t yz = s.td[1] * s.td[2], px = t / yz, py = (t - px * yz) / s.td[2], pz = t - px * yz - py * s.td[2];
    p.sx = s.b[0] + (px < s.r[0] ? 1u : 0u);
    p.sy = s.b[1] + (py < s.r[1] ? 1u : 0u);
    p.sz = s.b[2] + (pz < s.r[2] ? 1u : 0u);
    p.ox = px * s.b[0] + (px < s.r[0] ? px : s.r[0]);
    p.oy = py * s.b[1] + (py < s.r[1] ? py : s.r[1]);
    p.oz = pz * s.b[2] + (pz < s.r[2] ? pz : s.r[2]);
    p.b1 = nblk3(p.sx, g.Bs);
    p.b2 = nblk3(p.sy, g.Bs);
    p.b3 = nblk3(p.sz, g.Bs);
    const uint32_t cols = p.b1 * p.b2, segs = (p.b1 + kLaneSeg3 - 1) / kLaneSeg3;
    const uint32_t nz = tile_nz3(g.Bs), lane = g.Bs == 4 ? g.wlane * kLaneRun3 : 0u;
    Sums3 c = {{cols * p.b3, p.sx * p.sy, p.sx * p.sz, p.sy * p.sz, nz ? cols * ((p.b3 + nz - 1) / nz) : 0u, cols,
        lane ? (cols * p.b3 + lane - 1) / lane : 0u, cols * ((p.b3 + 63) / 64), p.b2 * segs, (segs - 1) * p.sy * p.sz,
        p.b1 * p.sz}};
    return c;
}

// The sums over the sub-volumes before it.
ZK_HD void place3(Part3& p, const Sums3& c)
{
    p.g0 = p.nbc = c.v[0];
    p.zr0 = c.v[1];
    p.yc0 = c.v[2];
    p.xc0 = c.v[3];
    p.u0 = c.v[4];
    p.c0 = c.v[5];
    p.l0 = c.v[6];
    p.v0 = c.v[7];
    p.d0 = c.v[8];
    p.t0 = c.v[9];
    p.h0 = c.v[10];
}

// Fill g and parts[T] (sub-volumes in thread order, ZCCL/src/ZCCL_float.c:
// 1901-1935); false when the geometry is out of range or a sub-volume would be
// empty (the reference's DSize3D_init underflows then).
ZK_HD bool make_geom3(uint64_t d1, uint64_t d2, uint64_t d3, int Bs, int T, Geom3* g, Part3* parts)
{
    if (T < 1 || T > kMaxParts3 || Bs < 1 || (uint32_t) Bs > kMaxBs3 || d1 < 1 || d2 < 1 || d3 < 1)
        return false;
    if (d1 * d2 * d3 > kMaxN)
        return false;
    g->d1 = (uint32_t) d1;
    g->d2 = (uint32_t) d2;
    g->d3 = (uint32_t) d3;
    g->Bs = (uint32_t) Bs;
    g->T = (uint32_t) T;
    const Split3 s = split3(*g);
    if (!s.b[0] || !s.b[1] || !s.b[2])
        return false;
    g->wlane = (uint64_t) g->d1 * g->d2 * g->d3 < kLaneFew3 ? kLaneSlim3 : kLaneWide3;
    Sums3 sum = {};
    for (uint32_t t = 0; t < g->T; t++) {
        const Sums3 c = part3(*g, s, t, parts[t]);
        place3(parts[t], sum);
        for (uint32_t i = 0; i < kSums3; i++)
            sum.v[i] += c.v[i];
    }
    g->nblocks = sum.v[0];
    g->zrows = sum.v[1];
    g->ycols = sum.v[2];
    g->xcols = sum.v[3];
    g->nunits = sum.v[4];
    g->ncols = sum.v[5];
    g->nlane = sum.v[6];
    g->nrows = sum.v[8];
    g->ntail = sum.v[9];
    g->nhcol = sum.v[10];
    const uint32_t b3lo = nblk3(s.b[2], g->Bs), b3hi = nblk3(s.b[2] + (s.r[2] ? 1u : 0u), g->Bs);
    g->wruns = (b3hi + 63) / 64;
    const bool runs = Bs == 4 && b3lo >= kLaneMinB3 && b3hi <= 64 * kLaneRuns3 &&
                      (uint64_t) g->nrows * g->wruns >= kLaneWaves3 && g->nhcol >= kLaneCols3;
    g->nruns = runs ? sum.v[7] : 0u;
    g->edges = (s.b[0] | s.b[1] | s.b[2]) & 3 || s.r[0] || s.r[1] || s.r[2] ? 1u : 0u;  // (block side 4)
    return true;
}

// Payload bytes of a block of n values at width w (no width byte).
ZK_HD uint32_t payload3(uint32_t w, uint32_t n) { return w ? block_bytes(w, n) - 1 : 0u; }

// Worst case: every block at width 32.
ZK_HD uint64_t worst_case_bytes3(const Geom3& g, const Part3* parts)
{
    uint64_t tot = 8ull * g.T + g.nblocks;
    for (uint32_t t = 0; t < g.T; t++) {
        const Part3& p = parts[t];
        const uint64_t n = (uint64_t) p.sx * p.sy * p.sz;
        tot += 4 * n + n / 8 + (uint64_t) p.b1 * p.b2 * p.b3;
    }
    return tot;
}

// Index of the sub-volume holding global block gb (binary search over g0).
ZK_HD uint32_t part_of_block(const Part3* parts, uint32_t T, uint32_t gb)
{
    uint32_t lo = 0, hi = T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (parts[mid].g0 <= gb)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Sub-volume of workgroup tile v of the lane compress, by binary search.
ZK_HD uint32_t part_of_lane_tile(const Part3* parts, uint32_t T, uint32_t v)
{
    uint32_t lo = 0, hi = T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (parts[mid].l0 <= v)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Sub-volume of a tiled work item (first chunk u0, or first block column c0
// with cols set), by binary search over the table.
ZK_HD uint32_t part_of_unit(const Part3* parts, uint32_t T, uint32_t v, bool cols)
{
    uint32_t lo = 0, hi = T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if ((cols ? parts[mid].c0 : parts[mid].u0) <= v)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// A chunk of the tiled kernels: block column (bx, by) of sub-volume p, cut to
// tile_nz3(Bs) blocks along z; rel is the chunk's index inside p (column
// major: rel = (bx * b2 + by) * chunks per column + ch).
struct Chunk3 {
    uint32_t bx, by, ch;   // block column and chunk along z
    uint32_t ex, ey;       // extents of the column's blocks in x and y
    uint32_t lz0, wz, nbz; // chunk's first local z, z values, blocks
    uint32_t gcol;         // global index of the chunk's first block
};

ZK_HD Chunk3 chunk_of3(const Part3& p, uint32_t rel, uint32_t Bs)
{
    const uint32_t nz = tile_nz3(Bs), wzmax = nz * Bs;
    Chunk3 c;
    const uint32_t nch = (p.b3 + nz - 1) / nz;
    const uint32_t col = rel / nch;
    c.ch = rel - col * nch;
    c.bx = col / p.b2;
    c.by = col - c.bx * p.b2;
    c.ex = p.sx - c.bx * Bs < Bs ? p.sx - c.bx * Bs : Bs;
    c.ey = p.sy - c.by * Bs < Bs ? p.sy - c.by * Bs : Bs;
    c.lz0 = c.ch * wzmax;
    c.wz = p.sz - c.lz0 < wzmax ? p.sz - c.lz0 : wzmax;
    c.nbz = (c.wz + Bs - 1) / Bs;
    c.gcol = p.g0 + (c.bx * p.b2 + c.by) * p.b3 + c.ch * nz;
    return c;
}

// Device workspace of one 3-D call, in order: 256 bytes of status words
// (status[0] stream size, status[1] error bits, status[2] the next tile ticket), the per-block size words,
// their exclusive scan (u64), the scan's per-group sums (+ the total) and the
// sub-volume table.
constexpr uint32_t kScan3Group = 1024;  // entries per scan group

struct Ws3 {
    uint64_t words, offs, sums, parts, bytes;
};

ZK_HD Ws3 ws3_layout(uint32_t nblocks, uint32_t T)
{
    Ws3 w;
    const uint64_t groups = ceil_div(nblocks ? nblocks : 1, kScan3Group);
    w.words = 256;
    w.offs = w.words + align_up(4ull * nblocks, 256);
    w.sums = w.offs + align_up(8ull * nblocks + 8, 256);
    w.parts = w.sums + align_up(8ull * groups + 8, 256);
    w.bytes = w.parts + align_up(sizeof(Part3) * T, 256);
    return w;
}

}  // namespace zk
