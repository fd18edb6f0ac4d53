// zccl_lane.hip -- block-per-lane kernels for 36-value blocks, the
// reference's default block length (examples/compression_allreduce.c,
// jobs/*.sh): the fused homomorphic sum, decompress with the carries of a parsed
// stream, and compress.
//
// Layout (of the sum; the others' stand at their sections).  A wave owns one tile of 64 consecutive blocks of one segment and
// every lane owns one whole block.  An operand's tile bytes move into the
// wave's LDS buffer with range-checked direct-to-LDS loads (a read past the
// operand's stream returns zeros, so no read ever leaves the stream) and each
// lane reads its block with aligned dword reads, decodes its 36 deltas and adds
// them in int32.  No workgroup barrier sits on this path: the only per-operand
// cross-lane step is one DPP scan of block sizes that places each lane's block.
// The next operand's loads are in flight while the current one is decoded.
//
// Each wave is a tile of the decoupled lookback; a workgroup of four or eight
// waves takes one ticket for as many consecutive tiles.  The summed block is
// re-encoded into the wave's own LDS buffer with OR-writes of dwords (the
// buffer is zeroed first, and a lane ORs zeros wherever its dwords overlap a
// neighbour's bytes, so overlapping writes need no ordering) and leaves with
// 16-byte stores.
//
// A segment's short last block takes the same path as a whole one (its fields
// are placed by its length).  Blocks of width 16 and more have a decoder of
// their own, after the others of their tile; tiles larger than half the buffer
// take a pass of their own through the whole buffer.
// Measured against one decoder for whole blocks below width 16 with the others
// read value by value from memory: two 1 MB operands 15.7 -> 13.8 us, sixteen 8 MB
// ones 60 -> 31 us, 8 sums of 8 x 2^24 values 457 -> 422 us, the staged allreduce of
// 4 ranks' velocities (widths 15 to 17) 383 -> 220 us, decompress of 16411 values (a
// short block in every tile) 11.4 -> 8.9 us.
//
// Wire format and arithmetic (reference):
//   block      width byte, sign bitmap MSB first, (w>>3) high bytes per
//              value, MSB-first low (w&7) bits     ZCCL/src/ZCCL_TypeManager.c:12-91, 824-848
//   sum        deltas add in int32, block re-encoded at the width of the
//              largest magnitude                   ZCCL/src/ZCCLd_float.c:1099-1219
//   width      (int)log2f((float)max)+1             ZCCL/src/ZCCLd_float.c:1205
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "zccl_device.h"
#include "zccl_internal.h"
#include "zccl_kernels.h"
#include "zccl_pack.h"

namespace zk {

// Dynamic LDS: one output buffer per wave, 16-byte aligned (the buffers are
// zeroed with 16-byte stores).
extern __shared__ __attribute__((aligned(16))) uint32_t zk_lds[];

namespace {

constexpr uint32_t L = kLaneL;          // values per block
constexpr uint32_t SB = (L + 7) / 8;    // sign bytes of a whole block
constexpr uint32_t NHI = L / 4;         // dwords of one high byte per value
constexpr uint32_t NGRP = (L + 7) / 8;  // groups of (up to) 8 values in the low bits
constexpr uint32_t kWorstBlock = 1 + SB + 4 * L;   // 150 bytes at width 32
// Output buffer of one wave: 10 KB, so that a CU's 160 KB of LDS hold those of
// sixteen waves, and nothing else (the sum's loop holds 108 to 120 registers, and
// more than 96 leave four waves to a SIMD).  The worst tile's bytes (64 blocks of
// kWorstBlock) fit, with the reach of the block reads and OR-writes past them.
constexpr uint32_t kOutBuf = 10240;
// Block reads and writes cover 36 values whatever the block holds: a short
// last block's reach at most 6 + 4 * 37 bytes past its first byte.
constexpr uint32_t kReach = 160;
static_assert(kReach >= 1 + SB + 4 * (L + 1), "the reach of a short block's reads and writes");
static_assert(kLaneTileBlocks * kWorstBlock + 16 + kReach <= kOutBuf, "a worst-case tile fits a wave buffer");
static_assert(kOutBuf % 16 == 0, "wave buffers stay 16-byte aligned");

static_assert(L % 4 == 0 && L > 32 && L <= 40, "the lane decoder is laid out for 36-value blocks");

// Encoded size of a whole block at width w (w = 0..32): 1 + SB + 36 B +
// ceil(36 r / 8) = 6 + ceil(9 w / 2).
// a * b + c for a, b below 2^24: one full-rate instruction (the compiler
// picks a quarter-rate 32-bit multiply where it cannot prove the range).
__device__ __forceinline__ uint32_t mad_u24(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t d;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

__device__ __forceinline__ uint32_t full_block_bytes(uint32_t w) { return w ? 6u + (mad_u24(w, 9u, 1u) >> 1) : 1u; }

// block_bytes for n <= L values at width w <= 32.
__device__ __forceinline__ uint32_t lane_block_bytes(uint32_t w, uint32_t n)
{
    return w ? 1u + ((n + 7u) >> 3) + mad_u24(w >> 3, n, (mad_u24(w & 7u, n, 7u) >> 3)) : 1u;
}

using View = __amdgpu_buffer_rsrc_t;

// Range-checked view of [base, base + bytes) (base 4-byte aligned, bytes a
// multiple of 4).  A buffer load returns zeros for every dword that does not
// lie wholly inside the view, whatever its alignment: a dword load at an
// unaligned offset that reaches past the view's last dword reads as zero even
// where its first bytes are inside.
__device__ __forceinline__ View make_view(const uint8_t* base, uint64_t bytes)
{
    const uint32_t n = bytes > 0xFFFFFFFCull ? 0xFFFFFFFCu : (uint32_t) bytes;
    return __builtin_amdgcn_make_buffer_rsrc((void*) base, (short) 0, (int) n, 0x00020000);
}

__device__ __forceinline__ uint4 bl16(View v, uint32_t off)
{
    const auto x = __builtin_amdgcn_raw_buffer_load_b128(v, off, 0, 0);
    return make_uint4(x[0], x[1], x[2], x[3]);
}

// A value that every lane holds, in scalar registers.
__device__ __forceinline__ uint64_t uniform64(uint64_t v)
{
    const uint32_t hi = (uint32_t) __builtin_amdgcn_readfirstlane((uint32_t) (v >> 32));
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readfirstlane((uint32_t) v);
    return ((uint64_t) hi << 32) | lo;
}

// Read-only data of the launch (descriptors, input indices) through the
// scalar cache when the address is the same for the whole wave.
template <typename T>
__device__ __forceinline__ T ldc(const T* p)
{
    return *(const __attribute__((address_space(4))) T*) (uintptr_t) p;
}


// a * b + c for a, b of 24 bits (signed) and any c, in one instruction.
__device__ __forceinline__ uint32_t mad_i24(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t d;
    asm volatile("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

// A lane's block in registers: the sign words (value j at bit 31 - j, value
// 32 + j of s2 likewise), the big-endian dwords at the first byte of each
// group of 8 values' low bits, and, where some lane of the wave has a width
// in [8, 16), one high byte per value.
struct Block {
    uint32_t s, s2;
    uint32_t ge[2 * NGRP];
    uint32_t hi[NHI];
};

// Read a block of nj <= L values and width w < 16 from tile bytes in LDS (the
// block at byte o of st): a short block's fields are placed by nj like a
// whole one's, so both take this path; values past nj read what follows.
// wide: some lane of the wave has w >= 8 (uniform).
__device__ __forceinline__ void read_block(const uint32_t* st, uint32_t o, uint32_t w, uint32_t nj, bool wide, Block& q)
{
    const uint32_t* p = st + (o >> 2);
    const uint32_t x0 = __builtin_amdgcn_alignbyte(p[1], p[0], o), x1 = __builtin_amdgcn_alignbyte(p[2], p[1], o);
    q.s = __builtin_amdgcn_perm(x1, x0, 0x01020304u);  // sign bytes 0..3 big-endian
    q.s2 = x1 << 16;                                   // sign byte 4 on top
    const uint32_t hp = o + 1 + ((nj + 7) >> 3);
    uint32_t a = hp, r = w;
    if (wide) {
        const uint32_t* ph = st + (hp >> 2);
        uint32_t d = ph[0];
#pragma unroll
        for (uint32_t i = 0; i < NHI; i++) {
            const uint32_t e = ph[i + 1];
            q.hi[i] = __builtin_amdgcn_alignbyte(e, d, hp);
            d = e;
        }
        a += w & 8 ? nj : 0u;
        r = w & 7;
    }
#pragma unroll
    for (uint32_t g = 0; g < NGRP; g++, a += r) {
        const uint32_t* pg = st + (a >> 2);
        const uint32_t E0 = pg[0], E1 = pg[1], E2 = pg[2];
        q.ge[2 * g] = __builtin_bswap32(__builtin_amdgcn_alignbyte(E1, E0, a));
        q.ge[2 * g + 1] = __builtin_bswap32(__builtin_amdgcn_alignbyte(E2, E1, a));
    }
}

// The values of a block of width w < 16: f(j, magnitude, +1 or -1).  A zero
// width gives zeros whatever was read.  wide (uniform): the high bytes were
// read; they join the low bits group by group behind a branch of their own, so
// tiles without any skip them and the decoder stays one piece of code (two
// whole decoders behind one branch cost the sum 10 to 36 spilled registers per
// operand).  Three instructions per value and the sum's multiply-add: a
// bit-field extract at one of four places of the half group's window, another
// for the sign.  (Shifts, masks and FP32 adds that take 2 cycles each in their
// place were five instructions and slower: the sum issues, it does not wait for
// the units.)
// ZCCL/src/ZCCL_TypeManager.c:423-517 (extract), :906-950 (signs).
template <typename F>
__device__ __forceinline__ void each_value(const Block& q, uint32_t w, bool wide, F f)
{
    const uint32_t r = w & 7, hb = w & 8;  // hb: bits per high byte (0 or 8)
    const uint32_t sh[4] = {32 - r, 32 - 2 * r, 32 - 3 * r, 32 - 4 * r};
    // Sign words: a value's sign bit moved to an odd bit with a one below it,
    // so the 2-bit field there reads -1 (sign set) or +1 as a signed number:
    // so the even values, se (shifted up one) the odd ones.
    uint32_t so = (q.s & 0xAAAAAAAAu) | 0x55555555u, se = ((q.s << 1) & 0xAAAAAAAAu) | 0x55555555u;
    uint32_t so2 = (q.s2 & 0xAAAAAAAAu) | 0x55555555u, se2 = ((q.s2 << 1) & 0xAAAAAAAAu) | 0x55555555u;
    // (opaque to the optimiser, which would otherwise extract the sign bit
    // alone and OR in the one: two instructions per value instead of one)
    asm volatile("" : "+v"(so), "+v"(se), "+v"(so2), "+v"(se2));
#pragma unroll
    for (uint32_t g = 0; g < NGRP; g++) {
        __builtin_amdgcn_sched_barrier(0);  // group by group: few registers live
        const uint32_t n = 8 * g + 8 <= L ? 8u : L - 8 * g;
        // the group's low bits big-endian: value 8g + c's field is r bits from
        // bit 64 - (c+1) r; value 4's window is bits 4r.. of the two dwords
        // (any value when r = 0)
        uint32_t m[8];
#pragma unroll
        for (uint32_t c = 0; c < n; c++) {
            const uint32_t win =
                c < 4 ? q.ge[2 * g] : __builtin_amdgcn_alignbit(q.ge[2 * g], q.ge[2 * g + 1], sh[3]);
            m[c] = __builtin_amdgcn_ubfe(win, sh[c & 3], r);
        }
        if (wide) {
#pragma unroll
            for (uint32_t c = 0; c < n; c++)
                m[c] |= __builtin_amdgcn_ubfe(q.hi[2 * g + (c >> 2)], 8 * (c & 3), hb) << r;
        }
#pragma unroll
        for (uint32_t c = 0; c < n; c++) {
            const uint32_t j = 8 * g + c, i = j & 31;
            const uint32_t sw = j < 32 ? ((i & 1) ? se : so) : ((i & 1) ? se2 : so2);
            f(j, m[c], (uint32_t) __builtin_amdgcn_sbfe((int32_t) sw, (31 - i) & ~1u, 2));
        }
    }
}

// The same for widths with B = w >> 3 = 2, 3 or 4 high bytes per value (lanes
// of that class only), straight from LDS: f(j, magnitude, sign word whose bit
// 31 is the value's sign).
template <uint32_t B, typename F>
__device__ __forceinline__ void each_value_high(const uint32_t* st, uint32_t o, uint32_t w, uint32_t nj, F f)
{
    static_assert(B >= 2 && B <= 4, "high bytes of a width from 16");
    const uint32_t r = w & 7, mask = (1u << r) - 1u;
    const uint32_t hp = o + 1 + ((nj + 7) >> 3);
    const uint32_t sh[4] = {32 - r, 32 - 2 * r, 32 - 3 * r, 32 - 4 * r};
    uint32_t s = __builtin_bswap32(lds_at(st, o + 1)), s2 = lds_at(st, o + 5) << 24;
    const uint32_t* ph = st + (hp >> 2);
    uint32_t a = hp + B * nj;
#pragma unroll
    for (uint32_t g = 0; g < NGRP; g++, a += r) {
        __builtin_amdgcn_sched_barrier(0);  // group by group: few registers live
        const uint32_t n = 8 * g + 8 <= L ? 8u : L - 8 * g;
        const uint32_t* pg = st + (a >> 2);
        const uint32_t E0 = pg[0], E1 = pg[1], E2 = pg[2];
        const uint32_t e0 = __builtin_bswap32(__builtin_amdgcn_alignbyte(E1, E0, a));
        const uint32_t e1 = __builtin_bswap32(__builtin_amdgcn_alignbyte(E2, E1, a));
        uint32_t h[2 * B + 1];  // the group's high bytes in memory order
        uint32_t d = ph[2 * B * g];
#pragma unroll
        for (uint32_t i = 0; i < n * B / 4; i++) {
            const uint32_t e = ph[2 * B * g + i + 1];
            h[i] = __builtin_amdgcn_alignbyte(e, d, hp);
            d = e;
        }
        h[n * B / 4] = 0;
        uint32_t win = e0;
#pragma unroll
        for (uint32_t c = 0; c < n; c++) {
            const uint32_t j = 8 * g + c;
            if (c == 4)
                win = __builtin_amdgcn_alignbit(e0, e1, sh[3]);
            const uint32_t m = (win >> (sh[c & 3] & 31)) & mask;
            uint32_t v;
            if constexpr (B == 2)
                v = (c & 1) ? h[c >> 1] >> 16 : h[c >> 1] & 0xFFFFu;
            else if constexpr (B == 3)
                v = __builtin_amdgcn_alignbyte(h[(3 * c) / 4 + 1], h[(3 * c) / 4], (3 * c) & 3) & 0xFFFFFFu;
            else
                v = h[c];
            // (two high bytes and r bits are below 2^24: the denormal product)
            const uint32_t mag = B == 2 ? as_u(__builtin_fmaf(as_f(v), as_f((127u + r) << 23), as_f(m))) : (v << r) | m;
            if (j < 32) {
                f(j, mag, s);
                s += s;
            } else {
                f(j, mag, s2);
                s2 += s2;
            }
        }
    }
}

// Lanes of the wave whose block takes each_value_high (w >= 16, `on`), by
// class.
template <typename F>
__device__ __forceinline__ void each_high_lane(const uint32_t* st, uint32_t o, uint32_t w, uint32_t nj, bool on, F f)
{
    if (on && (w >> 3) == 2)
        each_value_high<2>(st, o, w, nj, f);
    if (on && (w >> 3) == 3)
        each_value_high<3>(st, o, w, nj, f);
    if (on && w == 32)
        each_value_high<4>(st, o, w, nj, f);
}

// Add a block of any width (nj values, nj <= L) from LDS to acc, four values at
// a time; values past nj add garbage that the caller clears.  Each value's
// high bytes are read on their own: few registers, for the sum's rare tiles.
__device__ __forceinline__ void decode_any(const uint32_t* st, uint32_t o, uint32_t w, uint32_t nj, uint32_t (&acc)[L])
{
    w = stay(w);  // (or the loop around this would keep 45 offsets made from it)
    const uint32_t B = w >> 3, r = w & 7;
    const uint32_t hmask = B >= 4 ? ~0u : (1u << (8 * B)) - 1u;
    const uint32_t hp = o + 1 + ((nj + 7) >> 3), lp = hp + B * nj;
    uint32_t s = __builtin_bswap32(lds_at(st, o + 1)), s2 = lds_at(st, o + 5) << 24;
#pragma unroll
    for (uint32_t u = 0; u < L / 4; u++) {
        __builtin_amdgcn_sched_barrier(0);
        uint32_t H[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            H[c] = lds_at(st, hp + (4 * u + c) * B) & hmask;
        uint32_t lo = __builtin_bswap32(lds_at(st, lp + ((4 * u * r) >> 3))) << ((4 * u * r) & 4u);
        uint32_t& sw = u < 8 ? s : s2;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            const uint64_t x = (((uint64_t) H[c] << 32) | lo) << r;
            lo = (uint32_t) x;
            acc[4 * u + c] += signed_of((uint32_t) (x >> 32), sw);
            sw += sw;
        }
    }
}

// Encode the blocks of the lanes with w > 0 (nj <= L values; those past nj are
// zero) at byte o of the wave's zeroed buffer: width byte, sign bitmap MSB
// first, (w >> 3) high bytes per value, then the low r bits of every
// magnitude as an MSB-first stream (groups of 8 values fill r whole bytes).
// s: signs of values 0..31 (value j at bit 31 - j), s2: signs of values
// 32..35 (value 32 at bit 3); m: magnitudes.  The zeros past a short block's
// values land at most kReach bytes past its start.
// ZCCL/src/ZCCL_TypeManager.c:12-91 (fixed-length bits), :824-848 (signs).
__device__ __forceinline__ void encode_blocks(uint32_t* ob, uint32_t o, uint32_t w, uint32_t nj, uint32_t s, uint32_t s2,
    const uint32_t (&m)[L])
{
    const uint32_t hp = o + 1 + ((nj + 7) >> 3);
    const bool wide = __any(w >= 8);
    if (w) {
        const uint32_t sb = __builtin_bswap32(s);  // sign bytes 0..3 in memory order
        const uint32_t x[2] = {w | (sb << 8), (sb >> 24) | (s2 << (8 + 40 - L))};
        or_words(ob, o, x);
    }
    if (wide)
        encode_high_class(ob, hp, w, m);
    encode_low(ob, hp + (w >> 3) * nj, w, m);
}

// The operands of one sum: in device memory (read through the scalar cache)
// or in the kernel arguments.
struct SumIO {
    const HomsumIO* io;
    __device__ const uint8_t* bytes(int r) const { return ldc(&io->in[r].bytes); }
    __device__ const uint8_t* index(int r) const { return ldc(&io->in[r].index); }
};

struct ArgIO {
    const HomsumIO& io;
    __device__ const uint8_t* bytes(int r) const { return io.in[r].bytes; }
    __device__ const uint8_t* index(int r) const { return io.in[r].index; }
};

// Staging area of one operand's tile bytes: half of the wave's output buffer
// (the buffer is free until the encode), less the reach of the block reads
// past the staged bytes; the whole buffer for a tile that fits no half.
constexpr uint32_t kStageHalf = kOutBuf / 2;
constexpr uint32_t kStageCap = kStageHalf - kReach;
static_assert(kStageHalf % 16 == 0, "stage halves stay 16-byte aligned");

// Move the first tot bytes of view v into LDS at st with 16-byte
// direct-to-LDS buffer loads, 64 lanes per instruction; the view's range
// check zero-fills past the stream.
__device__ __forceinline__ void stage_bytes(View v, uint32_t tot, uint32_t* st)
{
    const uint32_t lane = threadIdx.x & 63, nch = (tot + 15) >> 4;
#pragma unroll 1
    for (uint32_t run = 0; run * 64 < nch; run++) {
        const uint32_t ch = run * 64 + lane;
        if (ch < nch)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(v,
                (__attribute__((address_space(3))) void*) ((uint8_t*) st + run * 1024), 16, 16 * ch, 0, 0, 0);
    }
}

__device__ __forceinline__ uint32_t staged_len(uint32_t tot) { return 16 * ((tot + 15) >> 4); }

// Shared state of a workgroup of lane waves that owns one lookback tile:
// each wave's bytes, and the tile's stream offset.
struct WgShared {
    uint32_t wtot[kLaneWaves];
    unsigned long long ex;
};

// The state of a workgroup of a sum, in the last bytes of its last wave's buffer,
// which neither the staging nor the encoder writes (the block reads past half
// one's bytes take it for garbage).  As static LDS beside the buffers it left a
// CU three workgroups of four waves for four, and one of eight for two: 8 operands
// of 2^24 values in one pass 90.7 -> 87.5 us by four waves, 100.4 -> 80.1 by eight.
struct SumShared {
    unsigned long long ticket;
    WgShared wg;
};
static_assert(kStageHalf + kStageCap + sizeof(SumShared) <= kOutBuf && sizeof(SumShared) % 8 == 0 &&
        kLaneTileBlocks * kWorstBlock + 16 + kReach + sizeof(SumShared) <= kOutBuf,
    "the workgroup's state lies behind what the waves write");
static_assert(16 / kLaneWaves * kLaneWaves * kOutBuf <= 160 * 1024, "sixteen waves' buffers fit a CU's LDS");

template <uint32_t W>
__device__ __forceinline__ SumShared& sum_shared()
{
    return *reinterpret_cast<SumShared*>(zk_lds + (W * kOutBuf - sizeof(SumShared)) / 4);
}

// Forms of the lane sum's output side.
enum SumMode : int {
    kSumWave = 0,    // single pass, a lookback tile per wave
    kSumStaged = 1,  // pass one of the two-pass sum: no lookback; the tile's bytes go to
                     // slot sidx of the stage area `area` of R tiles, its sizes and seed to
                     // record sidx, and only the widths to the output index
    kSumWg = 2,      // single pass, a lookback tile per workgroup of kLaneWaves waves
};

// One tile of a fused k-operand sum, executed by one wave.  obuf: the wave's
// LDS buffer (kOutBuf bytes, 16-byte aligned).  kSumWg: t is the wave's tile
// of the lane tiling, t_wg the workgroup's lookback tile (the last of the
// launch when wg_last), wsh the workgroup's shared state; every wave of the
// workgroup calls this (a wave past its segment's blocks with an empty tile).
template <int Mode, typename Src>
__device__ __forceinline__ void homsum_tile_lane(const Geom& g, const Tiling& tl, int k, const Src& src,
    uint8_t* out, uint64_t out_cap, uint8_t* oindex, unsigned long long* size_out, uint64_t t,
    unsigned long long* status, WsHeader* ws, uint32_t nchains, uint32_t* obuf, uint8_t* area = nullptr,
    uint64_t R = 0, uint64_t sidx = 0, uint64_t t_wg = 0, bool wg_last = false, WgShared* wsh = nullptr,
    const Tile* xe = nullptr)
{
    const uint32_t lane = threadIdx.x & 63;
    const Tile x = xe ? *xe : tile_of(g, tl, (uint32_t) t);
    const bool has = lane < x.nblk;
    const uint32_t nj = has ? min(tile_block_len(g, x, lane), L) : 0u;
    bool bad_byte = false, bad_width = false, bad_over = false;

    // ---- operand table: lane r < k holds operand r's stream, index, tile
    // offset and stream size, read once per tile; each operand's values come
    // out of it with readlane, so no operand waits on a scalar load chain
    const uint8_t* tb_bytes = nullptr;
    const uint8_t* tb_index = nullptr;
    uint64_t tb_goff = 0, tb_size = 0;
    uint32_t carry = 0;
    if (lane < (uint32_t) k) {
        tb_bytes = src.bytes((int) lane);
        tb_index = src.index((int) lane);
        const IndexView iv = index_view(g, tb_index);
        tb_goff = iv.group_off[x.grp0];
        tb_size = iv.meta[0];
        carry = iv.carry[t];
    }
    // (readlane returns int: widen through uint32_t, never by sign extension)
    auto rl64 = [](uint64_t v, int r) -> uint64_t {
        const uint32_t hi = (uint32_t) __builtin_amdgcn_readlane((uint32_t) (v >> 32), r);
        const uint32_t lo = (uint32_t) __builtin_amdgcn_readlane((uint32_t) v, r);
        return ((uint64_t) hi << 32) | lo;
    };
    struct Op {
        const uint8_t* bytes;
        const uint8_t* index;
        uint64_t goff, size;
    };
    auto op_of = [&](int r) {
        Op o;
        o.bytes = (const uint8_t*) rl64((uint64_t) tb_bytes, r);
        o.index = (const uint8_t*) rl64((uint64_t) tb_index, r);
        o.goff = rl64(tb_goff, r);
        o.size = rl64(tb_size, r);
        return o;
    };
    auto widths = [&](const Op& o) -> uint32_t { return has ? (uint32_t) o.index[x.g0 + lane] : 0u; };

    // this lane's block of an operand: width, size, offset in the operand's
    // view of the tile bytes (one scan of the block sizes), and whether the
    // tile lies inside its stream.  The view starts at the 4-byte aligned
    // address at or below the tile's bytes and ends with the stream's last
    // dword.
    struct Loc {
        View v;
        uint32_t w, bs, o, tot;
        bool skip;
    };
    auto locate = [&](const Op& p, uint32_t wq) {
        Loc c;
        c.w = wq;
        if (c.w > 32) {
            bad_width = true;
            c.w = 0;
        }
        c.bs = has ? (nj == L ? full_block_bytes(c.w) : lane_block_bytes(c.w, nj)) : 0u;
        const uint32_t incl = wave_scan_dpp(c.bs);
        c.tot = __builtin_amdgcn_readlane(incl, 63);
        c.skip = p.goff > p.size || c.tot > p.size - p.goff;
        const uint8_t* base = p.bytes + p.goff;
        const uint32_t delta = (uint32_t) ((uintptr_t) base & 3u);
        const uint64_t len = c.skip ? 0ull : align_up(delta + (p.size - p.goff), 4);
        c.v = make_view(base - delta, len);
        c.o = delta + incl - c.bs;
        c.tot += delta;  // bytes of the view that hold the tile
        return c;
    };
    // stage an operand's tile bytes into LDS half `half`; false when they do
    // not fit there
    auto stage = [&](const Loc& c, uint32_t half) -> bool {
        if (c.skip || staged_len(c.tot) > kStageCap)
            return false;
        stage_bytes(c.v, c.tot, obuf + half * (kStageHalf / 4));
        return true;
    };

    uint32_t acc[L];
#pragma unroll
    for (uint32_t j = 0; j < L; j++)
        acc[j] = 0;
    // bit r (uniform): operand r's tile does not fit a half and is left to the
    // pass below
    uint32_t whole = 0;

    // ---- operand pipeline: operand r+1's tile bytes move into the other LDS
    // half while operand r is decoded, operand r+2's widths are on their way
    {
        Op on = op_of(0);
        Loc cn = locate(on, widths(on));
        bool hn = stage(cn, 0);
        // the sum's carry into the tile: the operands' carries add in int32
        // (while the first operand's bytes are on their way)
        carry = wave_scan_dpp(carry);
        if (lane == 63 && x.ngrp)
            index_view(g, oindex).carry[t] = carry;
        if (hn || cn.skip) {
            Op o2;
            uint32_t wq2 = 0;
            if (k > 1) {
                o2 = op_of(1);
                wq2 = widths(o2);
            }
            // (a loop that runs at least once: its sums then have no second life
            // as the zeros of an empty one)
            int r = 0;
            do {
                const Loc c = cn;
                const bool half = hn;
                __builtin_amdgcn_s_waitcnt(0);  // operand r's bytes are in LDS, operand r+1's widths in registers
                // a lane of a wider block, or of a tile that is not here, decodes
                // zeros (without a branch: one would copy the sums)
                const uint32_t w = half && c.w < 16 ? c.w : 0u, o = half ? c.o : 0u;
                const bool wide = __any(w >= 8);
                const uint32_t* st = obuf + ((uint32_t) r & 1u) * (kStageHalf / 4);
                bad_byte |= (has && half) & (((const uint8_t*) st)[o] != c.w);
                Block q;
                read_block(st, o, w, nj, wide, q);
                // (phase fences keep the scheduler from interleaving the block
                // reads, the next operand's staging and the decode, which would
                // hold all their values at once)
                __builtin_amdgcn_sched_barrier(0);
                if (r + 1 < k) {
                    cn = locate(o2, wq2);
                    hn = stage(cn, (uint32_t) (r + 1) & 1u);
                }
                if (r + 2 < k) {
                    o2 = op_of(r + 2);
                    wq2 = widths(o2);
                }
                __builtin_amdgcn_sched_barrier(0);
                bad_over |= c.skip;
                whole |= !half && !c.skip ? 1u << r : 0u;
                each_value(q, w, wide, [&](uint32_t j, uint32_t v, uint32_t sign) { acc[j] = mad_i24(v, sign, acc[j]); });
                // (its bytes stay until operand r+2's)
                if (half && __builtin_expect(__any(c.w >= 16), 0)) {
                    if (c.w >= 16)
                        decode_any(st, c.o, c.w, nj, acc);
                }
            } while (++r < k);
        } else {
            // the first does not fit a half: nor will most of the others
            whole = ~0u >> (32 - k);
        }
    }
    // the operands left over, one at a time through the whole buffer, the next
    // one's widths on their way with the bytes of one.  (Twelve operands of 365 KB
    // with widths 15 to 17: 43 us, where a second fetch for every tile with a block
    // from width 16, and a pass of zeros for every one larger than a half, took 51;
    // eight of 16 MB: 48 and 55.)
    if (uint32_t left = whole; __builtin_expect(left != 0, 0)) {
        int r = __builtin_ctz(left);
        Op op = op_of(r);
        uint32_t wq = widths(op);
        while (true) {
            const Loc c = locate(op, wq);
            const bool mine = has && !c.skip;
            bad_over |= c.skip;
            if (!c.skip)
                stage_bytes(c.v, c.tot, obuf);
            left &= left - 1;
            if (left) {
                r = __builtin_ctz(left);
                op = op_of(r);
                wq = widths(op);
            }
            __builtin_amdgcn_s_waitcnt(0);
            bad_byte |= mine & (((const uint8_t*) obuf)[c.o] != c.w);
            if (mine && c.w)
                decode_any(obuf, c.o, c.w, nj, acc);
            if (!left)
                break;
        }
    }
    if (__any(nj < L)) {
        // values past a short block's end decoded what follows it
#pragma unroll
        for (uint32_t j = 0; j < L; j++)
            if (j >= nj)
                acc[j] = 0;
    }
    __builtin_amdgcn_sched_barrier(0);
    // signs (s: value j at bit 31 - j; s2: value 35 at bit 0), then the
    // magnitudes in place of the sums
    uint32_t s = 0, s2 = 0;
#pragma unroll
    for (uint32_t j = 0; j < L; j++) {
        if (j < 32)
            s = __builtin_amdgcn_alignbit(s, acc[j], 31);  // (s << 1) | sign of value j
        else
            s2 = __builtin_amdgcn_alignbit(s2, acc[j], 31);
    }
    // (phase fence: without it the scheduler computes the magnitudes before
    // the sign words and keeps both arrays live)
    __builtin_amdgcn_sched_barrier(0);
    uint32_t (&m)[L] = acc;
#pragma unroll
    for (uint32_t j = 0; j < L; j++)
        m[j] = mag(m[j]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_sched_barrier(0);
    if (__any(bad_width) && lane == 0)
        raise_error(ws, ZK_ERR_WIDTH);
    if (__any(bad_byte) && lane == 0)
        raise_error(ws, ZK_ERR_MISMATCH);
    if (__any(bad_over) && lane == 0)
        raise_error(ws, ZK_ERR_OVERRUN);

    // seed of the segment (its first tile): the operands' seeds add in int32
    uint32_t seed = 0;
    if (x.lt == 0) {
        uint32_t sv = 0;
        if (lane < (uint32_t) k) {
            const IndexView iv = index_view(g, tb_index);
            const uint64_t so = iv.seed_off[x.s];
            if (so + 4 <= tb_size)
                sv = load_u32_bytes(tb_bytes + so);
            else
                raise_error(ws, ZK_ERR_OVERRUN);
        }
        seed = (uint32_t) wave_sum64(sv);
    }

    // ---- widths, sizes, offsets
    uint32_t mx = 0;
#pragma unroll
    for (uint32_t j = 0; j < L; j++)
        mx = max(mx, m[j]);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t w = has ? dwidth(mx) : 0u;
    const uint32_t bs = has ? (nj == L ? full_block_bytes(w) : lane_block_bytes(w, nj)) : 0u;
    const uint32_t incl = wave_scan_dpp(bs);
    const uint32_t excl = incl - bs;
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    if (Mode == kSumWave && lane == 0)
        lookback_publish(status, t, 0, total, 0);  // successors see the aggregate now

    if constexpr (Mode == kSumWg) {
        // the workgroup's tile: its waves' bytes in wave order, one lookback
        const uint32_t wv = threadIdx.x >> 6;
        if (lane == 0)
            wsh->wtot[wv] = total;
        __syncthreads();
        uint32_t woff = 0, gtot = 0;
#pragma unroll
        for (uint32_t i = 0; i < kLaneWaves; i++) {
            const uint32_t v = wsh->wtot[i];
            woff += i < wv ? v : 0u;
            gtot += v;
        }
        if (threadIdx.x == 0)
            lookback_publish(status, t_wg, 0, gtot, 0);  // successors see the aggregate now
        const uint32_t nz = (total + 64 + 15) / 16;
        for (uint32_t i = lane; i < nz; i += 64)
            reinterpret_cast<uint4*>(obuf)[i] = make_uint4(0, 0, 0, 0);
        encode_blocks(obuf, excl, w, nj, s, s2, m);
        if (wv == 0) {
            const unsigned long long ex = lookback(status, t_wg, 0, gtot, 0, ws, true);
            if (lane == 0)
                wsh->ex = ex;
        }
        __syncthreads();
        const uint64_t hdr = 8ull * g.T + 4ull * (x.s + 1);
        const uint64_t P0 = hdr + wsh->ex;  // the workgroup tile's stream offset
        const uint64_t P = P0 + woff;       // this wave's
        const bool fits = P0 + gtot <= out_cap;
        if (fits)
            store_wave(obuf, out + P, total);
        if (!fits && threadIdx.x == 0)
            raise_error(ws, ZK_ERR_NOSPACE);
        IndexView ox = index_view(g, oindex);
        if (has)
            ox.widths[x.g0 + lane] = (uint8_t) w;
        if ((lane & 15) == 0 && lane / 16 < x.ngrp)
            ox.group_off[x.grp0 + lane / 16] = P + excl;
        if (lane == 0 && x.lt == 0) {
            const uint64_t so = P0 - 4;
            if (so + 4 <= out_cap) {
                store_bytes(out + so, &seed, 4);
                if (x.s < g.T) {
                    const unsigned long long h = so - 8ull * g.T;
                    store_bytes(out + 8ull * x.s, &h, 8);
                }
            }
            ox.seed_off[x.s] = so;
        }
        if (threadIdx.x == 0 && wg_last) {
            // the last tile ends the stream: if it fits, every tile fits
            const unsigned long long sz = fits ? P0 + gtot : 0ull;
            ox.meta[0] = sz;
            if (size_out)
                *size_out = sz;
            chain_finished(ws, nchains);
        }
        return;
    }

    if constexpr (Mode == kSumStaged) {
        uint8_t* slot = area + (8 + sizeof(StageRec)) * R + kStageSlot * sidx;
        const uint32_t nz = (total + 64 + 15) / 16;
        for (uint32_t i = lane; i < nz; i += 64)
            reinterpret_cast<uint4*>(obuf)[i] = make_uint4(0, 0, 0, 0);
        encode_blocks(obuf, excl, w, nj, s, s2, m);
        // whole 16-byte chunks: the slot is the tile's own (total <= kStageSlot, a multiple of 16)
        for (uint32_t i = lane; i < (total + 15) / 16; i += 64)
            reinterpret_cast<uint4*>(slot)[i] = reinterpret_cast<const uint4*>(obuf)[i];
        if (has)
            index_view(g, oindex).widths[x.g0 + lane] = (uint8_t) w;
        const uint32_t e16 = __builtin_amdgcn_readlane(excl, 16), e32 = __builtin_amdgcn_readlane(excl, 32),
                       e48 = __builtin_amdgcn_readlane(excl, 48);
        if (lane == 0) {
            StageRec rec;
            rec.total = total;
            rec.e16 = (uint16_t) e16;
            rec.e32 = (uint16_t) e32;
            rec.e48 = (uint16_t) e48;
            rec.pad = 0;
            rec.seed = seed;
            reinterpret_cast<StageRec*>(area + 8 * R)[sidx] = rec;
        }
        return;
    }

    // ---- encode into the LDS buffer and store
    const uint64_t hdr = 8ull * g.T + 4ull * (x.s + 1);
    const uint32_t nz = (total + 64 + 15) / 16;
    for (uint32_t i = lane; i < nz; i += 64)
        reinterpret_cast<uint4*>(obuf)[i] = make_uint4(0, 0, 0, 0);
    encode_blocks(obuf, excl, w, nj, s, s2, m);
    // the tile's stream offset: after its encoding, so predecessors had longer to publish
    const unsigned long long ex = lookback(status, t, 0, total, 0, ws, true);
    if (hdr + ex + total <= out_cap)
        store_wave(obuf, out + hdr + ex, total);
    const uint64_t P = hdr + ex;
    const bool fits = P + total <= out_cap;
    if (!fits && lane == 0)
        raise_error(ws, ZK_ERR_NOSPACE);

    // ---- output index, seed and chunk header
    IndexView ox = index_view(g, oindex);
    if (has)
        ox.widths[x.g0 + lane] = (uint8_t) w;
    if ((lane & 15) == 0 && lane / 16 < x.ngrp)
        ox.group_off[x.grp0 + lane / 16] = P + excl;
    if (lane == 0) {
        if (x.lt == 0) {
            const uint64_t so = P - 4;
            if (so + 4 <= out_cap) {
                store_bytes(out + so, &seed, 4);
                if (x.s < g.T) {
                    const unsigned long long h = so - 8ull * g.T;
                    store_bytes(out + 8ull * x.s, &h, 8);
                }
            }
            ox.seed_off[x.s] = so;
        }
        if (t == tl.ntiles - 1) {
            // the last tile ends the stream: if it fits, every tile fits
            const unsigned long long sz = fits ? P + total : 0ull;
            ox.meta[0] = sz;
            if (size_out)
                *size_out = sz;
            chain_finished(ws, nchains);
        }
    }
}

// ---------------------------------------------------------------- decompress
//
// One pass, no wait between tiles: the index holds the quantized value before
// every tile (its carry).  Lane j decodes block j of the wave's tile (the sum's
// loaders and decoders, one operand), takes the running sums of the deltas in
// the lane, places the blocks with one scan of the block sums across the wave,
// dequantizes, and stores the values through the wave's LDS buffer with 16-byte
// stores.  Arithmetic: prefix sums of the deltas in int32 from the carry,
// x' = (float) q * eb (ZCCL/src/ZCCLd_float.c:588-628).
//
// Compress has a tile's carry in a register and a sum adds its operands'; a
// foreign stream's parse derives them: every tile's sum of deltas, scanned per
// segment from its seed (kCarrySums below, then k_lane_carry_scan).  Decoding
// every stream once more for those sums on each decompress, in two more
// launches, took half the call: without them 38.9 -> 21.9 us for 2^24 values
// (4.0 TB/s of stream and values) and 23.8 -> 11.4 us for 16 411.

// The segment's seed (0 with an error when its offset is past the stream).
__device__ __forceinline__ uint32_t segment_seed(const Geom& g, const uint8_t* bytes, const uint8_t* index,
    uint32_t s, WsHeader* ws)
{
    const IndexView iv = index_view(g, index);
    const uint64_t so = iv.seed_off[s], size = iv.meta[0];
    if (so + 4 <= size)
        return load_u32_bytes(bytes + so);
    raise_error(ws, ZK_ERR_OVERRUN);
    return 0;
}

// Launch tile tg of a decompress in the lane layout: one stream
// (DecompressArgs), or a batch (uniform: shared geometry and bound, per-job
// pointers; mixed: per-job descriptors).
struct DecJob {
    Geom g;
    Tiling tl;
    float eb;
    const uint8_t* bytes;
    const uint8_t* index;
    float* out;
    uint32_t t;         // tile inside the job
    uint64_t tile0;     // the job's first launch tile
};

__device__ __forceinline__ bool dec_job(const DecompressArgs& a, uint64_t tg, DecJob& d)
{
    if (tg >= a.job.tl.ntiles)
        return false;
    d.g = a.job.g;
    d.tl = a.job.tl;
    d.eb = a.job.p.eb;
    d.bytes = a.job.io.in[0].bytes;
    d.index = a.job.io.in[0].index;
    d.out = a.job.io.out;
    d.t = (uint32_t) tg;
    d.tile0 = 0;
    return true;
}

__device__ __forceinline__ bool dec_job(const BatchArgs& b, uint64_t tg, DecJob& d)
{
    if (tg >= b.total_tiles)
        return false;
    if (b.uniform) {
        const uint32_t j = __builtin_amdgcn_readfirstlane((uint32_t) (tg / b.tl.ntiles));
        const DecompressIO* io = (const DecompressIO*) b.jobs + j;
        d.g = b.g;
        d.tl = b.tl;
        d.eb = b.p.eb;
        d.bytes = ldc(&io->in[0].bytes);
        d.index = ldc(&io->in[0].index);
        d.out = ldc(&io->out);
        d.tile0 = (uint64_t) j * b.tl.ntiles;
    } else {
        uint32_t lo = 0, hi = b.njobs;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (ldc(&b.job_tile0[mid]) <= tg)
                lo = mid;
            else
                hi = mid;
        }
        const uint32_t j = __builtin_amdgcn_readfirstlane(lo);
        const DecompressJob* job = (const DecompressJob*) b.jobs + j;
        d.g = job->g;
        d.tl = job->tl;
        d.eb = ldc(&job->p.eb);
        d.bytes = ldc(&job->io.in[0].bytes);
        d.index = ldc(&job->io.in[0].index);
        d.out = ldc(&job->io.out);
        d.tile0 = ldc(&b.job_tile0[j]);
    }
    d.t = __builtin_amdgcn_readfirstlane((uint32_t) (tg - d.tile0));
    return true;
}

// One tile of a decompress pass as it moves through the pipeline: its launch
// index, the lane's width byte and the tile's offset and stream size from the
// index (job, geometry and tile are derived again where needed, with scalar
// work, so that three tiles in flight hold few registers); then the lane's
// block located in the tile bytes, and the bytes staged.
struct DecPre {
    bool ok;
    uint64_t idx;
    uint64_t goff, size;
    uint32_t wq;
    uint32_t carry;    // kValues: the tile's carry
};

struct DecLoc {
    View v;
    uint32_t w, o, tot, nj;
    bool has, skip, half;
};

// What a run over the tiles writes: their values, or (single streams) their
// sums of deltas in the place of the index carries.
enum DecMode : int { kValues, kCarrySums };

// Issue the index reads of launch tile tg.
template <int Mode, typename Args>
__device__ __forceinline__ DecPre dec_prefetch(const Args& a, uint64_t tg)
{
    DecPre p;
    DecJob d;
    p.ok = dec_job(a, tg, d);
    if (!p.ok)
        return p;
    const Geom& g = d.g;
    const Tile x = tile_of(g, d.tl, d.t);
    p.idx = tg;
    const IndexView iv = index_view(g, d.index);
    p.goff = iv.group_off[x.grp0];
    p.size = iv.meta[0];
    const uint32_t lane = threadIdx.x & 63;
    p.wq = lane < x.nblk ? (uint32_t) iv.widths[x.g0 + lane] : 0u;
    p.carry = Mode == kValues ? iv.carry[d.t] : 0u;
    return p;
}

// Locate the lane's block of tile p (one scan of the block sizes) and stage
// the tile's bytes into LDS half `half` of the wave buffer, if they fit there.
template <typename Args>
__device__ __forceinline__ DecLoc dec_locate(const Args& a, const DecPre& p, uint32_t* obuf, uint32_t half,
    bool& bad_width)
{
    DecJob d;
    dec_job(a, p.idx, d);
    const Geom& g = d.g;
    const Tile x = tile_of(g, d.tl, d.t);
    DecLoc c;
    const uint32_t lane = threadIdx.x & 63;
    c.has = lane < x.nblk;
    c.nj = c.has ? min(tile_block_len(g, x, lane), L) : 0u;
    c.w = p.wq;
    if (c.w > 32) {
        bad_width = true;
        c.w = 0;
    }
    const uint32_t bs = c.has ? (c.nj == L ? full_block_bytes(c.w) : lane_block_bytes(c.w, c.nj)) : 0u;
    const uint32_t binc = wave_scan_dpp(bs);
    const uint32_t tot0 = __builtin_amdgcn_readlane(binc, 63);
    // (the same in every lane: scalar, so that what depends on them branches)
    // (a tile without blocks starts right behind its segment's seed, so this is
    // the seed's check too; size 0: an index that holds no stream)
    const uint64_t goff = uniform64(p.goff), size = uniform64(p.size);
    c.skip = !size || goff > size || tot0 > size - goff;
    const uint8_t* base = d.bytes + goff;
    const uint32_t delta = (uint32_t) ((uintptr_t) base & 3u);
    const uint64_t vlen = c.skip ? 0ull : align_up(delta + (size - goff), 4);
    c.v = make_view(base - delta, vlen);
    c.o = delta + binc - bs;
    c.tot = tot0 + delta;
    c.half = !c.skip && staged_len(c.tot) <= kStageCap;
    if (c.half)
        stage_bytes(c.v, c.tot, obuf + half * (kStageHalf / 4));
    return c;
}

// Store the wave's blocks of values (lane l: v[0..nj), at base + 36 l; the
// lanes below nblk hold one, all whole but perhaps the last) so that every
// store instruction writes contiguous, 16-byte aligned chunks.  The blocks
// start D dwords past the 16-byte grid; chunk c of the wave covers dwords
// [4c - D, 4c - D + 4) from base.  A quarter of the wave (16 blocks, 144
// chunks) at a time: its lanes write their values to LDS (ob) at their
// offsets in the quarter's chunks, the lane before the quarter its last D
// values, and the wave stores the chunks with streaming (non-temporal)
// stores.  Lane 0's first chunk is partly the previous tile's and the last
// whole block's last D values start the next tile's (both by dword stores),
// and a segment's short last block goes value by value.  (Unaligned HBM
// writes, and 16-byte stores strided 144 bytes across the lanes, both ran at
// under half the rate of aligned contiguous ones.)
__device__ __forceinline__ void store_blocks(float* base, const float (&v)[L], uint32_t nj, uint32_t nblk,
    uint32_t* ob)
{
    typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));
    const uint32_t lane = threadIdx.x & 63;
    const bool full = lane < nblk && nj == L;
    const unsigned long long fm = __ballot(full);
    const uint32_t nfull = (uint32_t) __popcll(fm);  // whole blocks: a prefix of the lanes
    const bool next_full = lane < 63 && ((fm >> (lane + 1)) & 1ull);
    const uint32_t D = __builtin_amdgcn_readfirstlane((uint32_t) (((uintptr_t) base >> 2) & 3u));
    float* a0 = base - D;  // 16-byte aligned
    const uint32_t nch = 9 * nfull;
    float* of = reinterpret_cast<float*>(ob);
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        const uint32_t c0 = 144 * q;
        if (c0 >= nch)
            break;
        const uint32_t c1 = min(c0 + 144, nch);
        if (full && (lane >> 4) == q) {
            const uint32_t at = D + L * (lane & 15);
#pragma unroll
            for (uint32_t j = 0; j < L; j++)
                if (j < L - 3 || at + j < 576)
                    of[at + j] = v[j];
        }
        if (full && q > 0 && lane == 16 * q - 1) {
#pragma unroll
            for (uint32_t j = L - 3; j < L; j++)
                if (j >= L - D)
                    of[j - (L - D)] = v[j];
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (uint32_t c = c0 + lane; c < c1; c += 64) {
            const uint4 x = reinterpret_cast<const uint4*>(ob)[c - c0];
            float* g = a0 + 4 * c;
            if (c == 0 && D) {
                if (D <= 1)
                    g[1] = __uint_as_float(x.y);
                if (D <= 2)
                    g[2] = __uint_as_float(x.z);
                g[3] = __uint_as_float(x.w);
            } else {
                const u32x4v y = {x.x, x.y, x.z, x.w};
                __builtin_nontemporal_store(y, reinterpret_cast<u32x4v*>(g));
            }
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    float* p = base + lane * L;
    if (full && D && !next_full) {
#pragma unroll
        for (uint32_t m = L - 3; m < L; m++)
            if (m >= L - D)
                p[m] = v[m];
    }
    if (lane < nblk && !full) {
#pragma unroll
        for (uint32_t j = 0; j < L; j++)
            if (j < nj)
                p[j] = v[j];
    }
}

// A run over launch tiles first, first + stride, ... of one wave.  Per step,
// tile i is decoded while tile i+1's bytes move into the other LDS half and
// tile i+2's index entries are on their way (a tile too large for a half is
// staged alone).  The lane decoders are the sum's.
template <int Mode, typename Args>
__device__ __forceinline__ void dec_run(const Args& a, WsHeader* ws, uint64_t first, uint64_t stride, uint32_t* obuf)
{
    const uint32_t lane = threadIdx.x & 63;
    bool bad_width = false, bad_byte = false, bad_over = false;
    DecPre pc = dec_prefetch<Mode>(a, first);
    if (!pc.ok)
        return;
    __builtin_amdgcn_s_waitcnt(0);
    DecLoc cc = dec_locate(a, pc, obuf, 0, bad_width);
    DecPre pn = dec_prefetch<Mode>(a, first + stride);
    for (uint32_t half = 0;; half ^= 1u) {
        const uint32_t* st = obuf + (cc.half ? half * (kStageHalf / 4) : 0u);
        if (!cc.half && !cc.skip)  // (the other half's tile is decoded)
            stage_bytes(cc.v, cc.tot, obuf);
        __builtin_amdgcn_s_waitcnt(0);  // tile i's bytes in LDS, tile i+1's index entries in registers
        DecLoc cn;
        DecPre pnn;
        pnn.ok = false;
        auto next = [&] {
            if (pn.ok) {
                cn = dec_locate(a, pn, obuf, half ^ 1u, bad_width);
                pnn = dec_prefetch<Mode>(a, pn.idx + stride);
            }
        };
        // f(j, magnitude, +1 or -1) over the lane's values (zeros for a lane
        // without a block), f_high(j, magnitude, sign word) over those of a block
        // from width 16, and next() where it overlaps best
        auto values = [&](auto f, auto f_high) {
            if (!cc.skip) {
                bad_byte |= cc.has & (((const uint8_t*) st)[cc.o] != cc.w);
                const bool wide = __any(cc.w >= 8);
                const uint32_t w = cc.w < 16 ? cc.w : 0u;
                Block q;
                read_block(st, cc.o, w, cc.nj, wide, q);
                __builtin_amdgcn_sched_barrier(0);
                const bool high = wide && __any(cc.w >= 16);
                if (cc.half && !high)
                    next();
                __builtin_amdgcn_sched_barrier(0);
                each_value(q, w, wide, f);
                if (high)
                    each_high_lane(st, cc.o, cc.w, cc.nj, cc.w >= 16, f_high);
                return cc.half && !high;
            }
            return false;
        };
        bad_over |= cc.skip;
        if constexpr (Mode == kCarrySums) {
            // the block's sum only, of its nj values
            uint32_t b = 0;
            const bool ahead = values(
                [&](uint32_t j, uint32_t m, uint32_t sign) { b = mad_i24(j < cc.nj ? m : 0u, sign, b); },
                [&](uint32_t j, uint32_t m, uint32_t sw) { b += j < cc.nj ? signed_of(m, sw) : 0u; });
            if (!ahead)
                next();
            const uint32_t inc = wave_scan_dpp(b);
            if (lane == 63) {
                DecJob d;
                dec_job(a, pc.idx, d);
                index_view(d.g, d.index).carry[d.t] = inc;
            }
        } else {
            // the deltas, then their running sums (past a short block's
            // values: whatever follows it, never stored)
            uint32_t acc[L];
#pragma unroll
            for (uint32_t j = 0; j < L; j++)
                acc[j] = 0;
            const bool ahead =
                values([&](uint32_t j, uint32_t m, uint32_t sign) { acc[j] = mad_i24(m, sign, 0u); },
                    [&](uint32_t j, uint32_t m, uint32_t sw) { acc[j] = stay(signed_of(m, sw)); });
            if (!ahead)
                next();
#pragma unroll
            for (uint32_t j = 1; j < L; j++)
                acc[j] += acc[j - 1];
            const uint32_t run = acc[L - 1];
            DecJob d;
            dec_job(a, pc.idx, d);
            const Tile x = tile_of(d.g, d.tl, d.t);
            const uint32_t carry = pc.carry + wave_scan_dpp(run) - run;
            const float eb = d.eb;
            float vals[L];
#pragma unroll
            for (uint32_t jj = 0; jj < L; jj++)
                vals[jj] = dequant(carry + acc[jj], eb);
            // (this tile's LDS half is free: its bytes are in registers; the
            // other half may hold the next tile's)
            store_blocks(d.out + x.e0, vals, cc.nj, x.nblk, obuf + half * (kStageHalf / 4));
            if (lane == 0 && x.lt == 0)
                d.out[x.seg_a] = dequant(pc.carry, eb);  // the segment's first value, its seed
        }
        if (!pn.ok)
            break;
        pc = pn;
        cc = cn;
        pn = pnn;
    }
    if (__any(bad_width) && lane == 0)
        raise_error(ws, ZK_ERR_WIDTH);
    if (__any(bad_byte) && lane == 0)
        raise_error(ws, ZK_ERR_MISMATCH);
    if (__any(bad_over) && lane == 0)
        raise_error(ws, ZK_ERR_OVERRUN);
}

// Scan of one segment's tile sums into carries (in place): the seed plus the
// sums of the segment's earlier tiles, mod 2^32.  One workgroup.
template <uint32_t Threads>
__device__ __forceinline__ void carry_scan(const Geom& g, const uint8_t* bytes, const uint8_t* index, uint32_t s,
    WsHeader* ws)
{
    __shared__ uint32_t s_w[Threads / 64];
    __shared__ uint32_t s_seed;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint32_t cnt = s < g.T ? g.cT : g.cR;
    if (tid == 0)
        s_seed = segment_seed(g, bytes, index, s, ws);
    uint32_t* p = index_view(g, index).carry + (s < g.T ? s * g.cT : g.T * g.cT);
    const uint32_t per = (cnt + Threads - 1) / Threads;
    const uint32_t a = min(tid * per, cnt), b = min(a + per, cnt);
    uint32_t run = 0;
    for (uint32_t i = a; i < b; i++)
        run += p[i];
    const uint32_t inc = wave_scan_dpp(run);
    if (lane == 63)
        s_w[wv] = inc;
    __syncthreads();
    uint32_t before = s_seed + inc - run;
    for (uint32_t i = 0; i < wv; i++)
        before += s_w[i];
    for (uint32_t i = a; i < b; i++) {
        const uint32_t v = p[i];
        p[i] = before;
        before += v;
    }
}

// ---------------------------------------------------------------- compress
//
// A workgroup of four waves owns a tile of 256 blocks (make_lane_wg_tiling),
// wave w blocks 64w .. 64w + 63, one block per lane.  Each wave stages its
// blocks' values into its LDS buffer (16-byte direct-to-LDS loads through a
// range-checked view of them; reads past it return zeros) and lane 0 loads the
// value before them; each lane reads its block's 36 values, quantizes them
// (FP32 products rounded toward zero, below; FP64 where a wave's values reach
// further), takes the last quantized value of the lane below, the deltas, the
// sign words, the magnitudes and the width, and the wave scans the block
// sizes.  The workgroup adds its waves' sizes, publishes the tile's
// aggregate, encodes every block into the wave buffers (the lane encoders of
// the sum), resolves the tile's stream offset by the decoupled lookback
// (one chain per stream, as the slot kernel), and each wave stores its bytes.
// Arithmetic: ZCCL/src/ZCCL_float.c:563,577-606 (quantize, delta, width),
// ZCCL/src/ZCCL_TypeManager.c:12-91, 824-848 (packing, signs).

// Quantize by FP32: the reciprocal of the bound is an FP32 number (inverse_bound;
// the kernels' double holds no more, and turning it back loses nothing), its
// product with x is exact in 48 bits, and FP32 rounding toward zero keeps its integer part below 2^24; a second product with 2^-149,
// rounded toward zero too, drops the fraction and leaves the integer as a
// denormal's bits, so deltas are FP32 differences (exact below 2^23).  Two
// 2-cycle instructions and one to turn -0 into +0 in place of an FP64 product
// with its conversions and range checks (22 cycles).  `far` collects the
// largest magnitude, or NaN: the wave takes the FP64 form unless it is below
// kQuantSmall.  The products are volatile so that none moves above
// round_toward_zero(); nothing else in the kernel rounds FP32.
constexpr float kQuantSmall = 8388608.0f;  // 2^23

__device__ __forceinline__ void round_toward_zero()
{
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 3");
}

__device__ __forceinline__ void quant_small(float x, float inv, float& q, float& far)
{
    float p, t;
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(p) : "v"(x), "v"(inv));
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(t) : "s"(1u), "v"(p));
    q = t + 0.0f;
    asm("v_maximum3_f32 %0, |%1|, %2, %2" : "=v"(far) : "v"(p), "v"(far));
}

// v of the lane below; lane 0: first.
__device__ __forceinline__ float from_lane_below(float v, float first)
{
    return as_f((uint32_t) __builtin_amdgcn_update_dpp((int) as_u(first), (int) as_u(v), 0x138, 0xF, 0xF, false));  // wave_shr:1
}

constexpr uint32_t kCompBuf = 9728;  // a wave's values (2304 floats) or a worst-case 64-block encode + reach
static_assert(kCompBuf >= kLaneTileBlocks * kWorstBlock + 64 && kCompBuf >= (kLaneTileBlocks - 1) * kWorstBlock + kReach &&
        kCompBuf >= 4 * kLaneTileBlocks * L,
    "a compress wave buffer holds the staged values and the worst-case encode");
static_assert(kCompBuf % 16 == 0, "compress wave buffers stay 16-byte aligned");

// Tiles a workgroup takes with one ticket.  Tickets are adds to one address, 12
// ns each: the 1820 of a 2^24-value stream took 22 us of the kernel's 48; two
// tiles a ticket: 37 us (four: 35, but 131 us against 110 for the 16 streams that 4
// ranks of a staged allreduce compress, whose tiles then end together).  Up to
// kCompFew tiles, one for each compute unit, a tile has a workgroup of its own (16
// tiles: 9.4 us against 10.0; 336 tiles: 14.8 against 13.0).
constexpr uint32_t kCompPair = 2, kCompFew = 256;

struct CompShared {
    uint32_t wtot[kLaneWaves];
    unsigned long long ex;
};

__device__ __forceinline__ void compress_tile_lane(const Geom& g, const Tiling& tl, double inv, const float* xin,
    uint8_t* out, uint64_t out_cap, uint8_t* oindex, unsigned long long* size_out, uint64_t t,
    unsigned long long* status, WsHeader* ws, uint32_t nchains, uint32_t* obuf, CompShared& sh, bool live)
{
    round_toward_zero();
    const uint32_t lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) % kLaneWaves;  // wave of the tile
    const Tile x = tile_of(g, tl, (uint32_t) t);
    const uint32_t jb = kLaneTileBlocks * wv + lane;  // block of the tile
    const bool has = live & (jb < x.nblk);
    const uint32_t nj = has ? min(tile_block_len(g, x, jb), L) : 0u;
    // the wave's values
    const uint32_t nbw = (live & (x.nblk > kLaneTileBlocks * wv)) ? min(x.nblk - kLaneTileBlocks * wv, kLaneTileBlocks) : 0u;
    const uint32_t nvals = nbw ? (nbw - 1) * L + min(tile_block_len(g, x, kLaneTileBlocks * wv + nbw - 1), L) : 0u;
    const uint32_t v0 = x.e0 + kLaneTileBlocks * L * wv;  // input index of the wave's first value
    float xb = 0.0f;                                      // lane 0: the value before it
    if (nbw) {
        // (a view of the wave's values alone: its range check ends them with
        // zeros)
        const View vx = make_view((const uint8_t*) (xin + v0), 4ull * nvals);
#pragma unroll
        for (uint32_t run = 0; run < kLaneTileBlocks * L / 256; run++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vx,
                (__attribute__((address_space(3))) void*) ((uint8_t*) obuf + run * 1024), 16, 1024 * run + 16 * lane, 0,
                0, 0);
        if (lane == 0)
            xb = xin[v0 - 1];
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // quantize, deltas, signs and magnitudes (values past nj are zero)
    const float4* xv = reinterpret_cast<const float4*>(obuf) + lane * (L / 4);
    uint32_t m[L];
    uint32_t s = 0, s2 = 0, mx = 0;
    uint32_t before = 0;  // lane 0: the quantized value before the wave's first
    {
        const float finv = (float) inv;
        float q[L];
        float far = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < L / 4; i++) {
            const float4 v = xv[i];
            quant_small(v.x, finv, q[4 * i], far);
            quant_small(v.y, finv, q[4 * i + 1], far);
            quant_small(v.z, finv, q[4 * i + 2], far);
            quant_small(v.w, finv, q[4 * i + 3], far);
        }
        float qb;
        quant_small(xb, finv, qb, far);
        if (!__any(!(far < kQuantSmall))) {
            before = signed_of(as_u(qb) & 0x7FFFFFFFu, as_u(qb));
            float prev = from_lane_below(q[L - 1], qb);
#pragma unroll
            for (uint32_t j = 0; j < L; j++) {
                m[j] = as_u(q[j] - prev);
                prev = q[j];
            }
            if (__any(nj < L)) {
#pragma unroll
                for (uint32_t j = 0; j < L; j++)
                    if (j >= nj)
                        m[j] = 0;
            }
#pragma unroll
            for (uint32_t j = 0; j < L; j++) {
                if (j < 32)
                    s = __builtin_amdgcn_alignbit(s, m[j], 31);  // (s << 1) | sign of value j
                else
                    s2 = __builtin_amdgcn_alignbit(s2, m[j], 31);
                m[j] &= 0x7FFFFFFFu;
            }
        } else {
            // some value of the wave is 2^23 bounds from zero, or not a number
            before = (uint32_t) quant(xb, inv);
            uint32_t prev =
                as_u(from_lane_below(as_f((uint32_t) quant(reinterpret_cast<const float*>(xv)[L - 1], inv)), as_f(before)));
#pragma unroll
            for (uint32_t j = 0; j < L; j++) {
                const uint32_t qj = (uint32_t) quant(reinterpret_cast<const float*>(xv)[j], inv);
                const uint32_t d = j < nj ? qj - prev : 0u;
                prev = qj;
                if (j < 32)
                    s = __builtin_amdgcn_alignbit(s, d, 31);
                else
                    s2 = __builtin_amdgcn_alignbit(s2, d, 31);
                m[j] = mag(d);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < L; j++)
            mx = max(mx, m[j]);
    }
    const uint32_t w = has ? dwidth(mx) : 0u;
    const uint32_t bs = has ? (nj == L ? full_block_bytes(w) : lane_block_bytes(w, nj)) : 0u;
    const uint32_t incl = wave_scan_dpp(bs);
    const uint32_t excl = incl - bs;
    const uint32_t wtot = __builtin_amdgcn_readlane(incl, 63);
    if (lane == 0)
        sh.wtot[wv] = wtot;
    __syncthreads();  // every wave's values are read: the buffers are free for the encode
    uint32_t woff = 0, total = 0;
#pragma unroll
    for (uint32_t i = 0; i < kLaneWaves; i++) {
        const uint32_t v = sh.wtot[i];
        woff += i < wv ? v : 0u;
        total += v;
    }
    if (live & ((wv | lane) == 0))
        lookback_publish(status, t, 0, total, 0);  // successors see the aggregate now
    const uint32_t nz = (wtot + 64 + 15) / 16;
    for (uint32_t i = lane; i < nz; i += 64)
        reinterpret_cast<uint4*>(obuf)[i] = make_uint4(0, 0, 0, 0);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    encode_blocks(obuf, excl, w, nj, s, s2, m);
    if (live & (wv == 0)) {
        const unsigned long long ex = lookback(status, t, 0, total, 0, ws, true);
        if (lane == 0)
            sh.ex = ex;
    }
    __syncthreads();
    if (!live)
        return;
    const uint64_t P = 8ull * g.T + 4ull * (x.s + 1) + sh.ex;
    const bool fits = P + total <= out_cap;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (fits)
        store_wave(obuf, out + P + woff, wtot);
    else if ((wv | lane) == 0)
        raise_error(ws, ZK_ERR_NOSPACE);
    IndexView ox = index_view(g, oindex);
    const uint32_t ct = (x.s < g.T ? x.s * g.cT : g.T * g.cT) + kLaneWaves * x.lt + wv;  // the wave's lane tile
    if (lane == 0 && nbw)
        ox.carry[ct] = before;
    if (has)
        ox.widths[x.g0 + jb] = (uint8_t) w;
    if (has && (jb % g.IG) == 0)
        ox.group_off[x.grp0 + jb / g.IG] = P + woff + excl;
    if ((wv | lane) == 0) {
        if (x.nblk == 0 && x.ngrp)
            ox.group_off[x.grp0] = P;  // a segment of its seed alone keeps one group entry
        if (x.lt == 0) {
            const uint32_t seed = (uint32_t) quant(xin[x.seg_a], inv);
            if (x.nblk == 0)
                ox.carry[ct] = seed;
            const uint64_t so = P - 4;
            if (so + 4 <= out_cap) {
                store_bytes(out + so, &seed, 4);
                if (x.s < g.T) {
                    const unsigned long long h = so - 8ull * g.T;
                    store_bytes(out + 8ull * x.s, &h, 8);
                }
            }
            ox.seed_off[x.s] = so;
        }
        if (t == tl.ntiles - 1) {
            // the last tile ends the stream: if it fits, every tile fits
            const unsigned long long sz = fits ? P + total : 0ull;
            ox.meta[0] = sz;
            if (size_out)
                *size_out = sz;
            chain_finished(ws, nchains);
        }
    }
}

}  // namespace

// Waves (tiles) that share a ticket of a sum: tickets are adds to one address,
// 12 ns each, so beyond kSumFew tiles, one for each of the chip's 1024 SIMDs, eight
// waves share one; below, smaller workgroups start sooner and spread over more
// compute units.  us by four / eight waves: 343 tiles of 16 operands 29.6 / 36.5, 881
// 32.1 / 39.7, 912 of 8 23.9 / 28.2; 1824 34.2 / 31.3, 2168 (mixed batch) 38.5 / 38.7,
// 3727 (mixed, 16 operands) 69.0 / 64.5, 8656 (mixed, 4) 76.1 / 70.7, 7296 of 8 87.5 /
// 80.1.
constexpr uint32_t kSumMany = 8, kSumFew = 1024;

// One fused sum (kernel arguments hold its geometry and pointers).
template <uint32_t W>
__global__ void __launch_bounds__(64 * W, 4) k_homsum_lane(HomsumArgs a)
{
    uint64_t t0;
    unsigned long long* status;
    if (!launch_status(a.ws, a.job.tl.ntiles, t0, status, W, &sum_shared<W>().ticket))
        return;
    const uint32_t wv = threadIdx.x >> 6;
    const uint64_t t = t0 + wv;
    if (t >= a.job.tl.ntiles)
        return;
    const ArgIO src{a.job.io};
    homsum_tile_lane<kSumWave>(a.job.g, a.job.tl, a.job.p.k, src, a.job.io.out, a.job.io.out_cap, a.job.io.index,
        a.job.io.size_out, t, status, a.ws, 1, zk_lds + wv * (kOutBuf / 4));
}

// Uniform batch: shared geometry, per-job pointers in device memory; tiles of
// the jobs interleave (tile b is tile b / njobs of job b % njobs).
template <uint32_t W>
__global__ void __launch_bounds__(64 * W, 4) k_homsum_lane_batch(BatchArgs b)
{
    uint64_t t0;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, t0, status, W, &sum_shared<W>().ticket))
        return;
    const uint32_t wv = threadIdx.x >> 6;
    const uint64_t tg = t0 + wv;
    if (tg >= b.total_tiles)
        return;
    uint32_t jidx, t;
    if (b.interleave) {
        jidx = (uint32_t) tg % b.njobs;
        t = (uint32_t) tg / b.njobs;
    } else {
        jidx = 0;
        t = (uint32_t) tg;
    }
    jidx = __builtin_amdgcn_readfirstlane(jidx);
    t = __builtin_amdgcn_readfirstlane(t);
    const HomsumIO* io = (const HomsumIO*) b.jobs + jidx;
    const SumIO src{io};
    homsum_tile_lane<kSumWave>(b.g, b.tl, b.p.k, src, ldc(&io->out), ldc(&io->out_cap), ldc(&io->index),
        ldc(&io->size_out), t, status + (uint64_t) jidx * b.tl.ntiles * kStatusStride, b.ws, b.total_chains,
        zk_lds + wv * (kOutBuf / 4));
}

// Mixed batch: every job carries its own geometry; job j owns launch tiles
// [job_tile0[j], job_tile0[j+1]).
template <uint32_t W>
__global__ void __launch_bounds__(64 * W, 4) k_homsum_lane_mixed(BatchArgs b)
{
    uint64_t t0;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, t0, status, W, &sum_shared<W>().ticket))
        return;
    const uint32_t wv = threadIdx.x >> 6;
    const uint64_t tg = t0 + wv;
    if (tg >= b.total_tiles)
        return;
    uint32_t lo = 0, hi = b.njobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (ldc(&b.job_tile0[mid]) <= tg)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t jidx = __builtin_amdgcn_readfirstlane(lo);
    const uint64_t tile0 = ldc(&b.job_tile0[jidx]);
    const uint32_t t = __builtin_amdgcn_readfirstlane((uint32_t) (tg - tile0));
    const HomsumJob* job = (const HomsumJob*) b.jobs + jidx;
    const Geom g = job->g;
    const Tiling tl = job->tl;
    const SumIO src{&job->io};
    homsum_tile_lane<kSumWave>(g, tl, ldc(&job->p.k), src, ldc(&job->io.out), ldc(&job->io.out_cap), ldc(&job->io.index),
        ldc(&job->io.size_out), t, status + tile0 * kStatusStride, b.ws, b.total_chains, zk_lds + wv * (kOutBuf / 4));
}

// A persistent grid, wave w of workgroup b starting at launch tile 4b + w and
// striding by the grid's waves.
template <int Mode, typename Args>
__device__ __forceinline__ void dec_grid(const Args& a, WsHeader* ws)
{
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    dec_run<Mode>(a, ws, (uint64_t) blockIdx.x * kLaneWaves + wv, (uint64_t) gridDim.x * kLaneWaves,
        zk_lds + wv * (kOutBuf / 4));
}

__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_decompress_lane(DecompressArgs a)
{
    dec_grid<kValues>(a, a.ws);
}
__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_decompress_lane_batch(BatchArgs b)
{
    dec_grid<kValues>(b, b.ws);
}

// Carries of a parsed stream (none of a corrupt one, whose size is 0).
__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_lane_carry_sums(DecompressArgs a)
{
    if (index_view(a.job.g, a.job.io.in[0].index).meta[0])
        dec_grid<kCarrySums>(a, a.ws);
}
// (one wave to a segment of up to kCarryShort tiles: 4000000 values in 1000 segments
// of 2 tiles are parsed in 55 us, 62 with sixteen waves to each)
constexpr uint32_t kCarryShort = 256;
template <uint32_t Threads>
__global__ void __launch_bounds__(Threads) k_lane_carry_scan(DecompressArgs a)
{
    if (index_view(a.job.g, a.job.io.in[0].index).meta[0])
        carry_scan<Threads>(a.job.g, a.job.io.in[0].bytes, a.job.io.in[0].index, blockIdx.x, a.ws);
}

// Compress in the lane layout: one stream, a uniform batch (shared geometry
// and bound, per-job pointers, tiles of the jobs interleaved) or a mixed one.
template <uint32_t N>
__global__ void __launch_bounds__(64 * kLaneWaves * N, 4) k_compress_lane(CompressArgs a)
{
    __shared__ CompShared sh[N];
    const uint32_t part = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * kLaneWaves));
    uint64_t t;
    unsigned long long* status;
    if (!launch_status(a.ws, a.job.tl.ntiles, t, status, N))
        return;
    t += part;
    const bool live = t < a.job.tl.ntiles;
    compress_tile_lane(a.job.g, a.job.tl, a.job.p.inv, a.job.io.x, a.job.io.out, a.job.io.out_cap, a.job.io.index,
        a.job.io.size_out, live ? t : 0, status, a.ws, 1, zk_lds + (threadIdx.x >> 6) * (kCompBuf / 4), sh[part], live);
}

template <uint32_t N>
__global__ void __launch_bounds__(64 * kLaneWaves * N, 4) k_compress_lane_batch(BatchArgs b)
{
    __shared__ CompShared sh[N];
    const uint32_t part = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * kLaneWaves));
    uint64_t tg;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, tg, status, N))
        return;
    tg += part;
    const bool live = tg < b.total_tiles;
    if (!live)
        tg = b.total_tiles - 1;
    uint32_t jidx, t;
    if (b.interleave) {
        jidx = (uint32_t) tg % b.njobs;
        t = (uint32_t) tg / b.njobs;
    } else {
        jidx = 0;
        t = (uint32_t) tg;
    }
    jidx = __builtin_amdgcn_readfirstlane(jidx);
    t = __builtin_amdgcn_readfirstlane(t);
    const CompressIO* io = (const CompressIO*) b.jobs + jidx;
    compress_tile_lane(b.g, b.tl, b.p.inv, ldc(&io->x), ldc(&io->out), ldc(&io->out_cap), ldc(&io->index),
        ldc(&io->size_out), t, status + (uint64_t) jidx * b.tl.ntiles * kStatusStride, b.ws, b.total_chains,
        zk_lds + (threadIdx.x >> 6) * (kCompBuf / 4), sh[part], live);
}

template <uint32_t N>
__global__ void __launch_bounds__(64 * kLaneWaves * N, 4) k_compress_lane_mixed(BatchArgs b)
{
    __shared__ CompShared sh[N];
    const uint32_t part = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * kLaneWaves));
    uint64_t tg;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, tg, status, N))
        return;
    tg += part;
    const bool live = tg < b.total_tiles;
    if (!live)
        tg = b.total_tiles - 1;
    uint32_t lo = 0, hi = b.njobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (ldc(&b.job_tile0[mid]) <= tg)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t jidx = __builtin_amdgcn_readfirstlane(lo);
    const uint64_t tile0 = ldc(&b.job_tile0[jidx]);
    const uint32_t t = __builtin_amdgcn_readfirstlane((uint32_t) (tg - tile0));
    const CompressJob* job = (const CompressJob*) b.jobs + jidx;
    const Geom g = job->g;
    const Tiling tl = job->tl;
    compress_tile_lane(g, tl, ldc(&job->p.inv), ldc(&job->io.x), ldc(&job->io.out), ldc(&job->io.out_cap),
        ldc(&job->io.index), ldc(&job->io.size_out), t, status + tile0 * kStatusStride, b.ws, b.total_chains,
        zk_lds + (threadIdx.x >> 6) * (kCompBuf / 4), sh[part], live);
}

// Single-pass sum with a lookback tile per workgroup (layout 2): the
// workgroup's tile comes from make_lane_wg_tiling, each wave takes one tile
// of the lane tiling inside it.  The wave's lane tile (its index in t_lane),
// or an empty tile past its segment's blocks.
__device__ __forceinline__ Tile wg_wave_tile(const Geom& g, const Tiling& tl, const Tiling& tw, uint32_t t_wg,
    uint32_t wv, uint32_t& t_lane)
{
    const Tile xw = tile_of(g, tw, t_wg);
    const uint32_t base = xw.s < g.T ? xw.s * tl.tilesT : g.T * tl.tilesT;
    const uint32_t seg_tiles = xw.s < g.T ? tl.tilesT : tl.tilesR;
    const uint32_t lt = kLaneWaves * xw.lt + wv;
    t_lane = base + min(lt, seg_tiles - 1);
    Tile x = tile_of(g, tl, t_lane);
    if (lt >= seg_tiles) {
        x.nblk = 0;
        x.ngrp = 0;
        x.lt = lt;
    }
    return x;
}

__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_homsum_lane_wg(HomsumArgs a)
{
    SumShared& sh = sum_shared<kLaneWaves>();
    uint64_t t_wg;
    unsigned long long* status;
    if (!launch_status(a.ws, a.job.tl.ntiles, t_wg, status, 1, &sh.ticket))
        return;
    const uint32_t wv = threadIdx.x >> 6;
    const Tiling tl = make_lane_tiling(a.job.g);
    uint32_t t_lane;
    const Tile x = wg_wave_tile(a.job.g, tl, a.job.tl, (uint32_t) t_wg, wv, t_lane);
    const ArgIO src{a.job.io};
    homsum_tile_lane<kSumWg>(a.job.g, tl, a.job.p.k, src, a.job.io.out, a.job.io.out_cap, a.job.io.index,
        a.job.io.size_out, t_lane, status, a.ws, 1, zk_lds + wv * (kOutBuf / 4), nullptr, 0, 0, t_wg,
        t_wg == a.job.tl.ntiles - 1, &sh.wg, &x);
}

// (four workgroups per CU: at five the workgroup state spills)
__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_homsum_lane_wg_batch(BatchArgs b)
{
    SumShared& sh = sum_shared<kLaneWaves>();
    uint64_t tg;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, tg, status, 1, &sh.ticket))
        return;
    uint32_t jidx, t;
    if (b.interleave) {
        jidx = (uint32_t) tg % b.njobs;
        t = (uint32_t) tg / b.njobs;
    } else {
        jidx = 0;
        t = (uint32_t) tg;
    }
    jidx = __builtin_amdgcn_readfirstlane(jidx);
    t = __builtin_amdgcn_readfirstlane(t);
    const uint32_t wv = threadIdx.x >> 6;
    const Tiling tl = make_lane_tiling(b.g);
    uint32_t t_lane;
    const Tile x = wg_wave_tile(b.g, tl, b.tl, t, wv, t_lane);
    const HomsumIO* io = (const HomsumIO*) b.jobs + jidx;
    const SumIO src{io};
    homsum_tile_lane<kSumWg>(b.g, tl, b.p.k, src, ldc(&io->out), ldc(&io->out_cap), ldc(&io->index),
        ldc(&io->size_out), t_lane, status + (uint64_t) jidx * b.tl.ntiles * kStatusStride, b.ws, b.total_chains,
        zk_lds + wv * (kOutBuf / 4), nullptr, 0, 0, t, t == b.tl.ntiles - 1, &sh.wg, &x);
}

__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_homsum_lane_wg_mixed(BatchArgs b)
{
    SumShared& sh = sum_shared<kLaneWaves>();
    uint64_t tg;
    unsigned long long* status;
    if (!launch_status(b.ws, b.total_tiles, tg, status, 1, &sh.ticket))
        return;
    uint32_t lo = 0, hi = b.njobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (ldc(&b.job_tile0[mid]) <= tg)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t jidx = __builtin_amdgcn_readfirstlane(lo);
    const uint64_t tile0 = ldc(&b.job_tile0[jidx]);
    const uint32_t t = __builtin_amdgcn_readfirstlane((uint32_t) (tg - tile0));
    const HomsumJob* job = (const HomsumJob*) b.jobs + jidx;
    const Geom g = job->g;
    const Tiling tw = job->tl;
    const uint32_t wv = threadIdx.x >> 6;
    const Tiling tl = make_lane_tiling(g);
    uint32_t t_lane;
    const Tile x = wg_wave_tile(g, tl, tw, t, wv, t_lane);
    const SumIO src{&job->io};
    homsum_tile_lane<kSumWg>(g, tl, ldc(&job->p.k), src, ldc(&job->io.out), ldc(&job->io.out_cap),
        ldc(&job->io.index), ldc(&job->io.size_out), t_lane, status + tile0 * kStatusStride, b.ws, b.total_chains,
        zk_lds + wv * (kOutBuf / 4), nullptr, 0, 0, t, t == tw.ntiles - 1, &sh.wg, &x);
}

// ---------------------------------------------------------------- two-pass sum

// The hardware hands workgroup b of a launch to XCD b % 8.  The index this
// returns gives each XCD a contiguous run of workgroups (XCD x: runs of
// about nwg / 8 starting at x * nwg / 8), so tiles that share cache lines at
// their edges, and their index entries, meet in one L2.  A bijection on
// [0, nwg).
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nwg)
{
    const uint32_t q = nwg / 8, rem = nwg % 8, x = b % 8, s = b / 8;
    return x * q + min(x, rem) + s;
}

// Pass one of a single sum: tile t of workgroup-wave t / kLaneWaves, slot t.
__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_homsum_lane_staged(HomsumArgs a, uint8_t* stage)
{
    const uint32_t wv = threadIdx.x >> 6;
    const uint64_t t = (uint64_t) xcd_block(blockIdx.x, gridDim.x) * kLaneWaves + wv;
    if (t >= a.job.tl.ntiles)
        return;
    const ArgIO src{a.job.io};
    homsum_tile_lane<kSumStaged>(a.job.g, a.job.tl, a.job.p.k, src, a.job.io.out, a.job.io.out_cap, a.job.io.index,
        a.job.io.size_out, t, nullptr, a.ws, 1, zk_lds + wv * (kOutBuf / 4), stage, a.job.tl.ntiles, t);
}

// Pass one of a uniform batch: a workgroup takes kLaneWaves consecutive
// tiles of one job (ceil(ntiles / kLaneWaves) workgroups per job, jobs in
// order of the XCD-contiguous index), slot job * ntiles + tile.
__global__ void __launch_bounds__(64 * kLaneWaves, 4) k_homsum_lane_batch_staged(BatchArgs b, uint8_t* stage)
{
    const uint32_t wv = threadIdx.x >> 6;
    const uint32_t wpj = (uint32_t) ceil_div(b.tl.ntiles, kLaneWaves);
    const uint32_t g = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t jidx = __builtin_amdgcn_readfirstlane(g / wpj);
    const uint32_t t = __builtin_amdgcn_readfirstlane((g % wpj) * kLaneWaves + wv);
    if (jidx >= b.njobs || t >= b.tl.ntiles)
        return;
    const HomsumIO* io = (const HomsumIO*) b.jobs + jidx;
    const SumIO src{io};
    homsum_tile_lane<kSumStaged>(b.g, b.tl, b.p.k, src, ldc(&io->out), ldc(&io->out_cap), ldc(&io->index),
        ldc(&io->size_out), t, nullptr, b.ws, 1, zk_lds + wv * (kOutBuf / 4), stage, b.total_tiles,
        (uint64_t) jidx * b.tl.ntiles + t);
}

// Byte j (0..15) of a 16-byte chunk held in registers.
__device__ __forceinline__ uint32_t chunk_byte(const uint4& x, uint32_t j)
{
    const uint32_t w = j < 8 ? (j < 4 ? x.x : x.y) : (j < 12 ? x.z : x.w);
    return (w >> (8 * (j & 3))) & 0xFFu;
}

// Copy n bytes from src (16-byte aligned, a stage slot) to dst, one wave:
// 16-byte stores on dst's 16-byte grid, the partial first and last chunk
// byte by byte from registers, so no byte outside [dst, dst + n) is
// written.  The source is read through a range-checked view, four chunks
// per lane in flight; a partial first chunk reads the slot's first 16 bytes.
__device__ __forceinline__ void copy_wave(uint8_t* dst, const uint8_t* src, uint32_t n)
{
    const uint32_t lane = threadIdx.x & 63;
    const View v = make_view(src, kStageSlot);
    const uintptr_t d0 = (uintptr_t) dst, d1 = d0 + n;
    const uintptr_t c0 = d0 & ~(uintptr_t) 15;
    const uint32_t nch = n ? (uint32_t) ((d1 - c0 + 15) >> 4) : 0u;
    for (uint32_t base = 0; base < nch; base += 256) {
        uint4 x[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            const uint32_t c = base + 64 * u + lane;
            const uintptr_t ca = c0 + 16ull * c;
            x[u] = c < nch ? bl16(v, ca >= d0 ? (uint32_t) (ca - d0) : 0u) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            const uint32_t c = base + 64 * u + lane;
            const uintptr_t ca = c0 + 16ull * c;
            if (c >= nch)
                continue;
            if (ca >= d0 && ca + 16 <= d1) {
                *(uint4*) ca = x[u];
            } else {
                // x[u] holds source bytes from destination byte sb on (byte
                // indices fixed at compile time: a variable one would put
                // the chunks in memory, which the compiler maps to LDS)
                const uintptr_t sb = ca > d0 ? ca : d0, e = ca + 16 < d1 ? ca + 16 : d1;
#pragma unroll
                for (uint32_t i = 0; i < 16; i++)
                    if (sb + i < e)
                        *(uint8_t*) (sb + i) = (uint8_t) chunk_byte(x[u], i);
            }
        }
    }
}

// Stream offset of every tile of one sum (pass two, first kernel): one
// workgroup of 1024 threads per sum; thread i adds the sizes of tiles
// [8i, 8i + 8) of each round of 8192 tiles, then a workgroup scan.  A tile's
// offset counts the stream header, one seed per segment started and the
// sizes of all earlier tiles.
constexpr uint32_t kScanThreads = 1024;
constexpr uint32_t kScanPer = 8;

__device__ __forceinline__ void scan_sum(const Geom& g, const Tiling& tl, const uint8_t* stage, uint64_t R,
    uint64_t sidx0)
{
    __shared__ unsigned long long s_w[kScanThreads / 64];
    __shared__ unsigned long long s_run;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    unsigned long long* pos = (unsigned long long*) stage;
    const StageRec* recs = reinterpret_cast<const StageRec*>(stage + 8 * R);
    if (tid == 0)
        s_run = 0;
    for (uint32_t base = 0; base < tl.ntiles; base += kScanThreads * kScanPer) {
        uint32_t tot[kScanPer];
        uint64_t sum = 0;
#pragma unroll
        for (uint32_t u = 0; u < kScanPer; u++) {
            const uint32_t t = base + tid * kScanPer + u;
            tot[u] = t < tl.ntiles ? recs[sidx0 + t].total : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < kScanPer; u++)
            sum += tot[u];
        // workgroup exclusive scan of the per-thread sums (values < 2^32 per
        // wave: 64 x 8 tiles of at most 9600 bytes)
        const uint32_t incl = wave_scan_dpp((uint32_t) sum);
        if (lane == 63)
            s_w[wv] = incl;
        __syncthreads();
        unsigned long long before = s_run;
        for (uint32_t i = 0; i < wv; i++)
            before += s_w[i];
        uint64_t at = before + (incl - (uint32_t) sum);
#pragma unroll
        for (uint32_t u = 0; u < kScanPer; u++) {
            const uint32_t t = base + tid * kScanPer + u;
            if (t < tl.ntiles) {
                const Tile x = tile_of(g, tl, t);
                pos[sidx0 + t] = 8ull * g.T + 4ull * (x.s + 1) + at;
            }
            at += tot[u];
        }
        __syncthreads();
        if (tid == kScanThreads - 1)
            s_run = at;
        __syncthreads();
    }
}

// One tile's placement (pass two, second kernel), one wave: its bytes, the
// output index group offsets, for a segment's first tile the seed and chunk
// header, for the sum's last tile the stream size.
__device__ __forceinline__ void place_tile(const Geom& g, const Tiling& tl, uint32_t t, uint8_t* out,
    uint64_t out_cap, uint8_t* oindex, unsigned long long* size_out, const uint8_t* stage, uint64_t R,
    uint64_t sidx, WsHeader* ws)
{
    const uint32_t lane = threadIdx.x & 63;
    const StageRec rec = reinterpret_cast<const StageRec*>(stage + 8 * R)[sidx];
    const uint64_t P = ((const unsigned long long*) stage)[sidx];
    const Tile x = tile_of(g, tl, t);
    const bool fits = P + rec.total <= out_cap;
    if (!fits && lane == 0)
        raise_error(ws, ZK_ERR_NOSPACE);
    if (fits)
        copy_wave(out + P, stage + (8 + sizeof(StageRec)) * R + kStageSlot * sidx, rec.total);
    IndexView ox = index_view(g, oindex);
    if (lane < x.ngrp) {
        const uint32_t e = lane == 0 ? 0u : lane == 1 ? rec.e16 : lane == 2 ? rec.e32 : rec.e48;
        ox.group_off[x.grp0 + lane] = P + e;
    }
    if (lane == 0) {
        if (x.lt == 0) {
            const uint64_t so = P - 4;
            if (so + 4 <= out_cap) {
                store_bytes(out + so, &rec.seed, 4);
                if (x.s < g.T) {
                    const unsigned long long h = so - 8ull * g.T;
                    store_bytes(out + 8ull * x.s, &h, 8);
                }
            }
            ox.seed_off[x.s] = so;
        }
        if (t == tl.ntiles - 1) {
            // the last tile ends the stream: if it fits, every tile fits
            const unsigned long long sz = fits ? P + rec.total : 0ull;
            ox.meta[0] = sz;
            if (size_out)
                *size_out = sz;
        }
    }
}

__global__ void __launch_bounds__(kScanThreads) k_scan_lane(HomsumArgs a, const uint8_t* stage)
{
    scan_sum(a.job.g, a.job.tl, stage, a.job.tl.ntiles, 0);
}

__global__ void __launch_bounds__(kScanThreads) k_scan_lane_batch(BatchArgs b, const uint8_t* stage)
{
    scan_sum(b.g, b.tl, stage, b.total_tiles, (uint64_t) blockIdx.x * b.tl.ntiles);
}

__global__ void __launch_bounds__(64 * kLaneWaves) k_place_lane(HomsumArgs a, const uint8_t* stage)
{
    const uint64_t t = (uint64_t) xcd_block(blockIdx.x, gridDim.x) * kLaneWaves + (threadIdx.x >> 6);
    if (t >= a.job.tl.ntiles)
        return;
    place_tile(a.job.g, a.job.tl, (uint32_t) t, a.job.io.out, a.job.io.out_cap, a.job.io.index, a.job.io.size_out,
        stage, a.job.tl.ntiles, t, a.ws);
}

// Uniform batch: workgroups as in pass one.
__global__ void __launch_bounds__(64 * kLaneWaves) k_place_lane_batch(BatchArgs b, const uint8_t* stage)
{
    const uint32_t wpj = (uint32_t) ceil_div(b.tl.ntiles, kLaneWaves);
    const uint32_t g = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t jidx = __builtin_amdgcn_readfirstlane(g / wpj);
    const uint32_t t = __builtin_amdgcn_readfirstlane((g % wpj) * kLaneWaves + (threadIdx.x >> 6));
    if (jidx >= b.njobs || t >= b.tl.ntiles)
        return;
    const HomsumIO* io = (const HomsumIO*) b.jobs + jidx;
    place_tile(b.g, b.tl, t, ldc(&io->out), ldc(&io->out_cap), ldc(&io->index), ldc(&io->size_out), stage,
        b.total_tiles, (uint64_t) jidx * b.tl.ntiles + t, b.ws);
}

size_t lane_lds_bytes() { return (size_t) kLaneWaves * kOutBuf; }

// Workgroups of W waves, one ticket each.
template <uint32_t W, typename K, typename A>
static hipError_t launch_sum(K kernel, uint64_t ntiles, const A& args, hipStream_t s)
{
    hipLaunchKernelGGL(kernel, dim3((uint32_t) ceil_div(ntiles, W)), dim3(64 * W), W * kOutBuf, s, args);
    return hipGetLastError();
}

hipError_t launch_homsum_lane(const HomsumArgs& a, hipStream_t s)
{
    const uint64_t n = a.job.tl.ntiles;
    return n > kSumFew ? launch_sum<kSumMany>(k_homsum_lane<kSumMany>, n, a, s) :
                         launch_sum<kLaneWaves>(k_homsum_lane<kLaneWaves>, n, a, s);
}

hipError_t launch_homsum_lane_batch(const BatchArgs& b, hipStream_t s)
{
    const uint64_t n = b.total_tiles;
    if (b.uniform)
        return n > kSumFew ? launch_sum<kSumMany>(k_homsum_lane_batch<kSumMany>, n, b, s) :
                             launch_sum<kLaneWaves>(k_homsum_lane_batch<kLaneWaves>, n, b, s);
    return n > kSumFew ? launch_sum<kSumMany>(k_homsum_lane_mixed<kSumMany>, n, b, s) :
                         launch_sum<kLaneWaves>(k_homsum_lane_mixed<kLaneWaves>, n, b, s);
}

// (four: what the LDS buffers let a CU hold)
constexpr int kDecGroupsDefault = 4;
static std::atomic<int> g_dec_groups{kDecGroupsDefault};

bool set_decompress_groups_per_cu(int groups)
{
    if (groups == 0)
        groups = kDecGroupsDefault;
    if (groups < 1 || groups > kDecGroupsMax)
        return false;
    g_dec_groups.store(groups);
    return true;
}

int get_decompress_groups_per_cu() { return g_dec_groups.load(); }

uint32_t device_cu_count()
{
    static std::atomic<int> cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        dev = 0;
    int n = cus[dev].load();
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        cus[dev].store(n);
    }
    return (uint32_t) n;
}

// Workgroups of a persistent decompress grid: the tuned number per CU (at
// most as many as the device holds at once), or one per four tiles when that
// is fewer.
static uint32_t dec_groups(uint64_t tiles)
{
    return (uint32_t) std::min<uint64_t>(ceil_div(tiles, kLaneWaves), (uint64_t) device_cu_count() * g_dec_groups.load());
}

hipError_t launch_decompress_lane(const DecompressArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_decompress_lane, dim3(dec_groups(a.job.tl.ntiles)), dim3(64 * kLaneWaves), lane_lds_bytes(), s, a);
    return hipGetLastError();
}

hipError_t launch_decompress_lane_batch(const BatchArgs& b, hipStream_t s)
{
    hipLaunchKernelGGL(k_decompress_lane_batch, dim3(dec_groups(b.total_tiles)), dim3(64 * kLaneWaves), lane_lds_bytes(),
        s, b);
    return hipGetLastError();
}

hipError_t launch_lane_carries(const DecompressArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_lane_carry_sums, dim3(dec_groups(a.job.tl.ntiles)), dim3(64 * kLaneWaves), lane_lds_bytes(), s, a);
    if (std::max(a.job.g.cT, a.job.g.cR) <= kCarryShort)
        hipLaunchKernelGGL(k_lane_carry_scan<64>, dim3(a.job.g.S), dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL(k_lane_carry_scan<1024>, dim3(a.job.g.S), dim3(1024), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_homsum_lane_wg(const HomsumArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_homsum_lane_wg, dim3((uint32_t) a.job.tl.ntiles), dim3(64 * kLaneWaves), lane_lds_bytes(),
        s, a);
    return hipGetLastError();
}

hipError_t launch_homsum_lane_wg_batch(const BatchArgs& b, hipStream_t s)
{
    if (b.uniform)
        hipLaunchKernelGGL(k_homsum_lane_wg_batch, dim3((uint32_t) b.total_tiles), dim3(64 * kLaneWaves),
            lane_lds_bytes(), s, b);
    else
        hipLaunchKernelGGL(k_homsum_lane_wg_mixed, dim3((uint32_t) b.total_tiles), dim3(64 * kLaneWaves),
            lane_lds_bytes(), s, b);
    return hipGetLastError();
}

// Workgroups of N tiles each (kCompFew: where the line lies).
template <uint32_t N, typename K, typename A>
static hipError_t launch_comp(K kernel, uint64_t ntiles, const A& args, hipStream_t s)
{
    hipLaunchKernelGGL(kernel, dim3((uint32_t) ceil_div(ntiles, N)), dim3(64 * kLaneWaves * N), N * kLaneWaves * kCompBuf,
        s, args);
    return hipGetLastError();
}

hipError_t launch_compress_lane(const CompressArgs& a, hipStream_t s)
{
    const uint64_t n = a.job.tl.ntiles;
    return n > kCompFew ? launch_comp<kCompPair>(k_compress_lane<kCompPair>, n, a, s) :
                          launch_comp<1>(k_compress_lane<1>, n, a, s);
}

hipError_t launch_compress_lane_batch(const BatchArgs& b, hipStream_t s)
{
    const uint64_t n = b.total_tiles;
    if (b.uniform)
        return n > kCompFew ? launch_comp<kCompPair>(k_compress_lane_batch<kCompPair>, n, b, s) :
                              launch_comp<1>(k_compress_lane_batch<1>, n, b, s);
    return n > kCompFew ? launch_comp<kCompPair>(k_compress_lane_mixed<kCompPair>, n, b, s) :
                          launch_comp<1>(k_compress_lane_mixed<1>, n, b, s);
}

hipError_t launch_homsum_lane_staged(const HomsumArgs& a, uint8_t* stage, hipStream_t s)
{
    const uint64_t tiles = a.job.tl.ntiles;
    hipLaunchKernelGGL(k_homsum_lane_staged, dim3((uint32_t) ceil_div(tiles, kLaneWaves)), dim3(64 * kLaneWaves),
        lane_lds_bytes(), s, a, stage);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_scan_lane, dim3(1), dim3(kScanThreads), 0, s, a, (const uint8_t*) stage);
    hipLaunchKernelGGL(k_place_lane, dim3((uint32_t) ceil_div(tiles, kLaneWaves)), dim3(64 * kLaneWaves), 0, s, a,
        (const uint8_t*) stage);
    return hipGetLastError();
}

hipError_t launch_homsum_lane_batch_staged(const BatchArgs& b, uint8_t* stage, hipStream_t s)
{
    if (!b.uniform)
        return hipErrorInvalidValue;
    const uint32_t groups = (uint32_t) (ceil_div(b.tl.ntiles, kLaneWaves) * b.njobs);
    hipLaunchKernelGGL(k_homsum_lane_batch_staged, dim3(groups), dim3(64 * kLaneWaves), lane_lds_bytes(), s, b, stage);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_scan_lane_batch, dim3(b.njobs), dim3(kScanThreads), 0, s, b, (const uint8_t*) stage);
    hipLaunchKernelGGL(k_place_lane_batch, dim3(groups), dim3(64 * kLaneWaves), 0, s, b, (const uint8_t*) stage);
    return hipGetLastError();
}

}  // namespace zk
