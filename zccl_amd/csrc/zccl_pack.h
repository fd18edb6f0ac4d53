// zccl_pack.h -- device-side packing of one block per lane into a wave's LDS
// buffer, shared by the lane layout of the 1-D kernels (zccl_lane.hip) and the
// 3-D codec (zccl_sz3d.hip), and the exact small-integer arithmetic they use.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zk {

// Integers below 2^24 as FP32 bit patterns: a denormal's bits are its integer
// (in units of 2^-149), and the next binade's still are, so FP32 differences
// and fused multiply-adds of such patterns are exact integer arithmetic on
// sign-and-magnitude numbers.  They take half the time of the integer
// instructions that would do the same (measured on the MI355X, cycles per
// wave instruction and SIMD: add, subtract, multiply and fma FP32, and, or,
// xor, v_bitop3, right shifts 2; bit-field extracts, left shifts, 24-bit
// multiplies, v_perm, v_alignbit, min and max, conversions, FP64 4).
__device__ __forceinline__ float as_f(uint32_t v) { return __uint_as_float(v); }
__device__ __forceinline__ uint32_t as_u(float v) { return __float_as_uint(v); }

// v, computed here: without this the compiler moves what a group of values
// gives behind the branches of the groups after it (or what only a block's
// width gives ahead of a loop), and holds registers for all 36 values.
template <typename T>
__device__ __forceinline__ T stay(T v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Four bytes from any byte offset o of LDS words st (aligned dword reads: a
// misaligned LDS read takes 30 times as long), in memory order and as a
// big-endian word.
__device__ __forceinline__ uint32_t lds_at(const uint32_t* st, uint32_t o)
{
    const uint32_t* p = st + (o >> 2);
    return __builtin_amdgcn_alignbyte(p[1], p[0], o);  // uses o & 3
}

// Two's complement of a magnitude and a sign word (its bit 31).
__device__ __forceinline__ uint32_t signed_of(uint32_t m, uint32_t s)
{
    const uint32_t t = (uint32_t) ((int32_t) s >> 31);
    return (m ^ t) - t;
}

// |d| of an int32 delta as unsigned (|INT_MIN| = 2^31).
__device__ __forceinline__ uint32_t mag(uint32_t d) { return (uint32_t) max((int32_t) d, (int32_t) (0u - d)); }

// OR bytes into the wave's zeroed LDS buffer.
__device__ __forceinline__ void lds_or(uint32_t* p, uint32_t v)
{
    __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Byte-shift selector for v_perm: perm(x_i, x_{i-1}, sel) is the dword at
// 4i of a byte array placed sh bytes into the aligned grid.
__device__ __forceinline__ uint32_t shift_sel(uint32_t sh) { return 0x07060504u - sh * 0x01010101u; }

// OR the N dwords x (a byte array) at byte a of the buffer.
template <uint32_t N>
__device__ __forceinline__ void or_words(uint32_t* ob, uint32_t a, const uint32_t (&x)[N])
{
    const uint32_t sel = shift_sel(a & 3);
    uint32_t* p = ob + (a >> 2);
    uint32_t prev = 0;
#pragma unroll
    for (uint32_t i = 0; i < N; i++) {
        lds_or(p + i, __builtin_amdgcn_perm(x[i], prev, sel));
        prev = x[i];
    }
    lds_or(p + N, __builtin_amdgcn_perm(0u, prev, sel));
}

// The high bytes (B per value) of a block of width w >= 8 at byte a, four
// values at a time.  For B = 1 the bytes are put together by exact FP32
// multiply-adds.
template <uint32_t B, uint32_t N>
__device__ __forceinline__ void encode_high(uint32_t* ob, uint32_t a, uint32_t w, const uint32_t (&m)[N])
{
    const uint32_t r = w & 7, sel = shift_sel(a & 3);
    uint32_t* p = ob + (a >> 2);
    uint32_t prev = 0;
#pragma unroll
    for (uint32_t i = 0; i < N / 4; i++) {
        __builtin_amdgcn_sched_barrier(0);  // few registers live
        uint32_t h[4], x[B];
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            h[c] = m[4 * i + c] >> r;
        if constexpr (B == 1) {
            const uint32_t lo = as_u(__builtin_fmaf(as_f(h[1]), 256.0f, as_f(h[0])));
            const uint32_t hi = as_u(__builtin_fmaf(as_f(h[3]), 256.0f, as_f(h[2])));
            x[0] = lo | (hi << 16);
        } else if constexpr (B == 2) {
            x[0] = h[0] | (h[1] << 16);
            x[1] = h[2] | (h[3] << 16);
        } else if constexpr (B == 3) {
            x[0] = h[0] | (h[1] << 24);
            x[1] = (h[1] >> 8) | (h[2] << 16);
            x[2] = (h[2] >> 16) | (h[3] << 8);
        } else {
#pragma unroll
            for (uint32_t c = 0; c < 4; c++)
                x[c] = h[c];
        }
#pragma unroll
        for (uint32_t c = 0; c < B; c++) {
            lds_or(p + B * i + c, __builtin_amdgcn_perm(x[c], prev, sel));
            prev = x[c];
        }
    }
    lds_or(p + B * N / 4, __builtin_amdgcn_perm(0u, prev, sel));
}

// The high bytes of the lanes' blocks by class of width (from 8).  Separate
// branches: one with all of them would keep what they share live.
template <uint32_t N>
__device__ __forceinline__ void encode_high_class(uint32_t* ob, uint32_t a, uint32_t w, const uint32_t (&m)[N])
{
    if ((w >> 3) == 1)
        encode_high<1>(ob, a, w, m);
    if (__any(w >= 16)) {
        if ((w >> 3) == 2)
            encode_high<2>(ob, a, w, m);
        if ((w >> 3) == 3)
            encode_high<3>(ob, a, w, m);
        if (w == 32)
            encode_high<4>(ob, a, w, m);
    }
}

// The low w & 7 bits of every magnitude at byte a, an MSB-first stream: groups
// of 8 values fill r whole bytes.
template <uint32_t N>
__device__ __forceinline__ void encode_low(uint32_t* ob, uint32_t a, uint32_t w, const uint32_t (&m)[N])
{
    const uint32_t r = w & 7;
    if (!r)
        return;
    const uint32_t mask = (1u << r) - 1u;
    const float scale = as_f((127u + r) << 23);  // 2^r
#pragma unroll
    for (uint32_t g = 0; g < (N + 7) / 8; g++, a += r) {
        __builtin_amdgcn_sched_barrier(0);
        // four fields: two pairs by exact FP32 multiply-adds (14 bits at most each)
        uint32_t u[2] = {0, 0};
#pragma unroll
        for (uint32_t h = 0; h < 2; h++) {
            const uint32_t j = 8 * g + 4 * h;
            if (j < N) {
                const uint32_t f0 = m[j] & mask, f1 = m[j + 1] & mask, f2 = m[j + 2] & mask, f3 = m[j + 3] & mask;
                u[h] = (as_u(__builtin_fmaf(as_f(f0), scale, as_f(f1))) << (2 * r)) |
                       as_u(__builtin_fmaf(as_f(f2), scale, as_f(f3)));
            }
        }
        // 8 fields (the last group: 4 and zeros) = r bytes, top-aligned in Y
        const uint64_t G = ((uint64_t) u[0] << (4 * r)) | u[1];
        const uint64_t Y = G << (64 - 8 * r);
        const uint32_t z[2] = {__builtin_bswap32((uint32_t) (Y >> 32)), __builtin_bswap32((uint32_t) Y)};
        or_words(ob, a, z);
    }
}

// Write bytes [0, nbytes) of the wave's LDS buffer to dst with 16-byte stores
// on dst's 16-byte grid; the partial first and last chunk go out byte by
// byte, so bytes outside [dst, dst + nbytes) are never written.
__device__ __forceinline__ void store_wave(const uint32_t* ob, uint8_t* dst, uint32_t nbytes)
{
    const uint32_t lane = threadIdx.x & 63;
    const uintptr_t d0 = (uintptr_t) dst, d1 = d0 + nbytes;
    const uintptr_t c0 = d0 & ~(uintptr_t) 15;
    const uint32_t nch = nbytes ? (uint32_t) ((d1 - c0 + 15) >> 4) : 0u;
    for (uint32_t c = lane; c < nch; c += 64) {
        const uintptr_t ca = c0 + 16ull * c;
        if (ca >= d0 && ca + 16 <= d1) {
            const uint32_t o = (uint32_t) (ca - d0), wi = o >> 2, sh = o & 3;
            const uint32_t a = ob[wi], b = ob[wi + 1], cc = ob[wi + 2], dd = ob[wi + 3], e = ob[wi + 4];
            *(uint4*) ca = make_uint4(__builtin_amdgcn_alignbyte(b, a, sh), __builtin_amdgcn_alignbyte(cc, b, sh),
                __builtin_amdgcn_alignbyte(dd, cc, sh), __builtin_amdgcn_alignbyte(e, dd, sh));
        } else {
            const uintptr_t s = ca > d0 ? ca : d0, e = ca + 16 < d1 ? ca + 16 : d1;
            for (uintptr_t p = s; p < e; p++)
                *(uint8_t*) p = ((const uint8_t*) ob)[p - d0];
        }
    }
}

}  // namespace zk
