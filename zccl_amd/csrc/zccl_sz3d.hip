// zccl_sz3d.hip -- CDNA4 (gfx950) kernels of the 3-D SZp codec
// (SZp_compress3D_fast_openmp, ZCCL/src/ZCCL_float.c:1862-2048, and
// SZp_decompress3D_fast_openmp, ZCCL/src/ZCCLd_float.c:2873-3040).
//
// The reference walks each sub-volume with one CPU thread and running
// buffers; its residual is the exact 3-D difference dx dy dz q (zero outside
// the sub-volume) and its decoder the exact 3-D prefix sum, so both are done
// here with full parallelism:
//   compress   k3_table (sub-volume table) -> for block side 4 k3l_compress (one
//              lane per block, one pass); others k3_widths (one wave per block:
//              residuals from x, block max, width, payload size) -> scan of the
//              payload sizes -> k3_encode (one wave per block: width header
//              byte, sub-volume offset, sign bitmap and fixed-length bits with
//              the one-writer-per-byte unit encoder of the 1-D sum)
//   decompress k3_table -> for block side 4, rows of 32 to 256 blocks and enough of
//              them to fill the chip k3l_sizes, k3l_decode, k3l_ypass (one lane
//              per block, two passes over the volume); others k3_dsizes (widths
//              read from the stream's own header) -> scan -> k3_decode (residuals
//              into the output buffer as int32) -> k3_zpass / k3_ypass (inclusive
//              prefix sums along z and y) -> k3_xpass (along x, then
//              x' = (float)(q * 2 eb) in place)
// Arithmetic: q = (int)floor((double)x * (0.5 / eb) + 0.5) with the product and
// the sum rounded separately (the reference is built without FMA; this file is
// built with -ffp-contract=off); residuals and sums wrap in 32 bits.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "zccl_device.h"
#include "zccl_internal.h"
#include "zccl_kernels.h"
#include "zccl_pack.h"
#include "zccl_sz3d.h"
#include "zccl_unit.h"

namespace zk {

namespace {

__device__ __forceinline__ int32_t quant3(float v, double inv)
{
    const double p = floor(__dadd_rn(__dmul_rn((double) v, inv), 0.5));
    return (p >= -2147483648.0 && p < 2147483648.0) ? (int32_t) p : INT32_MIN;
}

__device__ __forceinline__ void raise3(unsigned long long* status, unsigned long long bit)
{
    atomicOr(&status[1], bit);
}

// Block of a sub-volume: position, extents and value count.
struct Blk3 {
    uint32_t bx, by, bz;
    uint32_t ex, ey, ez;
    uint32_t cnt;
};

__device__ __forceinline__ Blk3 block_of(const Part3& p, uint32_t lb, uint32_t Bs)
{
    Blk3 b;
    const uint32_t yz = p.b2 * p.b3;
    b.bx = lb / yz;
    const uint32_t rest = lb - b.bx * yz;
    b.by = rest / p.b3;
    b.bz = rest - b.by * p.b3;
    b.ex = min(Bs, p.sx - b.bx * Bs);
    b.ey = min(Bs, p.sy - b.by * Bs);
    b.ez = min(Bs, p.sz - b.bz * Bs);
    b.cnt = b.ex * b.ey * b.ez;
    return b;
}

// Residual of the value at local (lx, ly, lz) of sub-volume p: dx dy dz q with
// q = 0 outside the sub-volume (the reference's err_1 / err_2 / err_3 chain,
// ZCCL/src/ZCCL_float.c:1983-1990).
__device__ __forceinline__ uint32_t resid3(const float* x, const Geom3& g, const Part3& p, double inv,
    uint32_t lx, uint32_t ly, uint32_t lz)
{
    const uint64_t sx = (uint64_t) g.d2 * g.d3, sy = g.d3;
    const uint64_t i0 = ((uint64_t) (p.ox + lx) * g.d2 + (p.oy + ly)) * g.d3 + p.oz + lz;
    uint32_t acc = (uint32_t) quant3(x[i0], inv);
    if (lz)
        acc -= (uint32_t) quant3(x[i0 - 1], inv);
    if (ly) {
        acc -= (uint32_t) quant3(x[i0 - sy], inv);
        if (lz)
            acc += (uint32_t) quant3(x[i0 - sy - 1], inv);
    }
    if (lx) {
        acc -= (uint32_t) quant3(x[i0 - sx], inv);
        if (lz)
            acc += (uint32_t) quant3(x[i0 - sx - 1], inv);
        if (ly) {
            acc += (uint32_t) quant3(x[i0 - sx - sy], inv);
            if (lz)
                acc -= (uint32_t) quant3(x[i0 - sx - sy - 1], inv);
        }
    }
    return acc;
}

// Local coordinates of value e of block b (values in i, j, k order).
__device__ __forceinline__ void value_pos(const Blk3& b, uint32_t Bs, uint32_t e, uint32_t& lx, uint32_t& ly,
    uint32_t& lz)
{
    const uint32_t yz = b.ey * b.ez;
    const uint32_t i = e / yz, rest = e - i * yz, j = rest / b.ez, k = rest - j * b.ez;
    lx = b.bx * Bs + i;
    ly = b.by * Bs + j;
    lz = b.bz * Bs + k;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        v = max(v, (uint32_t) __shfl_xor(v, d, 64));
    return v;
}

__device__ __forceinline__ unsigned long long wave_incl_scan64(unsigned long long v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long y = __shfl_up(v, d, 64);
        if (lane >= d)
            v += y;
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_incl_scan32(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(v, d, 64);
        if (lane >= d)
            v += y;
    }
    return v;
}

constexpr uint32_t kSizeMask = (1u << 26) - 1;

// Sub-volume table, built on the device by one wave, a lane per sub-volume (no
// host copy on the stream the caller passes), and the status words and `nclear`
// lookback words cleared.  (One thread filling one sub-volume after the other took
// 6.4 us, the median over tables of 16 and of 4; by lanes 2.7.)
__global__ void __launch_bounds__(256) k3_table(Geom3 g, Split3 sp, Part3* parts, unsigned long long* status,
    unsigned long long* clear, uint32_t nclear)
{
    if (threadIdx.x < 64 && blockIdx.x == 0) {
        const uint32_t lane = threadIdx.x;
        if (lane < 3)
            status[lane] = 0;
        Sums3 run = {};
        for (uint32_t t0 = 0; t0 < g.T; t0 += 64) {
            Part3 p;
            const uint32_t t = t0 + lane;
            const Sums3 c = part3(g, sp, min(t, g.T - 1), p);
            Sums3 before;
#pragma unroll
            for (uint32_t i = 0; i < kSums3; i++) {
                const uint32_t inc = wave_scan_dpp(c.v[i]);
                before.v[i] = run.v[i] + inc - c.v[i];
                run.v[i] += __builtin_amdgcn_readlane(inc, 63);
            }
            place3(p, before);
            if (t < g.T)
                parts[t] = p;
        }
    }
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < nclear; i += gridDim.x * 256)
        clear[i] = 0;
}

// Width and payload size of every block: one wave per block.
__global__ void __launch_bounds__(256) k3_widths(Sz3Args a)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t gb = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (gb >= a.g.nblocks)
        return;
    const uint32_t t = __builtin_amdgcn_readfirstlane(part_of_block(a.parts, a.g.T, gb));
    const Part3 p = a.parts[t];
    const Blk3 b = block_of(p, gb - p.g0, a.g.Bs);
    uint32_t m = 0;
    for (uint32_t e = lane; e < b.cnt; e += 64) {
        uint32_t lx, ly, lz;
        value_pos(b, a.g.Bs, e, lx, ly, lz);
        m = max(m, mag32(resid3(a.x, a.g, p, a.inv, lx, ly, lz)));
    }
    m = wave_max(m);
    if (lane == 0) {
        const uint32_t w = m ? 32u - (uint32_t) __clz((int) m) : 0u;
        a.words[gb] = payload3(w, b.cnt) | (w << 26);
    }
}

// Payload sizes of a stream's blocks from its own header: one thread per block.
__global__ void __launch_bounds__(256) k3_dsizes(Sz3Args a)
{
    const uint32_t gb = blockIdx.x * blockDim.x + threadIdx.x;
    if (gb >= a.g.nblocks)
        return;
    const uint32_t t = part_of_block(a.parts, a.g.T, gb);
    const Part3 p = a.parts[t];
    const Blk3 b = block_of(p, gb - p.g0, a.g.Bs);
    uint64_t h;
    __builtin_memcpy(&h, a.in + 8ull * t, 8);
    const uint64_t wpos = 8ull * a.g.T + h + (gb - p.g0);
    uint32_t w = 0;
    if (wpos < a.in_size) {
        w = a.in[wpos];
        if (w > 32) {
            raise3(a.status, ZK_ERR_WIDTH);
            w = 0;
        }
    } else {
        raise3(a.status, ZK_ERR_OVERRUN);
    }
    a.words[gb] = payload3(w, b.cnt) | (w << 26);
}

// Exclusive scan of the payload sizes (low 26 bits of words[]) into offs[]:
// group sums, a scan of the group sums by one workgroup, then each group's
// local scan.  256 threads, kScan3Group = 1024 entries per group.
__global__ void __launch_bounds__(256) k3_scan_groups(Sz3Args a)
{
    __shared__ unsigned long long s_w[4];
    const uint32_t base = blockIdx.x * kScan3Group;
    unsigned long long v = 0;
    for (uint32_t i = threadIdx.x; i < kScan3Group; i += 256)
        if (base + i < a.g.nblocks)
            v += a.words[base + i] & kSizeMask;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        v += __shfl_xor(v, d, 64);
    if ((threadIdx.x & 63) == 0)
        s_w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        a.part_sums[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// One workgroup: exclusive scan of the group sums in place; the stream size
// (header, width bytes, payloads) goes to status[0] and the optional size
// word; a compress whose stream exceeds the output capacity raises NOSPACE.
__global__ void __launch_bounds__(256) k3_scan_top(Sz3Args a, uint32_t ngroups, int check_cap)
{
    __shared__ unsigned long long s_w[4];
    __shared__ unsigned long long s_carry;
    if (threadIdx.x == 0)
        s_carry = 0;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < ngroups; c0 += 256) {
        const uint32_t i = c0 + threadIdx.x;
        const unsigned long long v = i < ngroups ? a.part_sums[i] : 0ull;
        const unsigned long long inc = wave_incl_scan64(v);
        if ((threadIdx.x & 63) == 63)
            s_w[threadIdx.x >> 6] = inc;
        __syncthreads();
        unsigned long long pre = s_carry;
        for (uint32_t w = 0; w < (threadIdx.x >> 6); w++)
            pre += s_w[w];
        if (i < ngroups)
            a.part_sums[i] = pre + inc - v;
        __syncthreads();
        if (threadIdx.x == 255)
            s_carry = pre + inc;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned long long total = 8ull * a.g.T + a.g.nblocks + s_carry;
        a.status[0] = total;
        a.part_sums[ngroups] = s_carry;
        if (check_cap && total > a.out_cap)
            raise3(a.status, ZK_ERR_NOSPACE);
        if (a.size_out)
            *a.size_out = (check_cap && total > a.out_cap) ? 0ull : total;
    }
}

__global__ void __launch_bounds__(256) k3_scan_apply(Sz3Args a)
{
    __shared__ unsigned long long s_w[4];
    const uint32_t base = blockIdx.x * kScan3Group + threadIdx.x * 4;
    uint32_t v[4], run = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        v[c] = base + c < a.g.nblocks ? a.words[base + c] & kSizeMask : 0u;
        run += v[c];
    }
    const unsigned long long inc = wave_incl_scan64(run);
    if ((threadIdx.x & 63) == 63)
        s_w[threadIdx.x >> 6] = inc;
    __syncthreads();
    unsigned long long pre = a.part_sums[blockIdx.x] + inc - run;
    for (uint32_t w = 0; w < (threadIdx.x >> 6); w++)
        pre += s_w[w];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if (base + c < a.g.nblocks)
            a.offs[base + c] = pre;
        pre += v[c];
    }
}

// LDS bytes per wave for one block's payload: blocks whose payload fits are
// encoded (decoded) in LDS and moved with dword copies; larger ones work on
// global memory byte by byte.  Side 9 (729 values, at most 3008 bytes) fits.
constexpr uint32_t kStage3 = 4096;

// Make a wave's LDS writes visible to its other lanes.
__device__ __forceinline__ void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Header byte, sub-volume offset and payload of every block: one wave per
// block, 4-value units in consecutive lanes (so unit pairs share a wave).
__global__ void __launch_bounds__(256) k3_encode(Sz3Args a)
{
    __shared__ uint32_t s_stage[4][kStage3 / 4];
    __shared__ uint32_t s_res[4][256];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t gb = blockIdx.x * 4 + wv;
    if (gb >= a.g.nblocks || (a.status[1] & ZK_ERR_NOSPACE))
        return;
    const uint32_t t = __builtin_amdgcn_readfirstlane(part_of_block(a.parts, a.g.T, gb));
    const Part3 p = a.parts[t];
    const uint32_t lb = gb - p.g0, Bs = a.g.Bs;
    const Blk3 b = block_of(p, lb, Bs);
    const uint32_t word = a.words[gb], w = word >> 26, size = word & kSizeMask;
    const uint64_t sub = (uint64_t) p.nbc + a.offs[p.g0];  // sub-volume start after the header
    const uint64_t hdr = 8ull * a.g.T;
    if (lane == 0) {
        a.out[hdr + sub + lb] = (uint8_t) w;
        if (lb == 0)
            __builtin_memcpy(a.out + 8ull * t, &sub, 8);
    }
    if (!w)
        return;
    const uint64_t fo = hdr + p.nbc + (uint64_t) p.b1 * p.b2 * p.b3 + a.offs[gb];
    const bool staged = size <= kStage3;
    uint8_t* st = (uint8_t*) s_stage[wv];
    const uint32_t U = (b.cnt + 3) / 4;
    uint32_t* res = s_res[wv];
    for (uint32_t u0 = 0; u0 < U; u0 += 64) {
        // residuals of the next 256 values, one per lane per step, then each
        // unit lane takes its four
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            const uint32_t e = 4 * u0 + 64 * c + lane;
            uint32_t r = 0;
            if (e < b.cnt) {
                uint32_t lx, ly, lz;
                value_pos(b, Bs, e, lx, ly, lz);
                r = resid3(a.x, a.g, p, a.inv, lx, ly, lz);
            }
            res[64 * c + lane] = r;
        }
        wave_sync_lds();
        const uint32_t u = u0 + lane;
        const uint32_t cnt = u < U ? min(4u, b.cnt - 4 * u) : 0u;
        uint32_t d[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            d[c] = c < cnt ? res[4 * lane + c] : 0u;
        wave_sync_lds();
        const UnitFields f = unit_fields(w, d);
        const uint32_t pnib = __shfl_down(f.nib, 1, 64);
        const uint32_t plv = __shfl_down(f.lv, 1, 64);
        if (staged)
            emit_unit(st, 0, w, b.cnt, u, U, cnt, f, pnib, plv);
        else
            emit_unit(a.out, fo, w, b.cnt, u, U, cnt, f, pnib, plv);
    }
    if (staged) {
        // every payload byte has one writer; dword stores cover only whole
        // dwords of this payload, the tail goes out byte by byte
        wave_sync_lds();
        uint8_t* g = a.out + fo;
        const uint32_t nw = size / 4;
        for (uint32_t i = lane; i < nw; i += 64) {
            const uint32_t v = ((const uint32_t*) st)[i];
            __builtin_memcpy(g + 4 * i, &v, 4);
        }
        for (uint32_t i = 4 * nw + lane; i < size; i += 64)
            g[i] = st[i];
    }
}

// Byte j of a payload (0 past its end, which no well-formed block reads).
__device__ __forceinline__ uint32_t pbyte(const uint8_t* p, uint32_t size, uint32_t j)
{
    return j < size ? p[j] : 0u;
}

// Residuals of every block into the output buffer as int32 at their positions
// in the volume: one wave per block, one 4-value unit per lane.  A payload of
// at most kStage3 bytes is copied into LDS (dword loads, 16 zero bytes of
// slack) and decoded with the 1-D unit decoder; a larger one is read byte by
// byte from global memory.
// ZCCL/src/ZCCL_TypeManager.c:423-517 (fixed-length bits), :906-950 (signs).
__global__ void __launch_bounds__(256) k3_decode(Sz3Args a)
{
    __shared__ uint32_t s_stage[4][kStage3 / 4 + 8];
    __shared__ uint32_t s_res[4][256];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t gb = blockIdx.x * 4 + wv;
    if (gb >= a.g.nblocks)
        return;
    const uint32_t t = __builtin_amdgcn_readfirstlane(part_of_block(a.parts, a.g.T, gb));
    const Part3 p = a.parts[t];
    const uint32_t lb = gb - p.g0, Bs = a.g.Bs;
    const Blk3 b = block_of(p, lb, Bs);
    const uint32_t word = a.words[gb], w = word >> 26, size = word & kSizeMask;
    uint64_t h;
    __builtin_memcpy(&h, a.in + 8ull * t, 8);
    const uint64_t fo = 8ull * a.g.T + h + (uint64_t) p.b1 * p.b2 * p.b3 + (a.offs[gb] - a.offs[p.g0]);
    const bool inside = fo + size <= a.in_size;
    if (w && !inside && lane == 0)
        raise3(a.status, ZK_ERR_OVERRUN);
    const uint8_t* pl = a.in + fo;
    const uint32_t B = w >> 3, r = w & 7, sb = (b.cnt + 7) / 8;
    const bool staged = w && inside && size <= kStage3;
    uint8_t* st = (uint8_t*) s_stage[wv];
    if (staged) {
        const uint32_t nw = size / 4;
        for (uint32_t i = lane; i < nw; i += 64) {
            uint32_t v;
            __builtin_memcpy(&v, pl + 4 * i, 4);
            ((uint32_t*) st)[i] = v;
        }
        for (uint32_t i = 4 * nw + lane; i < size; i += 64)
            st[i] = pl[i];
        if (lane < 16)
            st[size + lane] = 0;
        wave_sync_lds();
    }
    int32_t* q = (int32_t*) a.y;
    uint32_t* res = s_res[wv];
    const uint32_t U = (b.cnt + 3) / 4;
    for (uint32_t u0 = 0; u0 < U; u0 += 64) {
        const uint32_t u = u0 + lane;
        const uint32_t cnt = u < U ? min(4u, b.cnt - 4 * u) : 0u;
        uint32_t v[4] = {0, 0, 0, 0};
        if (!cnt) {
        } else if (staged) {
            accumulate_unit(st - 1, w, b.cnt, sb, u, v);  // fields start right after the (absent) width byte
        } else if (w && inside) {
            for (uint32_t c = 0; c < cnt; c++) {
                const uint32_t e = 4 * u + c;
                uint32_t m = 0;
                for (uint32_t k = 0; k < B; k++)
                    m |= pbyte(pl, size, sb + e * B + k) << (8 * k);
                uint32_t lo = 0;
                for (uint32_t bit = e * r, s2 = 0; s2 < r; s2++, bit++)
                    lo = (lo << 1) | ((pbyte(pl, size, sb + B * b.cnt + (bit >> 3)) >> (7 - (bit & 7))) & 1u);
                m = (m << r) | lo;
                v[c] = ((pbyte(pl, size, e >> 3) >> (7 - (e & 7))) & 1u) ? 0u - m : m;
            }
        }
        // the unit lanes' values go through LDS so all lanes write them out,
        // one value each per step
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            res[4 * lane + c] = v[c];
        wave_sync_lds();
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            const uint32_t e = 4 * u0 + 64 * c + lane;
            if (e < b.cnt) {
                uint32_t lx, ly, lz;
                value_pos(b, Bs, e, lx, ly, lz);
                q[((uint64_t) (p.ox + lx) * a.g.d2 + (p.oy + ly)) * a.g.d3 + p.oz + lz] = (int32_t) res[64 * c + lane];
            }
        }
        wave_sync_lds();
    }
}

// Inclusive prefix sums along z: one wave per (sub-volume, x, y) row.
__global__ void __launch_bounds__(256) k3_zpass(Sz3Args a)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.g.zrows)
        return;
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].zr0 <= row)
            lo = mid;
        else
            hi = mid;
    }
    const Part3 p = a.parts[__builtin_amdgcn_readfirstlane(lo)];
    const uint32_t r = row - p.zr0, lx = r / p.sy, ly = r - lx * p.sy;
    uint32_t* q = (uint32_t*) a.y + ((uint64_t) (p.ox + lx) * a.g.d2 + (p.oy + ly)) * a.g.d3 + p.oz;
    uint32_t carry = 0;
    for (uint32_t z0 = 0; z0 < p.sz; z0 += 64) {
        const uint32_t z = z0 + lane;
        const uint32_t v = z < p.sz ? q[z] : 0u;
        const uint32_t inc = wave_incl_scan32(v) + carry;
        if (z < p.sz)
            q[z] = inc;
        carry = __shfl(inc, 63, 64);
    }
}

// Along y: one thread per (sub-volume, x, z) column, kAhead3 rows of loads in
// flight before their stores (512^3 with block side 8, us: y pass 239 without, 188
// with 8, 213 with 16; x pass 249, 204, 230; 64^3: 11.8, 5.1, 4.6 and 7.2, 5.1, 4.7).
constexpr uint32_t kAhead3 = 8;

__global__ void __launch_bounds__(256) k3_ypass(Sz3Args a)
{
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= a.g.ycols)
        return;
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].yc0 <= col)
            lo = mid;
        else
            hi = mid;
    }
    const Part3 p = a.parts[lo];
    const uint32_t c = col - p.yc0, lx = c / p.sz, lz = c - lx * p.sz;
    uint32_t* q = (uint32_t*) a.y + ((uint64_t) (p.ox + lx) * a.g.d2 + p.oy) * a.g.d3 + p.oz + lz;
    uint32_t run = 0;
    for (uint32_t y0 = 0; y0 < p.sy; y0 += kAhead3) {
        uint32_t v[kAhead3];
#pragma unroll
        for (uint32_t r = 0; r < kAhead3; r++)
            v[r] = q[(uint64_t) min(y0 + r, p.sy - 1) * a.g.d3];
#pragma unroll
        for (uint32_t r = 0; r < kAhead3; r++) {
            if (y0 + r < p.sy) {
                run += v[r];
                q[(uint64_t) (y0 + r) * a.g.d3] = run;
            }
        }
    }
}

// Along x, then dequantize in place: one thread per (sub-volume, y, z) column.
// x' = (float)((double)q * 2 eb), ZCCL/src/ZCCLd_float.c:3030.
__global__ void __launch_bounds__(256) k3_xpass(Sz3Args a)
{
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= a.g.xcols)
        return;
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].xc0 <= col)
            lo = mid;
        else
            hi = mid;
    }
    const Part3 p = a.parts[lo];
    const uint32_t c = col - p.xc0, ly = c / p.sz, lz = c - ly * p.sz;
    const uint64_t sx = (uint64_t) a.g.d2 * a.g.d3;
    uint32_t* q = (uint32_t*) a.y + ((uint64_t) p.ox * a.g.d2 + (p.oy + ly)) * a.g.d3 + p.oz + lz;
    float* y = a.y + (q - (uint32_t*) a.y);
    uint32_t run = 0;
    for (uint32_t x0 = 0; x0 < p.sx; x0 += kAhead3) {
        uint32_t v[kAhead3];
#pragma unroll
        for (uint32_t r = 0; r < kAhead3; r++)
            v[r] = q[min(x0 + r, p.sx - 1) * sx];
#pragma unroll
        for (uint32_t r = 0; r < kAhead3; r++) {
            if (x0 + r < p.sx) {
                run += v[r];
                y[(x0 + r) * sx] = (float) __dmul_rn((double) (int32_t) run, a.tw);
            }
        }
    }
}

// ------------------------------------------------------------ tiled path
// Block sides 4 and 8.  A workgroup takes one chunk: a (bx, by) column of
// blocks of one sub-volume, cut to Tile3::NZ blocks along z.  Compress
// quantizes the chunk's values and a one-value halo (x - 1, y - 1, z - 1; zero
// outside the sub-volume) once into LDS and takes every residual from there;
// the decoder decodes a chunk's blocks into an LDS tile of z rows and scans
// them along z there (carrying across the column's chunks), so only the y and
// x passes remain.

template <uint32_t BS>
struct Tile3 {
    static constexpr uint32_t NZ = tile_nz3(BS);             // blocks per chunk
    static constexpr uint32_t WZ = NZ * BS;                  // z values per chunk
    static constexpr uint32_t SZ = WZ + 1;                   // with the z halo
    static constexpr uint32_t S1 = BS + 1;                   // x and y with the halo
    static constexpr uint32_t U = BS * BS * BS / 4;          // units of a whole block
    static constexpr uint32_t BPW = U >= 64 ? 1u : 64u / U;  // blocks per wave step
    static constexpr uint32_t STEPS = U >= 64 ? U / 64 : 1u; // wave steps per block
    static constexpr uint32_t UPR = BS / 4;                  // units per z row of a block
    // worst-case payload (signs + 32-bit values), 16-byte multiple, + slack
    static constexpr uint32_t PAY = ((BS * BS * BS + 7) / 8 + 4 * BS * BS * BS + 15) / 16 * 16 + 32;
};

// Quantized values of a chunk and its halo into qt[(i * S1 + j) * SZ + k]:
// tile (i, j, k) holds q at local (bx Bs + i - 1, by Bs + j - 1, lz0 + k - 1).
// A wave takes RG rows at a time and issues all their loads before it
// quantizes any, so each wave keeps up to RG * KS loads in flight.
template <uint32_t BS>
__device__ __forceinline__ void load_qtile(const Sz3Args& a, const Part3& p, uint32_t bx, uint32_t by, uint32_t lz0,
    uint32_t wz, uint32_t ex, uint32_t ey, int32_t* qt)
{
    using C = Tile3<BS>;
    constexpr uint32_t KS = (C::SZ + 63) / 64, RG = 4;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (uint32_t r0 = RG * wv; r0 < C::S1 * C::S1; r0 += 4 * RG) {
        float v[RG][KS];
        bool live[RG];
#pragma unroll
        for (uint32_t h = 0; h < RG; h++) {
            const uint32_t row = r0 + h, i = row / C::S1, j = row - i * C::S1;
            live[h] = row < C::S1 * C::S1 && i <= ex && j <= ey && (i > 0 || bx > 0) && (j > 0 || by > 0);
            // element of (i - 1, j - 1, lz0) in the volume; every load below is
            // unconditional (clamped into the row, or element 0 for a dead row)
            // so the compiler keeps them all in flight
            const uint64_t rb = live[h] ?
                ((uint64_t) (p.ox + bx * BS + i - 1) * a.g.d2 + (p.oy + by * BS + j - 1)) * a.g.d3 + p.oz + lz0 : 0ull;
#pragma unroll
            for (uint32_t s = 0; s < KS; s++) {
                const uint32_t kk = min(lane + 64 * s, wz);
                const uint64_t e = rb + kk - ((kk > 0 || lz0 > 0) ? 1u : 0u);
                v[h][s] = a.x[live[h] ? e : 0ull];
            }
        }
#pragma unroll
        for (uint32_t h = 0; h < RG; h++) {
            const uint32_t row = r0 + h;
            if (row >= C::S1 * C::S1)
                continue;
            int32_t* dst = qt + row * C::SZ;
#pragma unroll
            for (uint32_t s = 0; s < KS; s++) {
                const uint32_t k = lane + 64 * s;
                if (k <= wz)
                    dst[k] = live[h] && (k > 0 || lz0 > 0) ? quant3(v[h][s], a.inv) : 0;
            }
        }
    }
}

// Column term of the residual at tile z index tk: the x-y difference of the
// four rows around (i, j) (value coordinates).
template <uint32_t BS>
__device__ __forceinline__ uint32_t col_term(const int32_t* qt, uint32_t i, uint32_t j, uint32_t tk)
{
    using C = Tile3<BS>;
    const int32_t* a0 = qt + ((i + 1) * C::S1 + (j + 1)) * C::SZ + tk;
    const int32_t* a2 = a0 - C::S1 * C::SZ;
    return (uint32_t) a0[0] - (uint32_t) a0[-(int) C::SZ] - (uint32_t) a2[0] + (uint32_t) a2[-(int) C::SZ];
}

// Residuals of unit u of a block whose first value has chunk-local z kb:
// returns the unit's value count (0..4) and its residuals in r[].
template <uint32_t BS>
__device__ __forceinline__ uint32_t unit_resid(const int32_t* qt, uint32_t ex, uint32_t ey, uint32_t ez, uint32_t cnt,
    uint32_t kb, uint32_t u, uint32_t r[4])
{
    using C = Tile3<BS>;
    const uint32_t n = 4 * u < cnt ? min(4u, cnt - 4 * u) : 0u;
    if (!n)
        return 0;
    if (cnt == BS * BS * BS) {
        // whole block: the unit is 4 consecutive values of one z row
        const uint32_t i = u / (BS * C::UPR), j = (u / C::UPR) % BS, k0 = kb + (u % C::UPR) * 4;
        uint32_t prev = col_term<BS>(qt, i, j, k0);
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            const uint32_t cur = col_term<BS>(qt, i, j, k0 + c + 1);
            r[c] = cur - prev;
            prev = cur;
        }
    } else {
        const uint32_t yz = ey * ez;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            r[c] = 0;
            if (c < n) {
                const uint32_t e = 4 * u + c, i = e / yz, rest = e - i * yz, j = rest / ez, k = rest - j * ez;
                r[c] = col_term<BS>(qt, i, j, kb + k + 1) - col_term<BS>(qt, i, j, kb + k);
            }
        }
    }
    return n;
}

template <uint32_t BS>
__device__ __forceinline__ Chunk3 chunk_of(const Part3& p, uint32_t rel)
{
    return chunk_of3(p, rel, BS);
}

// Width and payload size of every block of a chunk.
template <uint32_t BS>
__global__ void __launch_bounds__(256) k3t_widths(Sz3Args a)
{
    using C = Tile3<BS>;
    __shared__ int32_t qt[C::S1 * C::S1 * C::SZ];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t t = part_of_unit(a.parts, a.g.T, blockIdx.x, false);
    const Part3 p = a.parts[t];
    const Chunk3 c = chunk_of<BS>(p, blockIdx.x - p.u0);
    load_qtile<BS>(a, p, c.bx, c.by, c.lz0, c.wz, c.ex, c.ey, qt);
    __syncthreads();
    const uint32_t ul = C::BPW > 1 ? lane % C::U : lane;
    for (uint32_t base = wv * C::BPW; base < c.nbz; base += 4 * C::BPW) {
        const uint32_t bzl = base + (C::BPW > 1 ? lane / C::U : 0u);
        const uint32_t ez = bzl < c.nbz ? min(BS, c.wz - bzl * BS) : 0u;
        const uint32_t cnt = c.ex * c.ey * ez;
        uint32_t m = 0;
        for (uint32_t s = 0; s < C::STEPS; s++) {
            uint32_t r[4];
            const uint32_t n = unit_resid<BS>(qt, c.ex, c.ey, ez, cnt, bzl * BS, C::BPW > 1 ? ul : s * 64 + lane, r);
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
                if (k < n)
                    m = max(m, mag32(r[k]));
        }
        if (C::BPW > 1) {
#pragma unroll
            for (uint32_t d = C::U / 2; d >= 1; d >>= 1)
                m = max(m, (uint32_t) __shfl_xor(m, d, 64));
        } else {
            m = wave_max(m);
        }
        if (ul == 0 && bzl < c.nbz) {
            const uint32_t w = m ? 32u - (uint32_t) __clz((int) m) : 0u;
            a.words[c.gcol + bzl] = payload3(w, cnt) | (w << 26);
        }
    }
}

// Header byte, sub-volume offset and payload of every block of a chunk; the
// payloads are built in LDS by the unit encoder of the 1-D sum and stored with
// dword stores that cover only the block's own bytes.
template <uint32_t BS>
__global__ void __launch_bounds__(256) k3t_encode(Sz3Args a)
{
    using C = Tile3<BS>;
    __shared__ int32_t qt[C::S1 * C::S1 * C::SZ];
    __shared__ uint32_t s_pay[4][C::BPW][C::PAY / 4];
    if (a.status[1] & ZK_ERR_NOSPACE)
        return;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t t = part_of_unit(a.parts, a.g.T, blockIdx.x, false);
    const Part3 p = a.parts[t];
    const uint32_t rel = blockIdx.x - p.u0;
    const Chunk3 c = chunk_of<BS>(p, rel);
    const uint64_t hdr = 8ull * a.g.T;
    const uint64_t sub = (uint64_t) p.nbc + a.offs[p.g0];  // sub-volume start after the header
    if (rel == 0 && threadIdx.x == 0)
        __builtin_memcpy(a.out + 8ull * t, &sub, 8);
    load_qtile<BS>(a, p, c.bx, c.by, c.lz0, c.wz, c.ex, c.ey, qt);
    __syncthreads();
    const uint32_t ul = C::BPW > 1 ? lane % C::U : lane;
    const uint32_t step = C::BPW > 1 ? C::U : 64u;
    uint8_t* st = (uint8_t*) s_pay[wv][C::BPW > 1 ? lane / C::U : 0u];
    for (uint32_t base = wv * C::BPW; base < c.nbz; base += 4 * C::BPW) {
        const uint32_t bzl = base + (C::BPW > 1 ? lane / C::U : 0u);
        const bool valid = bzl < c.nbz;
        const uint32_t gb = c.gcol + bzl;
        const uint32_t word = valid ? a.words[gb] : 0u, w = word >> 26, size = word & kSizeMask;
        const uint32_t ez = valid ? min(BS, c.wz - bzl * BS) : 0u;
        const uint32_t cnt = c.ex * c.ey * ez, Ub = (cnt + 3) / 4;
        if (valid && ul == 0)
            a.out[hdr + sub + (gb - p.g0)] = (uint8_t) w;
        for (uint32_t s = 0; s < C::STEPS; s++) {
            const uint32_t u = C::BPW > 1 ? ul : s * 64 + lane;
            uint32_t d[4] = {0, 0, 0, 0};
            const uint32_t n = w ? unit_resid<BS>(qt, c.ex, c.ey, ez, cnt, bzl * BS, u, d) : 0u;
            const UnitFields f = unit_fields(w, d);
            const uint32_t pnib = __shfl_down(f.nib, 1, 64);
            const uint32_t plv = __shfl_down(f.lv, 1, 64);
            emit_unit(st, 0, w, cnt, u, Ub, n, f, pnib, plv);
        }
        wave_sync_lds();
        if (valid && w) {
            uint8_t* g = a.out + hdr + p.nbc + (uint64_t) p.b1 * p.b2 * p.b3 + a.offs[gb];
            const uint32_t nw = size / 4;
            for (uint32_t i = ul; i < nw; i += step) {
                const uint32_t v = ((const uint32_t*) st)[i];
                __builtin_memcpy(g + 4 * i, &v, 4);
            }
            for (uint32_t i = 4 * nw + ul; i < size; i += step)
                g[i] = st[i];
        }
        wave_sync_lds();
    }
}

// Residuals of a block column, chunk by chunk: blocks decoded into an LDS tile
// of z rows, each row scanned along z (carried across chunks) and written to
// the output buffer as int32.  ZCCL/src/ZCCL_TypeManager.c:423-517, :906-950.
template <uint32_t BS>
__global__ void __launch_bounds__(256) k3t_decode(Sz3Args a)
{
    using C = Tile3<BS>;
    __shared__ uint4 rt4[BS * BS * C::WZ / 4];
    __shared__ uint32_t s_pay[4][C::BPW][C::PAY / 4];
    __shared__ uint32_t s_carry[BS * BS];
    uint32_t* rt = (uint32_t*) rt4;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t t = part_of_unit(a.parts, a.g.T, blockIdx.x, true);
    const Part3 p = a.parts[t];
    const uint32_t nch = (p.b3 + C::NZ - 1) / C::NZ;
    uint64_t h;
    __builtin_memcpy(&h, a.in + 8ull * t, 8);
    const uint64_t pbase = 8ull * a.g.T + h + (uint64_t) p.b1 * p.b2 * p.b3;
    const unsigned long long o0 = a.offs[p.g0];
    for (uint32_t i = threadIdx.x; i < BS * BS; i += 256)
        s_carry[i] = 0;
    const uint32_t ul = C::BPW > 1 ? lane % C::U : lane;
    const uint32_t step = C::BPW > 1 ? C::U : 64u;
    uint8_t* st = (uint8_t*) s_pay[wv][C::BPW > 1 ? lane / C::U : 0u];
    for (uint32_t ch = 0; ch < nch; ch++) {
        const Chunk3 c = chunk_of<BS>(p, (blockIdx.x - p.c0) * nch + ch);
        for (uint32_t base = wv * C::BPW; base < c.nbz; base += 4 * C::BPW) {
            const uint32_t bzl = base + (C::BPW > 1 ? lane / C::U : 0u);
            const bool valid = bzl < c.nbz;
            const uint32_t gb = c.gcol + bzl;
            const uint32_t word = valid ? a.words[gb] : 0u, w = word >> 26, size = word & kSizeMask;
            const uint32_t ez = valid ? min(BS, c.wz - bzl * BS) : 0u;
            const uint32_t cnt = c.ex * c.ey * ez, sb = (cnt + 7) / 8;
            const uint64_t fo = pbase + ((valid ? a.offs[gb] : o0) - o0);
            const bool inside = fo + size <= a.in_size;
            if (valid && w && !inside && ul == 0)
                raise3(a.status, ZK_ERR_OVERRUN);
            const bool ok = valid && w && inside;
            if (ok) {
                // all of the payload's dword loads in flight before any store
                constexpr uint32_t PS = (C::PAY / 4 + (C::BPW > 1 ? C::U : 64u) - 1) / (C::BPW > 1 ? C::U : 64u);
                const uint8_t* pl = a.in + fo;
                const uint32_t nw = size / 4;
                uint32_t v[PS];
                // unconditional loads (clamped into the payload, or the stream's
                // first bytes when it has no whole dword) stay in flight together
#pragma unroll
                for (uint32_t m = 0; m < PS; m++) {
                    const uint32_t i = min(ul + m * step, nw ? nw - 1 : 0u);
                    __builtin_memcpy(&v[m], nw ? pl + 4 * i : a.in, 4);
                }
#pragma unroll
                for (uint32_t m = 0; m < PS; m++) {
                    const uint32_t i = ul + m * step;
                    if (i < nw)
                        ((uint32_t*) st)[i] = v[m];
                }
                for (uint32_t i = 4 * nw + ul; i < size; i += step)
                    st[i] = pl[i];
            }
            wave_sync_lds();
            for (uint32_t s = 0; s < C::STEPS; s++) {
                const uint32_t u = C::BPW > 1 ? ul : s * 64 + lane;
                const uint32_t n = 4 * u < cnt ? min(4u, cnt - 4 * u) : 0u;
                uint32_t v[4] = {0, 0, 0, 0};
                if (ok && n)
                    accumulate_unit(st - 1, w, cnt, sb, u, v);  // fields start right after the (absent) width byte
                if (n == 4 && cnt == BS * BS * BS) {
                    const uint32_t i = u / (BS * C::UPR), j = (u / C::UPR) % BS, k0 = bzl * BS + (u % C::UPR) * 4;
                    rt4[((i * BS + j) * C::WZ + k0) / 4] = make_uint4(v[0], v[1], v[2], v[3]);
                } else if (n) {
                    const uint32_t yz = c.ey * ez;
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++) {
                        if (k < n) {
                            const uint32_t e = 4 * u + k, i = e / yz, rest = e - i * yz, j = rest / ez;
                            rt[(i * BS + j) * C::WZ + bzl * BS + (rest - j * ez)] = v[k];
                        }
                    }
                }
            }
            wave_sync_lds();
        }
        __syncthreads();
        for (uint32_t row = wv; row < c.ex * c.ey; row += 4) {
            const uint32_t i = row / c.ey, j = row - i * c.ey;
            const uint32_t* src = rt + (i * BS + j) * C::WZ;
            uint32_t carry = s_carry[i * BS + j];
            uint32_t* q = (uint32_t*) a.y + ((uint64_t) (p.ox + c.bx * BS + i) * a.g.d2 + (p.oy + c.by * BS + j)) * a.g.d3 +
                p.oz + c.lz0;
            for (uint32_t k0 = 0; k0 < c.wz; k0 += 64) {
                const uint32_t k = k0 + lane;
                const uint32_t v = k < c.wz ? src[k] : 0u;
                const uint32_t inc = wave_incl_scan32(v) + carry;
                if (k < c.wz)
                    q[k] = inc;
                carry = __shfl(inc, 63, 64);
            }
            if (lane == 0)
                s_carry[i * BS + j] = carry;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ lane compress
// Block side 4.  One lane per block: the lane reads its block's 16 rows of four
// values and the rows one y and one x before them (16-byte loads, consecutive
// blocks of a row in consecutive lanes), quantizes, and takes the differences
// in registers: along z from its own values and the last of the lane below
// (lane 0 of a wave holds the block before the wave's run for that alone),
// along y from the row before, along x from the plane before.  The 64 residuals
// stay in the lane for the width, the wave scans the sizes, the lane encoders
// pack the payload in LDS, and the sizes of all tiles before it in stream
// order give its place: every value is read once (its halo rows come from the
// caches) and quantized 25/16 times.
//
// Two chunk kernels with the quantized values in LDS, a scan of the block sizes
// between them, read and quantized everything twice and took 617 us for a
// 512^3 volume (relative bound 1e-3); this takes 323.  250 without the wait for
// the tiles before one, with four waves a tile: the workgroups that wait finish
// together and the next ones load together.  Twelve waves a tile leave a third
// of the tickets (12 ns each: adds to one address follow one another) and of
// the lookback words: 323 us against 384 with four; 256^3: 58 against 64; but
// 128^3: 28 against 16 (half the compute units idle), hence the line at a wide
// tile for each of 256 units.  Not faster: sums over groups of 64 tiles (326 to
// 690), a workgroup that places a tile after the next one's differences (426).

// Payload bytes of the tiles before tile t, and of those before tile p0 <= t
// (a sub-volume's first), by one wave once t's own `agg` bytes are published:
// the decoupled lookback with four tiles a lane, 256 in a window (512 tiles
// are in flight).  Tiles are numbered by tickets, so those before one have all
// started; the wait is bounded.
__device__ __forceinline__ void places3(unsigned long long* status, uint32_t t, uint32_t p0, unsigned long long agg,
    unsigned long long* err, unsigned long long& at, unsigned long long& part)
{
    const uint32_t lane = threadIdx.x & 63;
    unsigned long long excl = 0, sp = kFlagInc;
    uint32_t spins = 0;
    for (int64_t end = t; end > 0; end -= 256) {
        unsigned long long sum = 0;
        bool inc = false;
        while (true) {
            sum = 0;
            inc = false;
            bool miss = false;
            if (p0)
                sp = st_poll(&status[p0 - 1]);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int64_t i = end - 1 - (int64_t) (4 * lane + c);
                const unsigned long long st = i >= 0 ? st_poll(&status[i]) : kFlagInc;
                // up to the nearest inclusive value, or the first missing one
                const bool use = !inc && !miss;
                miss |= use && (st >> 62) == 0;
                sum += use ? st & kValMask : 0ull;
                inc |= use && (st >> 62) == 2;
            }
            const unsigned long long mm = __ballot(miss), im = __ballot(inc);
            const unsigned long long need = im ? ((im & (~im + 1)) << 1) - 1 : ~0ull;
            if (!(mm & need))
                break;
            if (++spins > kSpinLimit) {
                if (lane == 0)
                    raise3(err, ZK_ERR_SPIN);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        const unsigned long long im = __ballot(inc);
        if (im && lane > (uint32_t) __builtin_ctzll(im))
            sum = 0;
        excl += wave_sum64(sum);
        if (im)
            break;
    }
    if (lane == 0)
        st_publish(&status[t], kFlagInc | ((excl + agg) & kValMask));
    while ((sp >> 62) != 2 && t != p0) {
        if (++spins > kSpinLimit) {
            if (lane == 0)
                raise3(err, ZK_ERR_SPIN);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
        sp = st_poll(&status[p0 - 1]);
    }
    at = excl;
    part = t == p0 ? excl : sp & kValMask;
}

// A wave's payloads (wider runs: a third of the lanes at a time), with the
// reach of the writes past a block of few values.
constexpr uint32_t kLaneBuf3 = 8192, kLaneReach3 = 8 + 4 * 64 + 16;
static_assert(22 * 264 + kLaneReach3 <= kLaneBuf3, "a third of the widest payloads fits");

// Where on: C runs of From values each, of which the first To count, closed up.
template <uint32_t From, uint32_t To, uint32_t C>
__device__ __forceinline__ void close3(uint32_t (&m)[64], bool on)
{
#pragma unroll
    for (uint32_t v = To; v < C * To; v++) {
        const uint32_t there = m[v], moved = m[v / To * From + v % To];
        m[v] = on ? moved : there;
    }
}

// The values of blocks with rows of R values (R < 4: only those, else all) closed
// up along z, then their n rows to a plane along y (n = 1 to 3; 0: no such blocks).
// (The empty asm ends each branch differently: the compiler would otherwise merge
// their last stores into one of a chosen address, and keep m in scratch memory.)
template <uint32_t R>
__device__ __forceinline__ void close_block3(uint32_t (&m)[64], bool rows, bool planes, uint32_t n)
{
    if (R < 4)
        close3<4, R, 16>(m, rows);
    if (n == 1) {
        close3<4 * R, R, 4>(m, rows && planes);
        asm volatile("; y1");
    } else if (n == 2) {
        close3<4 * R, 2 * R, 4>(m, rows && planes);
        asm volatile("; y2");
    } else if (n == 3) {
        close3<4 * R, 3 * R, 4>(m, rows && planes);
        asm volatile("; y3");
    }
}

template <uint32_t W>
__global__ void __launch_bounds__(64 * W, 3) k3l_compress(Sz3Args a)
{
    __shared__ __attribute__((aligned(16))) uint32_t s_buf[W][kLaneBuf3 / 4];
    __shared__ uint32_t s_tot[W], s_ticket;
    __shared__ unsigned long long s_ex, s_part;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (threadIdx.x == 0)
        s_ticket = (uint32_t) atomicAdd(&a.status[2], 1ull);
    __syncthreads();
    const uint32_t t = __builtin_amdgcn_readfirstlane(s_ticket);
    const uint32_t pi = __builtin_amdgcn_readfirstlane(part_of_lane_tile(a.parts, a.g.T, t));
    const Part3 p = a.parts[pi];
    const uint32_t nbp = p.b1 * p.b2 * p.b3;
    // this lane's block; the run's own blocks are those of lanes 1..63
    const int32_t lbs = (int32_t) (kLaneRun3 * (W * (t - p.l0) + wv) + lane) - 1;
    const bool own = lane > 0 && lbs < (int32_t) nbp;
    const uint32_t lb = (uint32_t) min(max(lbs, 0), (int32_t) nbp - 1);
    const uint32_t yz = p.b2 * p.b3;
    const uint32_t bx = lb / yz, rest = lb - bx * yz, by = rest / p.b3, bz = rest - by * p.b3;
    const uint32_t ex = min(4u, p.sx - 4 * bx), ey = min(4u, p.sy - 4 * by), ez = min(4u, p.sz - 4 * bz);
    const bool hx = bx > 0, hy = by > 0, hz = bz > 0;
    const bool edge = ex * ey * ez < 64;
    const bool any_edge = __any(edge), any_z = __any(ez < 4);
    // element offsets of rows -1..3 and values 1..3, clamped into the block and
    // its halo (what a clamped load returns is masked)
    const int32_t d3 = (int32_t) a.g.d3;
    int32_t ro[5];
#pragma unroll
    for (int32_t j = 0; j < 5; j++)
        ro[j] = min(max(j - 1, hy ? -1 : 0), (int32_t) ey - 1) * d3;
    const uint32_t z1 = min(1u, ez - 1), z2 = min(2u, ez - 1), z3 = ez - 1;
    const int64_t sx = (int64_t) a.g.d2 * d3;
    const float* base = a.x + ((int64_t) (p.ox + 4 * bx) * a.g.d2 + (p.oy + 4 * by)) * (int64_t) d3 + p.oz + 4 * bz;
    uint32_t m[64];
    uint32_t ep[16];  // the plane before's differences along z and y
#pragma unroll
    for (uint32_t v = 0; v < 16; v++)
        ep[v] = 0;
    // (the next plane's rows are on their way while one is differenced)
    float4 nx[5];
    auto load = [&](int32_t i) {
        const float* pl = base + min(max(i - 1, hx ? -1 : 0), (int32_t) ex - 1) * sx;
#pragma unroll
        for (uint32_t j = 0; j < 5; j++) {
            const float* q = pl + ro[j];
            if (any_z)
                nx[j] = make_float4(q[0], q[z1], q[z2], q[z3]);
            else
                nx[j] = ldf4(q);
        }
    };
    load(0);
#pragma unroll
    for (int32_t i = 0; i < 5; i++) {
        float4 x[5];
#pragma unroll
        for (uint32_t j = 0; j < 5; j++)
            x[j] = nx[j];
        if (i < 4)
            load(i + 1);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t dp[4] = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t j = 0; j < 5; j++) {
            uint32_t q[4] = {(uint32_t) quant3(x[j].x, a.inv), (uint32_t) quant3(x[j].y, a.inv),
                (uint32_t) quant3(x[j].z, a.inv), (uint32_t) quant3(x[j].w, a.inv)};
            // the last value of the lane below (wave_shr:1), zero at z = 0
            uint32_t qb = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) q[3], 0x138, 0xF, 0xF, false);
            qb = hz ? qb : 0u;
            const bool out = (i == 0 && !hx) || (j == 0 && !hy);
            uint32_t d[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
                d[k] = q[k] - (k ? q[k - 1] : qb);
            if (i == 0 || j == 0) {
#pragma unroll
                for (uint32_t k = 0; k < 4; k++)
                    d[k] = out ? 0u : d[k];
            }
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) {
                if (j > 0) {
                    const uint32_t e = d[k] - dp[k];
                    if (i > 0)
                        m[16 * (i - 1) + 4 * (j - 1) + k] = e - ep[4 * (j - 1) + k];
                    ep[4 * (j - 1) + k] = e;
                }
                dp[k] = d[k];
            }
        }
    }
    uint32_t* buf = s_buf[wv];
    const uint32_t cnt = ex * ey * ez;
    if (any_edge) {
        // blocks at a far edge: their values closed up in order, zeros behind
        // them.  A sub-volume's last blocks along a dim all have the same extent,
        // so each move is one select with its place known (289 x 44 x 41: 17 us, 28 by
        // one walk for every extent, half the lanes at a time through LDS).
        const bool y = ey < 4, z = ez < 4;
        const uint32_t n = __any(y) ? p.sy & 3 : 0u, k = any_z ? p.sz & 3 : 0u;
        close_block3<4>(m, !z, y, n);
        if (k == 1) {
            close_block3<1>(m, z, y, n);
            asm volatile("; z1");
        } else if (k == 2) {
            close_block3<2>(m, z, y, n);
            asm volatile("; z2");
        } else if (k == 3) {
            close_block3<3>(m, z, y, n);
            asm volatile("; z3");
        }
#pragma unroll
        for (uint32_t v = 0; v < 64; v++)
            m[v] = v < cnt ? m[v] : 0u;
    }
    // signs, magnitudes, width and size
    uint32_t s0 = 0, s1 = 0, mx = 0;
#pragma unroll
    for (uint32_t v = 0; v < 64; v++) {
        if (v < 32)
            s0 = __builtin_amdgcn_alignbit(s0, m[v], 31);  // (s0 << 1) | sign of value v
        else
            s1 = __builtin_amdgcn_alignbit(s1, m[v], 31);
        m[v] = mag(m[v]);
        mx = max(mx, m[v]);
    }
    const uint32_t w = own && mx ? 32u - (uint32_t) __clz((int) mx) : 0u;
    const uint32_t size = payload3(w, cnt);
    const uint32_t incl = wave_scan_dpp(size), excl = incl - size;
    const uint32_t wtot = __builtin_amdgcn_readlane(incl, 63);
    if (lane == 0)
        s_tot[wv] = wtot;
    __syncthreads();
    uint32_t woff = 0, total = 0;
#pragma unroll
    for (uint32_t i = 0; i < W; i++) {
        const uint32_t v = s_tot[i];
        woff += i < wv ? v : 0u;
        total += v;
    }
    if (threadIdx.x == 0)
        st_publish(&a.offs[t], (t ? kFlagAgg : kFlagInc) | total);
    const bool one = wtot + kLaneReach3 <= kLaneBuf3;
    uint8_t* dst = nullptr;
    bool fits = false;
    for (uint32_t q = 0; q < (one ? 1u : 3u); q++) {
        // the lanes of this round, their bytes [b0, b1) of the wave's
        const uint32_t b0 = q ? __builtin_amdgcn_readlane(excl, 22 * q) : 0u;
        const uint32_t b1 = one || q == 2 ? wtot : __builtin_amdgcn_readlane(excl, 22 * (q + 1));
        const uint32_t wq = one || lane / 22 == q ? w : 0u, o = excl - b0;
        for (uint32_t i = lane; i < (b1 - b0 + 32 + 15) / 16; i += 64)
            reinterpret_cast<uint4*>(buf)[i] = make_uint4(0, 0, 0, 0);
        wave_sync_lds();
        if (wq) {
            const uint32_t sb[2] = {__builtin_bswap32(s0), __builtin_bswap32(s1)};
            or_words(buf, o, sb);
        }
        const uint32_t hp = o + ((cnt + 7) >> 3);
        if (__any(wq >= 8))
            encode_high_class(buf, hp, wq, m);
        encode_low(buf, hp + cnt * (wq >> 3), wq, m);
        if (q == 0) {
            if (wv == 0) {
                unsigned long long at, part;
                places3(a.offs, t, p.l0, total, a.status, at, part);
                if (lane == 0) {
                    s_ex = at;
                    s_part = part;
                }
            }
            __syncthreads();
            const uint64_t P = 8ull * a.g.T + p.nbc + nbp + s_ex;  // the tile's first payload byte
            fits = P + total <= a.out_cap;
            dst = a.out + P + woff;
        }
        wave_sync_lds();
        if (fits)
            store_wave(buf, dst + b0, b1 - b0);
        wave_sync_lds();
    }
    const uint64_t sub = (uint64_t) p.nbc + s_part;  // sub-volume start after the header
    if (!fits && threadIdx.x == 0)
        raise3(a.status, ZK_ERR_NOSPACE);
    if (own && 8ull * a.g.T + sub + nbp <= a.out_cap)
        a.out[8ull * a.g.T + sub + lb] = (uint8_t) w;
    if (threadIdx.x == 0) {
        if (t == p.l0 && 8ull * (pi + 1) <= a.out_cap)
            __builtin_memcpy(a.out + 8ull * pi, &sub, 8);
        if (t == a.g.nlane - 1) {
            // the last tile ends the stream: if it fits, every tile fits
            const unsigned long long all = 8ull * a.g.T + a.g.nblocks + s_ex + total;
            a.status[0] = all;
            if (a.size_out)
                *a.size_out = all > a.out_cap ? 0ull : all;
        }
    }
}

// ---------------------------------------------------------- lane decompress
// Block side 4.  The 3-D prefix sum of the residuals, in two passes over the
// volume: k3l_decode decodes a row of blocks along z with one lane per block,
// sums along x in registers (kLaneSeg3 blocks one after the other, the last plane
// of the segment kept aside) and along z by wave scans, and writes the integers;
// k3l_ypass sums along y, adds the segments before its own and dequantizes in
// place.  The residuals never reach memory, which the tiled decoder's chunks
// wrote (330 us for a 512^3 volume at a relative bound of 1e-3), the y pass (248)
// and the x pass (238) read and wrote again: 849 us with the sizes.  This takes
// 385: decode 146 (512 MB written; four waves a SIMD, 142 us at its registers'
// limit, 176 with three), y pass 206 (1 GB at 5.2 TB/s, a copy reaches 5.5),
// sizes and kept planes 30.  Volumes with blocks of fewer values (Edges) need 156
// registers to move those to their places: 510^3 962 -> 565 us; in one kernel for
// both 512^3 took 493.

// Bytes of every run of 64 blocks, one lane per run: words[] holds the exclusive
// sums within 256 runs, part_sums[] the groups' sums (scanned by k3_scan_top).
__global__ void __launch_bounds__(256) k3l_sizes(Sz3Args a)
{
    __shared__ uint32_t s_w[4];
    const uint32_t u = blockIdx.x * 256 + threadIdx.x;
    uint32_t sum = 0;
    if (u < a.g.nruns) {
        uint32_t lo = 0, hi = a.g.T;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (a.parts[mid].v0 <= u)
                lo = mid;
            else
                hi = mid;
        }
        const Part3 p = a.parts[lo];
        const uint32_t nz = (p.b3 + 63) / 64, rel = u - p.v0, row = rel / nz, z0 = 64 * (rel - row * nz);
        const uint32_t bx = row / p.b2, by = row - bx * p.b2;
        const uint32_t face = min(4u, p.sx - 4 * bx) * min(4u, p.sy - 4 * by), n = min(64u, p.b3 - z0);
        uint64_t h;
        __builtin_memcpy(&h, a.in + 8ull * lo, 8);
        const uint64_t pos = 8ull * a.g.T + h + (uint64_t) row * p.b3 + z0;
        uint32_t far = 0;
        bool past = false;
#pragma unroll 8
        for (uint32_t i = 0; i < n; i++) {
            const bool in = pos + i < a.in_size;
            uint32_t w = in ? a.in[pos + i] : 0u;
            past |= !in;
            far = max(far, w);
            w = w > 32 ? 0u : w;
            sum += payload3(w, face * min(4u, p.sz - 4 * (z0 + i)));
        }
        if (far > 32)
            raise3(a.status, ZK_ERR_WIDTH);
        if (past)
            raise3(a.status, ZK_ERR_OVERRUN);
    }
    const uint32_t inc = wave_scan_dpp(sum);
    if ((threadIdx.x & 63) == 63)
        s_w[threadIdx.x >> 6] = inc;
    __syncthreads();
    uint32_t pre = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
        pre += w < (threadIdx.x >> 6) ? s_w[w] : 0u;
        all += s_w[w];
    }
    if (u < a.g.nruns)
        a.words[u] = pre + inc - sum;
    if (threadIdx.x == 0)
        a.part_sums[blockIdx.x] = all;
}

// Residuals of a block of width w and cnt values in stream order, its payload at
// byte o of st; those past cnt are garbage.
__device__ __forceinline__ void decode_block3(const uint32_t* st, uint32_t o, uint32_t w, uint32_t cnt, uint32_t (&m)[64])
{
    const uint32_t r = w & 7, B = w >> 3;
    const uint32_t hp = o + ((cnt + 7) >> 3);
    const uint32_t sh[4] = {32 - r, 32 - 2 * r, 32 - 3 * r, 32 - 4 * r};
    uint32_t a = hp + B * cnt;
#pragma unroll
    for (uint32_t g = 0; g < 8; g++, a += r) {
        __builtin_amdgcn_sched_barrier(0);  // group by group: few registers live
        const uint32_t* pg = st + (a >> 2);
        const uint32_t E0 = pg[0], E1 = pg[1], E2 = pg[2];
        const uint32_t e0 = __builtin_bswap32(__builtin_amdgcn_alignbyte(E1, E0, a));
        const uint32_t e1 = __builtin_bswap32(__builtin_amdgcn_alignbyte(E2, E1, a));
        const uint32_t e4 = __builtin_amdgcn_alignbit(e0, e1, sh[3]);
#pragma unroll
        for (uint32_t c = 0; c < 8; c++)
            m[8 * g + c] = __builtin_amdgcn_ubfe(c < 4 ? e0 : e4, sh[c & 3], r);
    }
    if (__any(B == 1)) {
        const uint32_t hb = B == 1 ? 8u : 0u;
#pragma unroll
        for (uint32_t i = 0; i < 16; i++) {
            const uint32_t h = lds_at(st, hp + 4 * i);
#pragma unroll
            for (uint32_t c = 0; c < 4; c++)
                m[4 * i + c] |= __builtin_amdgcn_ubfe(h, 8 * c, hb) << r;
        }
    }
    if (__any(B >= 2)) {
        const uint32_t hm = B >= 4 ? ~0u : B >= 2 ? (1u << (8 * B)) - 1u : 0u;
#pragma unroll
        for (uint32_t e = 0; e < 64; e++) {
            if (e % 4 == 0)
                __builtin_amdgcn_sched_barrier(0);
            m[e] |= (lds_at(st, hp + e * B) & hm) << r;
        }
    }
    const uint32_t s0 = __builtin_bswap32(lds_at(st, o)), s1 = __builtin_bswap32(lds_at(st, o + 4));
#pragma unroll
    for (uint32_t e = 0; e < 64; e++) {
        const uint32_t sg = (uint32_t) __builtin_amdgcn_sbfe((int32_t) (e < 32 ? s0 : s1), 31 - (e & 31), 1);
        m[e] = (m[e] ^ sg) - sg;
    }
}

// Rows of four values of blocks with N rows to a plane, from stream order to
// their places; zeros in the rows the blocks don't have.
template <uint32_t N>
__device__ __forceinline__ void spread_rows3(uint32_t (&m)[64])
{
#pragma unroll
    for (uint32_t v = 64; v-- > 0;) {
        const uint32_t i = v / 16, j = (v / 4) % 4, k = v % 4;
        m[v] = j < N ? m[4 * (i * N + j) + k] : 0u;
    }
}

// A wave's payloads (longer runs: a third of the lanes at a time), with the
// reach of the reads past a block of few values.
constexpr uint32_t kRunBuf3 = 6144, kRunReach3 = 8 + 4 * 64 + 16;
static_assert(22 * 264 + kRunReach3 <= kRunBuf3, "a third of the widest payloads fits");

template <uint32_t W, bool Edges>
__global__ void __launch_bounds__(64 * W, Edges ? 3 : 4) k3l_decode(Sz3Args a)
{
    __shared__ __attribute__((aligned(16))) uint32_t s_buf[W][kRunBuf3 / 4];
    __shared__ uint32_t s_z[2][W][16];
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t* buf = s_buf[wv];
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].d0 <= blockIdx.x)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t pi = __builtin_amdgcn_readfirstlane(lo);
    const Part3 p = a.parts[pi];
    const uint32_t nseg = (p.b1 + kLaneSeg3 - 1) / kLaneSeg3, nz = (p.b3 + 63) / 64;
    const uint32_t by = (blockIdx.x - p.d0) / nseg, seg = blockIdx.x - p.d0 - by * nseg;
    const uint32_t ey = Edges ? min(4u, p.sy - 4 * by) : 4u;
    uint64_t h;
    __builtin_memcpy(&h, a.in + 8ull * pi, 8);
    const uint64_t wpos = 8ull * a.g.T + h, ppos = wpos + (uint64_t) p.b1 * p.b2 * p.b3;
    const unsigned long long o0 = a.part_sums[p.v0 >> 8] + a.words[p.v0];
    const uint32_t bz = 64 * wv + lane;
    const bool own = bz < p.b3;
    const uint32_t ez = Edges && own ? min(4u, p.sz - 4 * bz) : 4u;
    const bool last_z = Edges && (p.sz & 3) && (p.b3 - 1) / 64 == wv;  // some lane's ez is below 4
    uint32_t c[16];  // the plane before, summed along x
#pragma unroll
    for (uint32_t v = 0; v < 16; v++)
        c[v] = 0;
    uint32_t m[64];
    const uint32_t bx1 = min(kLaneSeg3 * (seg + 1), p.b1);
    for (uint32_t bx = kLaneSeg3 * seg; bx < bx1; bx++) {
        const uint32_t ex = Edges ? min(4u, p.sx - 4 * bx) : 4u, cnt = ex * ey * ez;
        const uint32_t row = bx * p.b2 + by, u = p.v0 + row * nz + min(wv, nz - 1);
        const uint64_t wp = wpos + (uint64_t) row * p.b3 + bz;
        uint32_t w = own && wp < a.in_size ? a.in[wp] : 0u;
        w = w > 32 ? 0u : w;
        const uint64_t fo = ppos + (a.part_sums[u >> 8] + a.words[u] - o0);
        const uint32_t size = payload3(w, cnt), incl = wave_scan_dpp(size), excl = incl - size;
        const uint32_t wtot = __builtin_amdgcn_readlane(incl, 63);
        const uint32_t avail = fo < a.in_size ? (uint32_t) min((uint64_t) wtot, a.in_size - fo) : 0u;
        const bool ok = w && excl + size <= avail;
        if (w && !ok)
            raise3(a.status, ZK_ERR_OVERRUN);
        const uint8_t* src = a.in + (fo < a.in_size ? fo : 0);
        const bool one = wtot + kRunReach3 <= kRunBuf3;
#pragma unroll 1
        for (uint32_t q = 0; q < (one ? 1u : 3u); q++) {
            // the lanes of this round, their bytes [b0, b1) of the run's
            const uint32_t b0 = q ? __builtin_amdgcn_readlane(excl, 22 * q) : 0u;
            const uint32_t b1 = min(avail, one || q == 2 ? wtot : __builtin_amdgcn_readlane(excl, 22 * (q + 1)));
            const uint32_t nb = b1 > b0 ? b1 - b0 : 0u;
            wave_sync_lds();
#pragma unroll 1
            for (uint32_t i = lane; i < nb / 16; i += 64) {
                uint4 v;
                __builtin_memcpy(&v, src + b0 + 16 * i, 16);
                reinterpret_cast<uint4*>(buf)[i] = v;
            }
            if (lane < nb % 16)
                ((uint8_t*) buf)[nb / 16 * 16 + lane] = src[b0 + nb / 16 * 16 + lane];
            wave_sync_lds();
            if (one || lane / 22 == q)
                decode_block3(buf, ok ? excl - b0 : 0u, ok ? w : 0u, cnt, m);
        }
        // values of the blocks at a far edge to their places, zeros in the others:
        // the last block along z (one lane) through LDS, ...
        if (last_z) {
            wave_sync_lds();
            if (ez < 4) {
#pragma unroll
                for (uint32_t t = 0; t < 16; t++)
                    reinterpret_cast<uint4*>(buf)[t] = make_uint4(m[4 * t], m[4 * t + 1], m[4 * t + 2], m[4 * t + 3]);
            }
            wave_sync_lds();
        }
        // ... the last along y and x in registers (one extent for the wave)
        if (ey == 1)
            spread_rows3<1>(m);
        else if (ey == 2)
            spread_rows3<2>(m);
        else if (ey == 3)
            spread_rows3<3>(m);
        if (ex < 4) {
#pragma unroll
            for (uint32_t v = 16; v < 64; v++)
                m[v] = v / 16 < ex ? m[v] : 0u;
        }
        if (last_z && ez < 4) {
            const uint32_t n = __builtin_amdgcn_readfirstlane(ez);
            uint32_t e = 0;
#pragma unroll
            for (uint32_t t = 0; t < 16; t++) {
                const bool in = t / 4 < ex && t % 4 < ey;
                m[4 * t] = in ? buf[e] : 0u;
                m[4 * t + 1] = in && n > 1 ? buf[e + 1] : 0u;
                m[4 * t + 2] = in && n > 2 ? buf[e + 2] : 0u;
                m[4 * t + 3] = 0;
                e += in ? n : 0u;
            }
        }
        // along x, from the plane before
#pragma unroll
        for (uint32_t v = 0; v < 64; v++)
            m[v] += v < 16 ? c[v] : m[v - 16];
#pragma unroll
        for (uint32_t v = 0; v < 16; v++)
            c[v] = m[48 + v];
        // along z
        uint32_t tot[16];
#pragma unroll
        for (uint32_t t = 0; t < 16; t++) {
#pragma unroll
            for (uint32_t k = 1; k < 4; k++)
                m[4 * t + k] += m[4 * t + k - 1];
            const uint32_t own_sum = m[4 * t + 3], inc = wave_scan_dpp(own_sum), ex0 = inc - own_sum;
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
                m[4 * t + k] += ex0;
            tot[t] = inc;
        }
        if (W > 1 && nz > 1) {
            if (lane == 63) {
#pragma unroll
                for (uint32_t t = 0; t < 16; t++)
                    s_z[bx & 1][wv][t] = tot[t];
            }
            __syncthreads();
            for (uint32_t i = 0; i < wv; i++) {
#pragma unroll
                for (uint32_t t = 0; t < 16; t++) {
                    const uint32_t before = s_z[bx & 1][i][t];
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++)
                        m[4 * t + k] += before;
                }
            }
        }
        uint32_t* q = (uint32_t*) a.y + ((uint64_t) (p.ox + 4 * bx) * a.g.d2 + (p.oy + 4 * by)) * a.g.d3 + p.oz;
#pragma unroll
        for (uint32_t t = 0; t < 16; t++) {
            if (t / 4 < ex && t % 4 < ey) {
                uint32_t* qr = q + ((uint64_t) (t / 4) * a.g.d2 + t % 4) * a.g.d3;
                if (own && ez == 4) {
                    const uint4 v = make_uint4(m[4 * t], m[4 * t + 1], m[4 * t + 2], m[4 * t + 3]);
                    __builtin_memcpy(__builtin_assume_aligned(qr + 4 * bz, 4), &v, 16);
                } else if (own) {
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++)
                        if (k < ez)
                            qr[4 * bz + k] = m[4 * t + k];
                }
            }
        }
    }
    if (seg + 1 < nseg && own) {
        uint32_t* tail = (uint32_t*) a.offs + p.t0 + ((uint64_t) seg * p.sy + 4 * by) * p.sz + 4 * bz;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
                if (j < ey && k < ez)
                    tail[j * p.sz + k] = m[48 + 4 * j + k];
    }
}

// Last planes of the segments summed over the segments before: one thread per
// (sub-volume, y, z).
__global__ void __launch_bounds__(256) k3l_tails(Sz3Args a)
{
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= a.g.xcols)
        return;
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].xc0 <= col)
            lo = mid;
        else
            hi = mid;
    }
    const Part3 p = a.parts[lo];
    const uint32_t nseg = (p.b1 + kLaneSeg3 - 1) / kLaneSeg3, face = p.sy * p.sz;
    uint32_t* tail = (uint32_t*) a.offs + p.t0 + (col - p.xc0);
    uint32_t run = 0;
    for (uint32_t s = 0; s + 1 < nseg; s++) {
        run += tail[(uint64_t) s * face];
        tail[(uint64_t) s * face] = run;
    }
}

// Along y, with the segments before, and dequantized in place: one thread per
// (sub-volume, block along x, z), its four columns kRowsY3 rows at a time (all
// their loads in flight before the first store; 512^3: 2 rows 386 us, 4 rows 261,
// 8 rows 206, 16 rows 204 with half the waves;
// 8 rows of two columns 216, of one 240, whose kept planes are read more often).
// x' = (float)((double)q * 2 eb), ZCCL/src/ZCCLd_float.c:3030.
constexpr uint32_t kRowsY3 = 8;

__global__ void __launch_bounds__(256) k3l_ypass(Sz3Args a)
{
    const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= a.g.nhcol)
        return;
    uint32_t lo = 0, hi = a.g.T;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.parts[mid].h0 <= col)
            lo = mid;
        else
            hi = mid;
    }
    const Part3 p = a.parts[lo];
    const uint32_t bx = (col - p.h0) / p.sz, z = (col - p.h0) - bx * p.sz, seg = bx / kLaneSeg3;
    const uint32_t ex = min(4u, p.sx - 4 * bx);
    const uint64_t d3 = a.g.d3, plane = (uint64_t) a.g.d2 * d3;
    uint32_t* q = (uint32_t*) a.y + ((uint64_t) (p.ox + 4 * bx) * a.g.d2 + p.oy) * d3 + p.oz + z;
    // (planes past the sub-volume: the last one again, not stored)
    uint64_t po[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
        po[i] = min(i, ex - 1) * plane;
    const uint32_t* tail = (const uint32_t*) a.offs + p.t0 + (uint64_t) (seg ? seg - 1 : 0u) * p.sy * p.sz + z;
    uint32_t run[4] = {0, 0, 0, 0};
    for (uint32_t y0 = 0; y0 < p.sy; y0 += kRowsY3) {
        uint32_t v[kRowsY3][4], t[kRowsY3];
#pragma unroll
        for (uint32_t r = 0; r < kRowsY3; r++) {
            const uint32_t y = min(y0 + r, p.sy - 1);
            t[r] = seg ? tail[(uint64_t) y * p.sz] : 0u;
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
                v[r][i] = q[y * d3 + po[i]];
        }
#pragma unroll
        for (uint32_t r = 0; r < kRowsY3; r++) {
            if (y0 + r < p.sy) {
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) {
                    run[i] += v[r][i] + t[r];
                    if (i < ex)
                        ((float*) q)[(y0 + r) * d3 + po[i]] = (float) __dmul_rn((double) (int32_t) run[i], a.tw);
                }
            }
        }
    }
}

}  // namespace

static hipError_t scan3(const Sz3Args& a, int check_cap, hipStream_t s)
{
    const uint32_t groups = (uint32_t) ceil_div(a.g.nblocks ? a.g.nblocks : 1, kScan3Group);
    hipLaunchKernelGGL(k3_scan_groups, dim3(groups), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_scan_top, dim3(1), dim3(256), 0, s, a, groups, check_cap);
    hipLaunchKernelGGL(k3_scan_apply, dim3(groups), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sz3_table(const Geom3& g, Part3* parts, unsigned long long* status, unsigned long long* clear,
    uint32_t nclear, hipStream_t s)
{
    hipLaunchKernelGGL(k3_table, dim3(1 + std::min(nclear / 256, 255u)), dim3(256), 0, s, g, split3(g), parts, status,
        clear, nclear);
    return hipGetLastError();
}

template <uint32_t BS>
static hipError_t compress_tiled(const Sz3Args& a, hipStream_t s)
{
    hipLaunchKernelGGL(k3t_widths<BS>, dim3(a.g.nunits), dim3(256), 0, s, a);
    hipError_t e = scan3(a, 1, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k3t_encode<BS>, dim3(a.g.nunits), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <uint32_t BS>
static hipError_t decompress_tiled(const Sz3Args& a, hipStream_t s)
{
    hipLaunchKernelGGL(k3_dsizes, dim3((uint32_t) ceil_div(a.g.nblocks, 256)), dim3(256), 0, s, a);
    hipError_t e = scan3(a, 0, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k3t_decode<BS>, dim3(a.g.ncols), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_ypass, dim3((uint32_t) ceil_div(a.g.ycols, 256)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_xpass, dim3((uint32_t) ceil_div(a.g.xcols, 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sz3_compress(const Sz3Args& a, hipStream_t s)
{
    if (a.g.nlane) {
        if (a.g.wlane == kLaneSlim3)
            hipLaunchKernelGGL(k3l_compress<kLaneSlim3>, dim3(a.g.nlane), dim3(64 * kLaneSlim3), 0, s, a);
        else
            hipLaunchKernelGGL(k3l_compress<kLaneWide3>, dim3(a.g.nlane), dim3(64 * kLaneWide3), 0, s, a);
        return hipGetLastError();
    }
    if (a.g.nunits && a.g.Bs == 8)
        return compress_tiled<8>(a, s);
    const uint32_t waves = (uint32_t) ceil_div(a.g.nblocks, 4);
    hipLaunchKernelGGL(k3_widths, dim3(waves), dim3(256), 0, s, a);
    hipError_t e = scan3(a, 1, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k3_encode, dim3(waves), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <bool Edges>
static hipError_t decode_rows3(const Sz3Args& a, hipStream_t s)
{
    if (a.g.wruns == 1)
        hipLaunchKernelGGL((k3l_decode<1, Edges>), dim3(a.g.nrows), dim3(64), 0, s, a);
    else if (a.g.wruns == 2)
        hipLaunchKernelGGL((k3l_decode<2, Edges>), dim3(a.g.nrows), dim3(128), 0, s, a);
    else
        hipLaunchKernelGGL((k3l_decode<kLaneRuns3, Edges>), dim3(a.g.nrows), dim3(64 * kLaneRuns3), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sz3_decompress(const Sz3Args& a, hipStream_t s)
{
    if (a.g.nruns) {
        const uint32_t groups = (uint32_t) ceil_div(a.g.nruns, 256);
        hipLaunchKernelGGL(k3l_sizes, dim3(groups), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k3_scan_top, dim3(1), dim3(256), 0, s, a, groups, 0);
        const hipError_t e = a.g.edges ? decode_rows3<true>(a, s) : decode_rows3<false>(a, s);
        if (e != hipSuccess)
            return e;
        if (a.g.ntail)
            hipLaunchKernelGGL(k3l_tails, dim3((uint32_t) ceil_div(a.g.xcols, 256)), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k3l_ypass, dim3((uint32_t) ceil_div(a.g.nhcol, 256)), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    if (a.g.nunits && a.g.Bs == 4)
        return decompress_tiled<4>(a, s);
    if (a.g.nunits && a.g.Bs == 8)
        return decompress_tiled<8>(a, s);
    hipLaunchKernelGGL(k3_dsizes, dim3((uint32_t) ceil_div(a.g.nblocks, 256)), dim3(256), 0, s, a);
    hipError_t e = scan3(a, 0, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k3_decode, dim3((uint32_t) ceil_div(a.g.nblocks, 4)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_zpass, dim3((uint32_t) ceil_div(a.g.zrows, 4)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_ypass, dim3((uint32_t) ceil_div(a.g.ycols, 256)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k3_xpass, dim3((uint32_t) ceil_div(a.g.xcols, 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace zk
