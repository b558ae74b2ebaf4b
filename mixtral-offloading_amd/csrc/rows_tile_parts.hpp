// Pieces of the rows kernels of every code width.
#pragma once

#include "gemv_parts.hpp"
#include "rows_tile.hpp"

// The arguments stay where the launch put them: read through a pointer to them, not copied to be indexed.
#define HQQ_KERNARG __attribute__((address_space(4)))
#define HQQ_LDS __attribute__((address_space(3)))

namespace hqq {
namespace rows {

__device__ __forceinline__ f16x2 h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t u2(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }

__device__ __forceinline__ float uniform(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// A load from a base that is the same for the whole wave and a 32-bit byte offset of the lane.  (The sum of a pointer and a loop's
// position is hidden from the compiler, which would keep pointer + lane offset in two vector registers a load.)
template <typename T> __device__ __forceinline__ T load_at(const void *base, uint32_t offset)
{
    asm("" : "+s"(base));
    return *(const T __attribute__((address_space(1))) *)((const char __attribute__((address_space(1))) *)base + offset);
}

// Sixteen bytes a lane from base + offset to LDS byte `to` (the wave's) + 16 * lane, without passing the registers.  (By hand:
// the compiler would wait for the transfer before the next LDS read, whichever half of the buffer that reads.)  It is over
// when the wave has waited for kWaitLoads.
__device__ __forceinline__ void load_to_lds(uint32_t offset, const void *base, uint32_t to)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 : : "v"(offset), "s"(base), "s"(__builtin_amdgcn_readfirstlane(to)) : "memory");
}
constexpr int kWaitLoads = 0x0F70; // vmcnt(0), the other counters left alone

// What this block works on: its member, unit of output rows, part of K and block of batch rows; null: nothing.  Eight consecutive
// blocks run on eight dies: an entry of the list stands for a unit of each, and the batch rows of a unit follow one another, so
// that they find its codes in that die's cache.
__device__ __forceinline__ const Member HQQ_KERNARG *work_of(const Params HQQ_KERNARG &p, int &unit, int &kp, int &col)
{
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    int k = 0;
    while (k + 1 < p.n && p.m[k + 1].first <= slot)
        ++k;
    const Member HQQ_KERNARG &g = p.m[k];
    const int local = slot - g.first, r = local / g.ncol;
    col = local - r * g.ncol;
    const int ru = r * 8 + xcd;
    kp = ru / g.units, unit = ru - kp * g.units;
    return ru < g.units * g.kpb ? &g : nullptr;
}

// c mod columns, inv = floor(2^32 / columns): the quotient estimate is at most 2 short
__device__ __forceinline__ uint32_t mod_cols(uint32_t c, uint32_t cols, uint32_t inv)
{
    c -= __umulhi(c, inv) * cols;
    c -= c >= cols ? cols : 0;
    return c - (c >= cols ? cols : 0);
}

// TE table entries as a lane loaded them -> scales and scale * (C - zero), in pairs.  8-bit tables: a, b the scale's meta (scale,
// zero), sq, zq the bytes, the zero table's own meta as zneg, zoff (C - zero = zoff + code * zneg); each result is rounded once, from
// 32 bits.  fp16 tables: a the scales, b the zeros.  C = kStored: scales and minus zeros, rounded as hqq_dequantize rounds them (zneg:
// minus the meta's scale, zoff: its zero).
constexpr int kStored = -1;
template <bool F16T, int TE, int C, typename Halves, typename Bytes>
__device__ __forceinline__ void decode_tables(const Halves &a, const Halves &b, const Bytes &sq, const Bytes &zq, float zneg, float zoff,
                                              Halves &S, Halves &Z)
{
#pragma unroll
    for (int e = 0; e < TE / 2; ++e) {
        if constexpr (F16T) {
            S[e] = a[e];
            if constexpr (C == kStored) {
                Z[e] = u2(-h2(b[e]));
            } else if constexpr (C == 0) {
                Z[e] = u2(-(h2(b[e]) * h2(a[e])));
            } else {
                f16x2 zv;
#pragma unroll
                for (int o = 0; o < 2; ++o)
                    zv[o] = (f16)(((float)C - (float)h2(b[e])[o]) * (float)h2(a[e])[o]);
                Z[e] = u2(zv);
            }
        } else {
            f16x2 sv, zv;
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                uint32_t sw, zw;
                if constexpr (TE == 8)
                    sw = sq[e >> 1], zw = zq[e >> 1];
                else
                    sw = sq[0], zw = zq[0];
                const int sh = 8 * ((2 * e + o) & 3);
                const float sc = (float)((sw >> sh) & 0xFFu), zc = (float)((zw >> sh) & 0xFFu);
                if constexpr (C == kStored) {
                    sv[o] = (f16)((float)(f16)(sc - (float)h2(b[e])[o]) * (float)h2(a[e])[o]);
                    zv[o] = (f16)((float)(f16)(zc - zoff) * zneg);
                    continue;
                }
                const float d = __builtin_fmaf((float)h2(b[e])[o], -1.0f, sc);
                sv[o] = (f16)__builtin_fmaf(d, (float)h2(a[e])[o], 0.0f);
                zv[o] = (f16)__builtin_fmaf(__builtin_fmaf(zc, zneg, zoff), (float)sv[o], 0.0f);
            }
            S[e] = u2(sv), Z[e] = u2(zv);
        }
    }
}

} // namespace rows
} // namespace hqq
