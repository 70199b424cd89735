// Q4_K and Q2_K codes times their sub-block scales, and Q8_K block sums, as int8 limbs for the
// matrix cores (dense_q4k.hip, rows_q4k.hip, rows16.hip).
#pragma once
#include "common.hpp"
#include "lds_copy.hpp"

namespace yvex {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Two int8 limbs of sc * nibble for the four nibbles of one dword (already shifted so that the
// wanted nibble of every byte sits in its low four bits), value = 8 hi + lo. The 6-bit scale is
// split as sc = 8 high + low with both parts in 0..7: a limb byte nibble * part is at most 105, so
// one 16-bit lane multiply scales two bytes at once without a carry from one into the next.
__device__ __forceinline__ void q4k_limbs(unsigned x, unsigned short low, unsigned short high, unsigned &lo, unsigned &hi)
{
    const unsigned nibbles = x & 0x0f0f0f0fu;
    lo = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * u16x2{low, low});
    hi = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * u16x2{high, high});
}

// Pair sums of the 16 int16 block sums as two int8 limbs (value = 128 hi + lo, lo in 0..127).
__device__ __forceinline__ void q4k_bsum_limbs(const uint4 (&b)[2], uint2 &lo, uint2 &hi)
{
    const unsigned w[8] = {b[0].x, b[0].y, b[0].z, b[0].w, b[1].x, b[1].y, b[1].z, b[1].w};
    unsigned l[2] = {0u, 0u}, u[2] = {0u, 0u};
#pragma unroll
    for (unsigned s = 0; s < 8u; ++s) {
        const int pair = (int)(short)(w[s] & 0xffffu) + ((int)w[s] >> 16);
        l[s >> 2] |= ((unsigned)pair & 127u) << (8u * (s & 3u));
        u[s >> 2] |= ((unsigned)(pair >> 7) & 255u) << (8u * (s & 3u));
    }
    lo = make_uint2(l[0], l[1]);
    hi = make_uint2(u[0], u[1]);
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
static_assert(sizeof(f16x8) == 16, "an operand of a matrix instruction");

// Minimum terms on the f16 matrix instructions. A minimum is at most 63 and a sum of sixteen int8 values at
// most 2048 in magnitude, both whole numbers that f16 holds; their products and sums stay below 2^21, so the float a matrix
// core publishes is the exact sum, with nothing to join or convert.

// Eight bytes (at most 127) as f16: the byte below the high byte of 1024.0 is 1024 + byte.
__device__ __forceinline__ f16x8 bytes_to_f16(unsigned first, unsigned second)
{
    const f16x2 bias = {(_Float16)1024.0f, (_Float16)1024.0f};
    f16x2 pair[4];
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        const unsigned bits = __builtin_amdgcn_perm(0x64646464u, i < 2u ? first : second, i & 1u ? 0x04030402u : 0x04010400u);
        pair[i] = __builtin_bit_cast(f16x2, bits) - bias;
    }
    return f16x8{pair[0][0], pair[0][1], pair[1][0], pair[1][1], pair[2][0], pair[2][1], pair[3][0], pair[3][1]};
}

// Four bytes (at most 127) as f16, each twice.
__device__ __forceinline__ f16x8 byte_pairs_to_f16(unsigned bytes)
{
    const f16x2 bias = {(_Float16)1024.0f, (_Float16)1024.0f};
    f16x2 pair[4];
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        const unsigned bits = __builtin_amdgcn_perm(0x64646464u, bytes, 0x04000400u + 0x00010001u * i);
        pair[i] = __builtin_bit_cast(f16x2, bits) - bias;
    }
    return f16x8{pair[0][0], pair[0][1], pair[1][0], pair[1][1], pair[2][0], pair[2][1], pair[3][0], pair[3][1]};
}

// Q4_K: a minimum per 32 values. The sums of two neighbours (at most 4096 in magnitude) in two parts f16 holds, each on
// half of the K step: multiples of 32 for lanes of half 0, what is left for those of half 1. (dense_q4k.hip, whose lanes hold all
// sixteen sums anyway; on the operands below its tiles are 2 to 3 % slower.)
__device__ __forceinline__ f16x8 q4k_bsum_operand(const uint4 &b0, const uint4 &b1, unsigned half)
{
    const unsigned w[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
    const int part = half ? 31 : ~31;
    f16x8 out;
#pragma unroll
    for (unsigned s = 0; s < 8u; ++s) {
        const int pair = (int)(short)(w[s] & 0xffffu) + ((int)w[s] >> 16);
        out[s] = (_Float16)(short)(pair & part);
    }
    return out;
}

// Eight of a block's sums of sixteen values: a K step of sixteen on both halves of a wave. Q2_K has a minimum for each, Q4_K one for
// two (rows_q4k.hip: 453 -> 423 vector instructions a superblock and wave of 64 tokens against the operand above).
__device__ __forceinline__ f16x8 bsum_operand(const uint4 &b)
{
    const unsigned w[4] = {b.x, b.y, b.z, b.w};
    f16x8 out;
#pragma unroll
    for (unsigned s = 0; s < 4u; ++s) {
        out[2u * s] = (_Float16)(short)(w[s] & 0xffffu);
        out[2u * s + 1u] = (_Float16)(short)(w[s] >> 16);
    }
    return out;
}

// The sixteen int16 block sums as operands whose products with {m, 8 m, 8 m} add up to m * sum in one sum: the low
// three bits, and the rest (-256 .. 254) in two halves that fit int8.
__device__ __forceinline__ void q2k_bsum_pieces(const uint4 (&b)[2], v4i (&piece)[3])
{
    const unsigned w[8] = {b[0].x, b[0].y, b[0].z, b[0].w, b[1].x, b[1].y, b[1].z, b[1].w};
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        unsigned low = 0u, half = 0u, other = 0u;
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            const unsigned word = w[2u * i + k / 2u];
            const int sum = k % 2u ? (int)word >> 16 : (int)(short)(word & 0xffffu);
            const int rest = sum >> 3, first = rest >> 1;
            low |= ((unsigned)sum & 7u) << (8u * k);
            half |= ((unsigned)first & 255u) << (8u * k);
            other |= ((unsigned)(rest - first) & 255u) << (8u * k);
        }
        piece[0][i] = (int)low;
        piece[1][i] = (int)half;
        piece[2][i] = (int)other;
    }
}

// Four Q2_K codes (bits 0-1 of each byte) times their 4-bit scale, at most 45: one int8 limb. Two
// bytes share a 16-bit lane, the products stay inside their bytes.
__device__ __forceinline__ unsigned q2k_limb(unsigned codes, unsigned sc)
{
    const u16x2 twice = __builtin_bit_cast(u16x2, sc * 0x00010001u);
    return __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, codes & 0x03030303u) * twice);
}

}  // namespace yvex
