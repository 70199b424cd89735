// Q4_K and Q2_K codes times their sub-block scales, and Q8_K block sums, as int8 limbs for the
// matrix cores (rows_q4k.hip, rows16.hip).
#pragma once
#include "common.hpp"
#include "lds_copy.hpp"

namespace yvex {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Two int8 limbs of sc * nibble for the four nibbles of one dword, value = 8 hi + lo (see
// dense_q4k.hip).
__device__ __forceinline__ void q4k_limbs(unsigned x, unsigned sc, unsigned &lo, unsigned &hi)
{
    const unsigned nibbles = x & 0x0f0f0f0fu;
    const unsigned low = (sc & 7u) * 0x00010001u, high = ((sc >> 3) & 7u) * 0x00010001u;
    lo = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * __builtin_bit_cast(u16x2, low));
    hi = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * __builtin_bit_cast(u16x2, high));
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

// The sixteen int16 block sums as two int8 limbs (value = 128 hi + lo, lo in 0..127), in order.
__device__ __forceinline__ void q2k_bsum_limbs(const uint4 (&b)[2], v4i &lo, v4i &hi)
{
    const unsigned w[8] = {b[0].x, b[0].y, b[0].z, b[0].w, b[1].x, b[1].y, b[1].z, b[1].w};
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        unsigned l = 0u, u = 0u;
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            const unsigned word = w[2u * i + k / 2u];
            const int sum = k % 2u ? (int)word >> 16 : (int)(short)(word & 0xffffu);
            l |= ((unsigned)sum & 127u) << (8u * k);
            u |= ((unsigned)(sum >> 7) & 255u) << (8u * k);
        }
        lo[i] = (int)l;
        hi[i] = (int)u;
    }
}

// The same sums as operands whose products with {m, 8 m, 8 m} add up to m * sum in one sum: the low
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
