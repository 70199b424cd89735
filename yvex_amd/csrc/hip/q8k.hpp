// Q8_K blocks by 64-lane wavefronts, one at a time or four: max-|x| search and the sixteen
// 16-value sums across the lanes. Behaviour restated from
// src/backend/cuda/kernels.cu:436-489.
#pragma once
#include "common.hpp"

namespace yvex {

// v: this lane's four values of the block; returns their codes, the block's scale (in every lane) and the lane's codes' sum.
__device__ __forceinline__ unsigned q8k_codes(const float (&v)[4], unsigned lane, float &scale, int &sum, int *status)
{
    // the largest |x| and its first holder's sign: a maximum and a ballot, without permutes through LDS (six of 64-bit
    // keys, one waited for after another, before: 2048 x 4096 values 12.5 -> 10.4 us, 16 384 x 2048 39.5 -> 31.5, 19 x 7168
    // 2.7 -> 2.5)
    unsigned bits[4], largest = 0u;
    bool bad = false;
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        bits[i] = __float_as_uint(v[i]) & 0x7fffffffu;
        bad |= !finite_f32(v[i]);
        largest = bits[i] > largest ? bits[i] : largest;
    }
    if (bad) raise_status(status, 1);
    const unsigned top = wave_max_u32(largest);
    const unsigned sign = __float_as_uint(bits[0] == top ? v[0] : bits[1] == top ? v[1] : bits[2] == top ? v[2] : v[3]) & 0x80000000u;
    const unsigned holder = (unsigned)__builtin_ctzll(__ballot(largest == top));
    const float magnitude = __uint_as_float(top);
    const float signed_max = __uint_as_float(top | (unsigned)__builtin_amdgcn_readlane((int)sign, (int)holder));
    const float inverse = magnitude == 0.0f ? 0.0f : -127.0f / signed_max;
    scale = inverse == 0.0f ? 0.0f : 1.0f / inverse;
    unsigned packed = 0u;
    sum = 0;
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        int q = inverse == 0.0f ? 0 : __float2int_rn(inverse * v[i]);
        q = q > 127 ? 127 : q < -128 ? -128 : q;
        sum += q;
        packed |= ((unsigned)q & 255u) << (8u * i);
    }
    return packed;
}

// out: the block's 292 bytes.
__device__ __forceinline__ void q8k_quantize_values(const float (&v)[4], unsigned char *__restrict__ out,
                                                    unsigned lane, int *status)
{
    float scale;
    int sum;
    const unsigned packed = q8k_codes(v, lane, scale, sum, status);
    if (lane == 0u) *reinterpret_cast<float *>(out) = scale;
    *reinterpret_cast<unsigned *>(out + 4u + lane * 4u) = packed;
    sum = group_sum_i32<4>(sum);   // four lanes hold sixteen consecutive values
    if ((lane & 3u) == 0u) *reinterpret_cast<short *>(out + 260u + (lane >> 2) * 2u) = (short)sum;
}

// Largest value of the 16 lanes of a row, signed and unsigned, in every one of them.
__device__ __forceinline__ int row_max_i32(int v)
{
    int other = dpp_move<0x128, 0xf>(v);             // row_ror 8, 4, 2, 1
    v = other > v ? other : v;
    other = dpp_move<0x124, 0xf>(v);
    v = other > v ? other : v;
    other = dpp_move<0x122, 0xf>(v);
    v = other > v ? other : v;
    other = dpp_move<0x121, 0xf>(v);
    return other > v ? other : v;
}

__device__ __forceinline__ unsigned row_max_u32(unsigned v)
{
    return (unsigned)row_max_i32((int)(v ^ 0x80000000u)) ^ 0x80000000u;
}

// Four blocks by one wavefront, sixteen lanes a block: v[k][i] of lane l of a block is its value 4 (l + 16 k) + i. `live`: the
// block is stored. What bounds a quantizer of long batches is the vector ALU, not memory: a block a wavefront took
// 170 instructions, two divisions, a 64-lane maximum and a row number among them; here four blocks share 160.
// * The largest magnitude and its sign come from the largest of the values as signed and as unsigned integers, of which one
//   is the largest positive value's bits and the other the lowest negative one's (a NaN is above either infinity). Where
//   both are equally far from zero, the block's first decides, looked for in a branch of its own.
// * A code is the low byte of 1.5 * 2^23 + inverse * v, whose addition rounds as a conversion to the nearest does (a
//   magnitude whose inverse is not finite takes conversions and clamps); V_DOT4 adds a lane's codes.
// us a launch, a block a wavefront and four: 2048 x 4096 values 10.4 and 6.5, 2048 x 7168 16.5 and 12.5, 16 384 x 2048 33.3 and 25.5
// (6.8 TB/s; the 18 432 x 2048 of a long batch's layer, part of them out of the caches again, 32: 6.1), 333 x 4096 3.5 and 2.8, 19 x 7168 2.49 and 2.46, one row of 4096 2.5 and 2.2.
__device__ __forceinline__ void q8k_quantize_four(const float (&v)[4][4], unsigned char *__restrict__ out, unsigned lane,
                                                  bool live, int *status)
{
    const unsigned l = lane & 15u;
    int highest = __float_as_int(v[0][0]);
    unsigned lowest = __float_as_uint(v[0][0]);
#pragma unroll
    for (unsigned n = 1; n < 16u; ++n) {
        const int bits = __float_as_int(v[n >> 2][n & 3u]);
        highest = bits > highest ? bits : highest;
        lowest = (unsigned)bits > lowest ? (unsigned)bits : lowest;
    }
    highest = row_max_i32(highest);
    lowest = row_max_u32(lowest);
    const unsigned above = highest > 0 ? (unsigned)highest : 0u, below = lowest & 0x80000000u ? lowest & 0x7fffffffu : 0u;
    const unsigned top = above > below ? above : below;
    unsigned negative = below > above ? 0x80000000u : 0u;
    if (top >= 0x7f800000u && live) raise_status(status, 1);
    if (__ballot(above == below && top != 0u) != 0ull) {
        unsigned first = ~0u;                        // place in the block and sign
#pragma unroll
        for (unsigned n = 16u; n-- > 0u;) {
            const unsigned bits = __float_as_uint(v[n >> 2][n & 3u]);
            if ((bits & 0x7fffffffu) == top) first = (4u * (l + 16u * (n >> 2)) + (n & 3u)) << 1 | bits >> 31;
        }
        first = ~row_max_u32(~first);
        negative = first << 31;
    }
    const float inverse = top == 0u ? 0.0f : -127.0f / __uint_as_float(top | negative);
    const float scale = inverse == 0.0f ? 0.0f : 1.0f / inverse;
    unsigned packed[4];
    if (__ballot(!finite_f32(inverse)) == 0ull) {
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            unsigned code[4];
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) code[i] = __float_as_uint(inverse * v[k][i] + 12582912.0f);
            packed[k] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(code[3], code[2], 0x0c0c0400u),
                                              __builtin_amdgcn_perm(code[1], code[0], 0x0c0c0400u), 0x05040100u);
        }
    } else {
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            packed[k] = 0u;
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) {
                int q = inverse == 0.0f ? 0 : __float2int_rn(inverse * v[k][i]);
                q = q > 127 ? 127 : q < -128 ? -128 : q;
                packed[k] |= ((unsigned)q & 255u) << (8u * i);
            }
        }
    }
    int sums[4];                                     // four lanes hold sixteen consecutive values of a k
#pragma unroll
    for (unsigned k = 0; k < 4u; ++k) sums[k] = group_sum_i32<4>(dot4(packed[k], 0x01010101u, 0));
    if (!live) return;
    if (l == 0u) *reinterpret_cast<float *>(out) = scale;
#pragma unroll
    for (unsigned k = 0; k < 4u; ++k) *reinterpret_cast<unsigned *>(out + 4u + 4u * l + 64u * k) = packed[k];
    // (lane 4 s + k stores the sum of sixteen number s + 4 k)
    const int low = l & 1u ? sums[1] : sums[0], high = l & 1u ? sums[3] : sums[2];
    *reinterpret_cast<short *>(out + 260u + 2u * (l >> 2) + 8u * (l & 3u)) = (short)(l & 2u ? high : low);
}

// x: this lane's four values of the block in memory.
__device__ __forceinline__ void q8k_quantize_block(const float *__restrict__ x, unsigned char *__restrict__ out,
                                                   unsigned lane, int *status)
{
    const float v[4] = {x[0], x[1], x[2], x[3]};
    q8k_quantize_values(v, out, lane, status);
}

}  // namespace yvex
