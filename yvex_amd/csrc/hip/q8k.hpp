// One Q8_K block by one 64-lane wavefront: four values per lane, max-|x| search and the sixteen
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

// x: this lane's four values of the block in memory.
__device__ __forceinline__ void q8k_quantize_block(const float *__restrict__ x, unsigned char *__restrict__ out,
                                                   unsigned lane, int *status)
{
    const float v[4] = {x[0], x[1], x[2], x[3]};
    q8k_quantize_values(v, out, lane, status);
}

}  // namespace yvex
