// IQ2_XXS weights as pairs of int8 limbs for the matrix cores (prefill.hip, rows16.hip): the
// values of three LDS tables, level codes of a codebook entry, sign selectors of a sign field
// and limb words of a scale.
//
// A weight is level * sign * (2 s + 1), up to 43 * 31 = 1333, split into two int8 limbs, value =
// 128 hi + lo with hi in [1, 11] and lo in [-120, 63]. For one scale there are only three levels,
// so the six signed limb values of a group fit two registers and one V_PERM_B32 per four weights
// picks them: the selector byte of a weight is its level code (0..2) plus 4 when it is negative.
#pragma once
#include "common.hpp"

namespace yvex {

// Limb pair of one magnitude: low limb in bits 0-7, high limb in bits 8-15.
__device__ __forceinline__ unsigned iq2_limbs(unsigned level, unsigned factor)
{
    const unsigned magnitude = level * factor;
    unsigned hi = (magnitude + 64u) >> 7;
    if (hi == 0u) hi = 1u;
    const int lo = (int)magnitude - 128 * (int)hi;
    return ((unsigned)lo & 255u) | (hi << 8);
}

// Level codes of a codebook entry: byte l is 0, 1 or 2 for level 8, 25 or 43 of weight l.
__device__ __forceinline__ uint2 iq2_level_codes(unsigned entry)
{
    const uint2 m = iq2_magnitude_entry(entry);
    uint2 codes = make_uint2(0u, 0u);
#pragma unroll
    for (unsigned l = 0; l < 4u; ++l) {
        const unsigned a = (m.x >> (8u * l)) & 255u, b = (m.y >> (8u * l)) & 255u;
        codes.x |= (a == 8u ? 0u : a == 25u ? 1u : 2u) << (8u * l);
        codes.y |= (b == 8u ? 0u : b == 25u ? 1u : 2u) << (8u * l);
    }
    return codes;
}

// Sign selectors of a sign field: byte l is 4 when weight l is negative (7 stored bits + parity).
__device__ __forceinline__ uint2 iq2_sign_selectors(unsigned field)
{
    const uint2 m = iq2_signmask_entry(field);
    return make_uint2(m.x & 0x04040404u, m.y & 0x04040404u);
}

// Limb words of scale s: {+lo, -lo, +hi, -hi}, byte c = limb of level code c.
__device__ __forceinline__ uint4 iq2_limb_words(unsigned scale)
{
    const unsigned factor = 2u * scale + 1u;
    unsigned lo = 0u, hi = 0u;
    const unsigned levels[3] = {8u, 25u, 43u};
#pragma unroll
    for (unsigned c = 0; c < 3u; ++c) {
        const unsigned pair = iq2_limbs(levels[c], factor);
        lo |= (pair & 255u) << (8u * c);
        hi |= (pair >> 8) << (8u * c);
    }
    // byte-wise negation: no limb is zero, so (x ^ 0xff) + 1 never carries; byte 3 stays 0
    const unsigned neg_lo = ((lo ^ 0x00ffffffu) + 0x00010101u) & 0x00ffffffu;
    const unsigned neg_hi = ((hi ^ 0x00ffffffu) + 0x00010101u) & 0x00ffffffu;
    return make_uint4(lo, neg_lo, hi, neg_hi);
}

}  // namespace yvex
