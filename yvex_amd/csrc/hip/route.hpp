// Top-k routing of one row by one wavefront, four experts a lane (experts <= 256). Behaviour restated
// from src/backend/cuda/moe_kernels.cu:180-291 and src/graph/moe.c:539-585.
#pragma once
#include "common.hpp"

namespace yvex {

// What a lane reads of one row: the logits (or the scores a launch before this one has
// published: the float a double-precision score rounds to, what route_row works out from a logit
// otherwise) and the correction biases of experts 4 lane .. 4 lane + 3. The loads depend on
// nothing and sit under no condition on the lane (a lane past the last expert reads the last
// one's again), so a caller can ask for a row's values while it routes the row before: under
// `if (e < experts)` they were issued, and waited for, one expert after another.
struct RouteInputs {
    float value[4], bias[4];
};

__device__ __forceinline__ void route_inputs_load(RouteInputs &in, const float *__restrict__ values,
                                                  const float *__restrict__ bias, unsigned long long row,
                                                  unsigned lane, unsigned experts)
{
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        const unsigned e = lane * 4u + i < experts ? lane * 4u + i : experts - 1u;
        in.value[i] = values[row * experts + e];
        in.bias[i] = bias ? bias[e] : 0.0f;
    }
}

// One row by one wavefront. `published`: in.value holds scores, not logits. `chosen`: the selection for the workgroup's
// own use as well.
__device__ __forceinline__ void route_row(
    const RouteInputs &in, bool published, unsigned long long row, unsigned lane,
    unsigned experts, unsigned topk, int scoring, int normalize, double scaling,
    unsigned long long *__restrict__ selected, float *__restrict__ weights, int *status, unsigned *chosen = nullptr)
{
    float score[4];
    unsigned key[4];       // ordered as the biased scores are; zero: no expert, or one that is taken
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) {
        const unsigned e = lane * 4u + i;
        score[i] = 0.0f;
        key[i] = 0u;
        if (e < experts) {
            if (published) {
                score[i] = in.value[i];
            } else {
                const double s = route_score((double)in.value[i], scoring);
                score[i] = (float)s;      // (a NaN stays a NaN)
            }
            float biased = in.bias[i] + score[i];
            if (!finite_f32(score[i]) || !finite_f32(biased)) raise_status(status, 1);
            biased += 0.0f;   // -0 and +0 must compare equal
            const unsigned bits = __float_as_uint(biased);
            key[i] = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);       // (zero for a NaN only)
        }
    }
    double total = 0.0;
    float picked_score = 0.0f;   // lane r keeps the score of rank r
    for (unsigned rank = 0; rank < topk; ++rank) {
        // The largest key of the wave, then the lowest ordinal that has it: the first lane (a lane's ordinals are
        // below the next lane's), and in the lane the first of its four. No cross-lane permutes through LDS.
        const unsigned first = key[0] > key[1] ? key[0] : key[1], second = key[2] > key[3] ? key[2] : key[3];
        const unsigned top = wave_max_u32(first > second ? first : second);
        const unsigned place = key[0] == top ? 0u : key[1] == top ? 1u : key[2] == top ? 2u : 3u;
        const unsigned long long holders = __ballot(key[0] == top || key[1] == top || key[2] == top || key[3] == top);
        const unsigned winner = (unsigned)__builtin_ctzll(holders);
        const unsigned e = 4u * winner + (unsigned)__builtin_amdgcn_readlane((int)place, (int)winner);
        float s = 0.0f;
#pragma unroll
        for (unsigned i = 0; i < 4u; ++i)
            if (lane * 4u + i == e) {
                s = score[i];
                key[i] = 0u;
            }
        // (the winner's ordinal is the same in every lane: a lane read, no permute through LDS)
        s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), (int)(e >> 2)));
        total += (double)s;                 // rank order, in double (src/graph/moe.c:566-574)
        if (lane == rank) picked_score = s;
        if (lane == 0u) {
            selected[row * topk + rank] = e;
            if (chosen) chosen[rank] = e;
        }
    }
    if (normalize && !(total > 0.0 && total < 1.0e300)) raise_status(status, 1);
    if (lane < topk) {
        double value = (double)picked_score;
        if (normalize) value /= total;
        value *= scaling;
        const float w = (float)value;
        if (!finite_f32(w)) raise_status(status, 1);
        weights[row * topk + lane] = w;
    }
}

}  // namespace yvex
