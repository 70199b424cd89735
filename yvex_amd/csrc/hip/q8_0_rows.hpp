// Q8_0 weight rows against a few input rows that a workgroup of sixteen waves quantizes for itself: the codes and scales
// of the input rows' Q8_K blocks stay in LDS, a wave multiplies one weight row, and the launch that would have
// quantized them, or that this work rides along with, is saved. At decode width a launch costs more than what it does: a
// kernel that copies one word takes 2.3 us behind itself and 3.5 to 4 behind kernels that have gone through the caches.
//
// The arithmetic is matvec_block_kernel's, operation for operation and in its order: same bits.
#pragma once
#include "common.hpp"
#include "q8k.hpp"

namespace yvex {

constexpr unsigned kHeldWaves = 16u, kHeldThreads = 64u * kHeldWaves;
constexpr unsigned kHeldBlock = 272u;          // a Q8_K block in LDS: 256 codes, the scale, padding to 16 bytes

__host__ __device__ __forceinline__ constexpr unsigned long long held_bytes(unsigned long long input_rows,
                                                                            unsigned long long blocks)
{
    return input_rows * blocks * kHeldBlock;
}

__device__ __forceinline__ void hold_block(const float (&v)[4], unsigned char *held, unsigned lane, int *status)
{
    float scale;
    int sum;
    const unsigned packed = q8k_codes(v, lane, scale, sum, status);
    *reinterpret_cast<unsigned *>(held + 4u * lane) = packed;
    if (lane == 0u) *reinterpret_cast<float *>(held + 256u) = scale;
}

// The bytes of one 34-byte block as they are loaded (unit_load's scheme for rows on even addresses: the aligned dwords
// that hold the codes, and one beside them for the rest); shifted into place only when they are used.
struct HeldBlockBytes {
    uint4 lo, hi;
    unsigned tail;
};

__device__ __forceinline__ void held_request(const unsigned char *row, unsigned u, HeldBlockBytes &raw)
{
    const unsigned char *b = row + u * 34u + 2u;
    const unsigned shift = (unsigned)(unsigned long long)b & 3u;       // 0 or 2
    const unsigned char *at = b - shift;
    raw.lo = *reinterpret_cast<const uint4 *>(at);
    raw.hi = *reinterpret_cast<const uint4 *>(at + 16u);
    if (shift == 0u && u == 0u) raw.tail = (unsigned)*reinterpret_cast<const unsigned short *>(b - 2u) << 16;
    else raw.tail = *reinterpret_cast<const unsigned *>(shift ? at + 32u : at - 4u);
}

// U chunks of 64 blocks of a weight row on their way.
template <int U>
__device__ __forceinline__ void held_request_row(const unsigned char *row, unsigned base, unsigned units, unsigned lane,
                                                 HeldBlockBytes (&raw)[U])
{
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const unsigned u = base + 64u * j + lane;
        held_request(row, u < units ? u : units - 1u, raw[j]);
    }
}

// Those chunks against T held input rows; acc: the lane's part of the row sums.
template <int T, int U>
__device__ __forceinline__ void held_multiply(const unsigned char *row, unsigned base, unsigned units, unsigned lane,
                                              const HeldBlockBytes (&raw)[U], const unsigned char *held,
                                              unsigned held_row_bytes, double (&acc)[T])
{
#pragma unroll
    for (int j = 0; j < U; ++j) {
        if (j > 0 && base + 64u * j >= units) break;          // wave-uniform: no chunk here
        const unsigned u = base + 64u * j + lane;
        const bool live = u < units;
        const unsigned uu = live ? u : units - 1u;
        const unsigned shift = (unsigned)(unsigned long long)(row + uu * 34u + 2u) & 3u;
        const unsigned words[9] = {raw[j].lo.x, raw[j].lo.y, raw[j].lo.z, raw[j].lo.w, raw[j].hi.x,
                                   raw[j].hi.y, raw[j].hi.z, raw[j].hi.w, raw[j].tail};
        unsigned codes[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) codes[i] = __builtin_amdgcn_alignbyte(words[i + 1], words[i], shift);
        const float d = f16_bits_to_float((unsigned short)(shift ? raw[j].lo.x & 0xffffu : raw[j].tail >> 16));
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const unsigned char *block = held + t * held_row_bytes + (uu >> 3) * kHeldBlock;
            const uint4 first = *reinterpret_cast<const uint4 *>(block + 32u * (uu & 7u));
            const uint4 second = *reinterpret_cast<const uint4 *>(block + 32u * (uu & 7u) + 16u);
            const unsigned values[8] = {first.x, first.y, first.z, first.w, second.x, second.y, second.z, second.w};
            int dot = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = dot4(codes[i], values[i], dot);
            // the chain through a superblock's eight blocks, a lane each (matvec_block_kernel)
            const float scale = d * *reinterpret_cast<const float *>(block + 256u), value = (float)dot;
            float total = __builtin_fmaf(scale, value, 0.0f);
#pragma unroll
            for (int step = 1; step < 8; ++step) {
                const float before = __int_as_float(
                    __builtin_amdgcn_update_dpp(0, __float_as_int(total), 0x111, 0xf, 0xf, false));   // row_shr:1
                total = __builtin_fmaf(scale, value, before);
            }
            acc[t] += (double)(live && (lane & 7u) == 7u ? total : 0.0f);
        }
    }
}

// Weight row `row` against the T held rows, its first chunks already requested; the sums in every lane.
template <int T, int U>
__device__ __forceinline__ void held_row(const unsigned char *row, unsigned units, unsigned lane, HeldBlockBytes (&raw)[U],
                                         const unsigned char *held, unsigned held_row_bytes, float (&sums)[T])
{
    double acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = 0.0;
    held_multiply<T, U>(row, 0u, units, lane, raw, held, held_row_bytes, acc);
    for (unsigned base = 64u * U; base < units; base += 64u * U) {
        held_request_row<U>(row, base, units, lane, raw);
        held_multiply<T, U>(row, base, units, lane, raw, held, held_row_bytes, acc);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        sums[t] = (float)wave_sum_f64(acc[t]);
    }
}

// The rows [wave of the launch's `groups` workgroups] of up to two matrices (the second's rows count on behind the first's)
// against T held rows, with the first row's bytes requested ahead by the caller's `hold`, which quantizes the input rows.
template <int T, int U, typename At, typename Hold, typename Publish>
__device__ __forceinline__ void held_rows(unsigned long long rows, unsigned group, unsigned groups, unsigned units,
                                          unsigned char *held, At at, Hold hold, Publish publish)
{
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    unsigned long long row = (unsigned long long)group * kHeldWaves + wave;
    HeldBlockBytes raw[U];
    const unsigned char *from = at(row < rows ? row : rows - 1ull);
    hold.request(wave);
    held_request_row<U>(from, 0u, units, lane, raw);
    hold.finish(wave, held);
    __syncthreads();
    while (row < rows) {
        float sums[T];
        held_row<T, U>(from, units, lane, raw, held, (units >> 3) * kHeldBlock, sums);
        if (lane == 0u) {
#pragma unroll
            for (int t = 0; t < T; ++t) publish((unsigned)t, row, sums[t]);
        }
        row += (unsigned long long)groups * kHeldWaves;
        if (row >= rows) break;
        from = at(row);
        held_request_row<U>(from, 0u, units, lane, raw);
    }
}

// Input rows as they lie in memory.
struct HoldRows {
    const float *input;
    unsigned long long stride;
    unsigned blocks, tasks;          // Q8_K blocks a row, and of all rows
    int *status;
    float v[4];
    __device__ __forceinline__ void request(unsigned task)
    {
        const unsigned here = task < tasks ? task : tasks - 1u, in = here / blocks;
        const float *x = input + in * stride + 256u * (here - in * blocks) + 4u * (threadIdx.x & 63u);
#pragma unroll
        for (unsigned i = 0; i < 4u; ++i) v[i] = x[i];
    }
    __device__ __forceinline__ void finish(unsigned wave, unsigned char *held)
    {
        for (unsigned task = wave; task < tasks; task += kHeldWaves) {
            hold_block(v, held + task * kHeldBlock, threadIdx.x & 63u, status);
            if (task + kHeldWaves < tasks) request(task + kHeldWaves);
        }
    }
};

}  // namespace yvex
