// IQ2_XXS weight rows against a batch of Q8_K input rows where the matrix is small: 16 weight rows x 16 input rows a
// workgroup on V_MFMA_I32_16X16X32_I8, the row width shared by eight waves (the reference turns its tensor-core kernels on
// from 16 input rows, src/backend/cuda/private.h:461-464).
//
// The row-batch expert kernels give a wave whole rows: 32 rows of 2048 x 7168 are 64 waves on the device, each 28 superblocks
// one behind the other, 33 us for a matrix of 3.8 MB. Here a wave takes every eighth superblock. Lanes load consecutive
// dwords of consecutive rows, a superblock ahead, and the bytes pass through a window of LDS of the wave's own: 8.4 us,
// 1024 x 4096 by 64 rows 22.7 -> 6.8, 4096 x 4096 by 32 23.1 -> 11.3. What is left is the opening (2 us of tables and first
// loads) and the lookups, whose 64 lanes meet on some of the LDS banks.
//
// Arithmetic per 256-value superblock, as the sweeps form it: a K step is one 32-value sub-block of signed codebook levels
// (at most 43), dot = sum of its products (int32, exact), total = sum over the eight sub-blocks of (2 s + 1) dot, and
//     row += double(((0.125 d) d_a) float(total))          superblock by superblock, rounded to float once
// so the bits are theirs. Lane (r, q) holds group q of weight row r's sub-block (B, eight levels: one codebook and one sign
// lookup) and the same eight positions of input row r (A); accumulator i is weight row r against input row 4 q + i.
#include "common.hpp"
#include "launch.hpp"
#include "lds_copy.hpp"
#include "publish.hpp"

namespace yvex {

namespace {

struct DenseIq2Args {
    const unsigned char *encoded;
    unsigned long long row_count, row_bytes;
    unsigned blocks;                         // superblocks (256 columns) per row, even
    const unsigned char *act;                // Q8_K rows, blocks * 292 bytes each
    unsigned long long input_rows;
    float *out;
    int output_bf16;
    int *status;
    Publication publication;
};

constexpr unsigned kIq2Waves = 8u, kIq2Threads = 64u * kIq2Waves;
// the tables, replicated so that the lanes' lookups meet on fewer banks: levels [entry][8], signs {mask, ones} [entry][4]
constexpr unsigned kLevelReplicas = 8u, kSignReplicas = 4u;
constexpr unsigned kSignBase = 256u * kLevelReplicas * 8u, kWindowBase = kSignBase + 128u * kSignReplicas * 16u;
// LDS of a wave: 16 rows' seventeen dwords around a superblock, 16 input rows' codes (272 bytes a row), their scales
constexpr unsigned kRowDwords = 17u, kIq2Act = 16u * kRowDwords * 4u, kIq2ActPitch = 272u;
constexpr unsigned kIq2Scales = kIq2Act + 16u * kIq2ActPitch, kIq2Window = kIq2Scales + 64u;
constexpr unsigned kIq2LdsBytes = kWindowBase + kIq2Waves * kIq2Window;

__global__ __launch_bounds__(kIq2Threads) void dense_iq2_kernel(DenseIq2Args g)
{
    typedef int v4s __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) unsigned char dense_iq2_lds[];
    if (lds_address_of(dense_iq2_lds) != 0u) {   // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(g.status, 2);
        publish_when_last(g.publication, g.status, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
        return;
    }
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned r = lane & 15u, q = lane >> 4;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 16ull, tok0 = (unsigned long long)blockIdx.y * 16ull;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < 16ull ? g.row_count - row0 : 16ull);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < 16ull ? g.input_rows - tok0 : 16ull);
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;
    const unsigned char *const weights = g.encoded + row0 * g.row_bytes, *const acts = g.act + tok0 * act_row_bytes;
    // dwords 64 k + lane of 16 rows x 17 (a ragged edge repeats the last row)
    const unsigned char *weight_at[5];
#pragma unroll
    for (unsigned k = 0; k < 5u; ++k) {
        const unsigned piece = k < 4u ? 64u * k + lane : 256u + r, row = piece / kRowDwords;
        weight_at[k] = weights + (row < rows_here ? row : rows_here - 1u) * g.row_bytes + 4u * (piece - kRowDwords * row);
    }
    InputRows16 inputs(acts, act_row_bytes, toks_here, lane);
    unsigned ahead[5];
    auto request = [&](unsigned sb) {
        // (rows are whole dwords and an even number of superblocks: the aligned dwords around the last one end with the row)
        const unsigned long long w = (sb * 66ull) & ~3ull;
#pragma unroll
        for (unsigned k = 0; k < 5u; ++k) ahead[k] = *reinterpret_cast<const unsigned *>(weight_at[k] + w);
        inputs.request(sb);
    };
    if (wave < g.blocks) request(wave);
    // the tables, while the first superblock is on its way
    if (threadIdx.x < 256u) {
        const uint2 level = iq2_magnitude_of_digits(k_iq2_digits[threadIdx.x]);
#pragma unroll
        for (unsigned k = 0; k < kLevelReplicas; ++k) lds_write_uint2((threadIdx.x * kLevelReplicas + k) * 8u, level);
    } else if (threadIdx.x < 384u) {
        const uint2 mask = iq2_signmask_entry(threadIdx.x - 256u);
#pragma unroll
        for (unsigned k = 0; k < kSignReplicas; ++k)
            lds_write_uint4(kSignBase + ((threadIdx.x - 256u) * kSignReplicas + k) * 16u,
                            make_uint4(mask.x, mask.y, mask.x & 0x01010101u, mask.y & 0x01010101u));
    }
    __syncthreads();
    const unsigned window = kWindowBase + kIq2Window * wave;
    const unsigned w_row = window + r * kRowDwords * 4u, a_row = window + kIq2Act + r * kIq2ActPitch + 8u * q;
    const unsigned level_lane = (lane % kLevelReplicas) * 8u, sign_lane = kSignBase + (lane % kSignReplicas) * 16u;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (unsigned sb = wave; sb < g.blocks; sb += kIq2Waves) {
        // (LDS operations of one wave complete in order)
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) lds_write_u32(window + 256u * k + 4u * lane, ahead[k]);
        lds_write_u32(window + 1024u + 4u * r, ahead[4]);
        inputs.write(window + kIq2Act, kIq2ActPitch, window + kIq2Scales, lane);
        request(sb + kIq2Waves < g.blocks ? sb + kIq2Waves : sb);
        wave_lds_fence();
        // an even superblock starts on a dword (its records two bytes behind), an odd one two bytes behind one
        const unsigned shift = sb & 1u ? 0u : 2u, first = sb & 1u ? 1u : 0u;
        const unsigned head = lds_read_u32(w_row);
        const float d = 0.125f * f16_bits_to_float(sb & 1u ? head >> 16 : head & 0xffffu);
        const uint4 d4 = lds_read_uint4(window + kIq2Scales + 16u * q);
        const float d_a[4] = {__uint_as_float(d4.x), __uint_as_float(d4.y), __uint_as_float(d4.z), __uint_as_float(d4.w)};
        unsigned words[17];
#pragma unroll
        for (unsigned i = 0; i < 17u; ++i) words[i] = lds_read_u32(w_row + 4u * (first + i < 17u ? first + i : 16u));
        int total[4] = {0, 0, 0, 0};
#pragma unroll
        for (unsigned c = 0; c < 8u; ++c) {
            const unsigned grids = __builtin_amdgcn_alignbyte(words[2u * c + 1u], words[2u * c], shift);
            const unsigned aux = __builtin_amdgcn_alignbyte(words[2u * c + 2u], words[2u * c + 1u], shift);
            const uint2 level = lds_read_uint2(((grids >> (8u * q)) & 255u) * (8u * kLevelReplicas) + level_lane);
            const uint4 sign = lds_read_uint4(((aux >> (7u * q)) & 127u) * (16u * kSignReplicas) + sign_lane);
            const unsigned lo = (level.x ^ sign.x) + sign.z, hi = (level.y ^ sign.y) + sign.w;   // (levels are not zero: no carry)
            const uint2 tokens = lds_read_uint2(a_row + 32u * c);
            const long a = (long)(((unsigned long long)tokens.y << 32) | tokens.x), b = (long)(((unsigned long long)hi << 32) | lo);
            const v4s dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4s{0, 0, 0, 0}, 0, 0, 0);
            const int factor = (int)((aux >> 27) | 1u);                       // 2 s + 1
#pragma unroll
            for (int i = 0; i < 4; ++i) total[i] += __mul24(dot[i], factor);   // |dot| < 2^18
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += (double)(d * d_a[i] * (float)total[i]);
        wave_lds_fence();
    }
    __syncthreads();
    double *const partial = reinterpret_cast<double *>(dense_iq2_lds);
    if (wave) {
#pragma unroll
        for (int i = 0; i < 4; ++i) partial[((wave - 1u) * 4u + i) * 64u + lane] = acc[i];
    }
    __syncthreads();
    const unsigned long long row = row0 + r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (wave) break;
        const unsigned long long token = tok0 + 4u * q + i;
        double wide = acc[i];
#pragma unroll
        for (unsigned w = 0; w + 1u < kIq2Waves; ++w) wide += partial[(w * 4u + i) * 64u + lane];
        if (row >= g.row_count || token >= g.input_rows) continue;
        const float sum = (float)wide, value = g.output_bf16 ? bf16_round(sum) : sum;
        if (!finite_f32(value)) raise_status(g.status, 1);
        else store_published(g.publication, g.out + token * g.row_count + row, value);
    }
    publish_when_last(g.publication, g.status, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
}

}  // namespace

// From six input rows on (2048 x 7168 by 4 / 8 rows 7.5 / 11.6 us on the kernel of a few input rows, 8.2 / 8.2 here;
// 1024 x 4096 5.5 / 7.8 and 6.3 / 6.4; 7168 x 2048 7.2 / 11.7 and 8.5 / 8.8) while the tiles are few: the row-batch kernels take the
// same time up to some 2000 of them, this one's grows with them (row-batch kernels and this one: 2048 x 7168 by 32 / 64 / 128 / 256
// rows 33.0 / 33.6 / 36.2 / 44.6 and 8.4 / 14.6 / 26.1 / 49.8; 4096 x 4096 by 16 / 32 / 64 / 128 18.9 / 23.1 / 23.5 / 24.5 and
// 6.9 / 11.3 / 20.0 / 37.0; 7168 x 2048 by 16 / 32 / 64 15.5 / 15.9 / 16.4 and 9.0 / 15.3 / 25.0).
bool iq2_rows_small(uint64_t row_count, uint64_t row_width, uint64_t input_rows)
{
    const uint64_t tiles = (row_count + 15u) / 16u * ((input_rows + 15u) / 16u);
    return input_rows >= 6u && tiles <= (row_width >= 4096u ? 4u : 3u) * (uint64_t)compute_units();
}

int launch_iq2_rows_small(const uint8_t *encoded, uint64_t row_count, uint64_t row_width, uint64_t row_bytes,
                          const void *act_q8k, uint64_t input_rows, float *out, bool output_bf16, int *status,
                          hipStream_t stream, Publisher *publisher)
{
    const uint64_t row_tiles = (row_count + 15u) / 16u, token_tiles = (input_rows + 15u) / 16u;
    if (!row_count || !input_rows || row_width % 512u || row_width / 256u * 66u != row_bytes || row_tiles > 0x7fffffffull ||
        token_tiles > 65535ull)
        return ST_BOUNDS;
    if (((uintptr_t)encoded & 3u) || ((uintptr_t)act_q8k & 3u)) return ST_INVALID_ARG;
    YVEX_ALLOW_DYNAMIC_LDS(dense_iq2_kernel, kIq2LdsBytes);
    // A workgroup has its compute unit to itself, and one that publishes keeps it from the next until its stores are in
    // memory, so a launch ends the operation while it is one round. us a call, published by the launch and behind it:
    // 1024 x 4096 by 64 rows 17.8 and 18.3 (one round), 4096 x 4096 by 32 / 48 / 64 23.6 / 29.1 / 34.2 and 22.8 / 27.4 / 31.8 (two, three,
    // four rounds), 16384 x 4096 by 8 34.3 and 31.7, 2048 x 7168 by 64 / 128 27.1 / 41.4 and 26.3 / 38.8.
    dense_iq2_kernel<<<dim3((unsigned)row_tiles, (unsigned)token_tiles), kIq2Threads, kIq2LdsBytes, stream>>>(
        DenseIq2Args{encoded, row_count, row_bytes, (unsigned)(row_width / 256u), (const unsigned char *)act_q8k, input_rows,
                     out, output_bf16 ? 1 : 0, status, take_publication(publisher, row_tiles * token_tiles, (uint64_t)compute_units())});
    return check_launch("dense_iq2");
}

}  // namespace yvex
