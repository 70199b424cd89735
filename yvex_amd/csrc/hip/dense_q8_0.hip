// Q8_0 weight rows against a batch of Q8_K input rows on the int8 matrix cores: the dense
// projection at prefill width (the reference turns its tensor-core kernels on from 16 input rows
// for every format that takes Q8 activations, src/backend/cuda/private.h:461-464,
// src/backend/cuda/qtype.c:252-255).
//
// Arithmetic, as the reference's primitive forms it for one 256-value superblock
// (src/backend/cuda/kernel_primitives.h:342-359) and the CPU path adds a row's superblocks
// (src/gguf/quant_compute.c:152-172):
//     dot_b = sum_i q_i * a_i                              (int32, exact: one K step of V_MFMA_I32_32X32X32_I8)
//     total = fmaf(d_b * d_a, float(dot_b), total)         b = 0 .. 7 in order, floats, from zero
//     row  += double(total)                                superblock by superblock, rounded to float once
// A block has a scale of its own, so every matrix instruction starts anew and its sixteen
// results a lane are brought to float and chained on the vector ALU (two instructions each); the products of the
// scales come from the matrix cores (scale_products; the 16 x 16 tiles multiply).
//
// A workgroup owns 32 weight rows x 32 input rows; its four waves take every fourth superblock
// (eight blocks, 272 bytes a row) and their partial tiles are added in wave order, so results do
// not depend on timing. The input rows are the A operand and the weight rows the B operand: lane (r, h) holds bytes
// 16 h .. 16 h + 15 of input row r's block and
// of weight row r's block, and accumulator i of that lane is weight row r against input row
// 8 (i / 4) + 4 h + i % 4, so a block's scale is one value a lane. Blocks start on 2-byte
// boundaries (34 bytes each): the codes of an even block are read as five aligned dwords and
// shifted into place, those of an odd block are dword-aligned as they lie.
#include "common.hpp"
#include "launch.hpp"
#include "lds_copy.hpp"
#include "publish.hpp"

namespace yvex {

namespace {

struct DenseQ80Args {
    const unsigned char *encoded;
    unsigned long long row_count, row_bytes;
    unsigned blocks;                         // superblocks (256 columns) per row
    const unsigned char *act;                // Q8_K rows, blocks * 292 bytes each
    unsigned long long input_rows;
    const float *additive;
    float *out;
    unsigned long long out_stride;
    int output_bf16;
    int *status;
    const unsigned char *encoded_second;     // a second matrix of the same shape (blockIdx.z = 1), or null
    float *out_second;
    Publication publication;
};

__device__ __forceinline__ void choose_matrix(DenseQ80Args &g)
{
    if (blockIdx.z) {
        g.encoded = g.encoded_second;
        g.out = g.out_second;
    }
}

// float(sum) of a matrix instruction's sums without a conversion each. The instruction starts from the bits of
// 1 / (2 pi) as an integer instead of zero, which its encoding holds as an inline constant; the sums of one
// block are below 2^20 and the constant's mantissa is 2 292 099 above its binade's first, 6 096 508 below its last, so the
// bits of a result are those of the float kStart + 2^-26 sum, and one multiply-add, which the vector ALU issues at twice the
// rate of a conversion, leaves float(sum) exactly: 2^26 (kStart + 2^-26 sum) - 2^26 kStart. (Not a subtraction with the
// 2^26 left to a block's scale: that scale times a row's reaches neither as far up nor as far down as a float's range then.)
constexpr unsigned kStartBits = 0x3e22f983u;

// The 2^26, in a vector register: the multiply-add then holds the 2^26 kStart in its encoding. 4096 x 4096 by 2048 rows on the
// 128 x 128 tiles 124.8 us so, 127.9 with both in registers, 125.3 with the factor in the encoding (means of 18 runs).
__device__ __forceinline__ float sum_scale()
{
    float scale = 67108864.0f;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(scale));
#endif
    return scale;
}

// The block's sums from kStartBits on, as floats. Written out because the compiler puts a start other than zero into
// sixteen registers. The results are in their registers behind the last wait states (eleven for a matrix
// instruction of eight passes), so that whatever follows may read or reuse them; the first ones cover operands that vector
// instructions have just written.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ v16f block_sums(v4i tokens, v4i codes)
{
    v16f dot;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("s_nop 1\n\t"
        "v_mfma_i32_32x32x32_i8 %0, %1, %2, 0.15915494\n\t"
        "s_nop 12"
        : "=&v"(dot) : "v"(tokens), "v"(codes));
#else
    (void)tokens;
    (void)codes;
    for (int i = 0; i < 16; ++i) dot[i] = 0.0f;
#endif
    return dot;
}
#pragma clang diagnostic pop

__device__ __forceinline__ uint4 read16(unsigned address)
{
    const v4i v = lds_read_v4i(address);
    return make_uint4((unsigned)v[0], (unsigned)v[1], (unsigned)v[2], (unsigned)v[3]);
}

constexpr unsigned kStagedPitch = 272u;

// The products d_b * d_a of two neighbouring blocks where their sums are, sixteen of the first and sixteen of the second: two outer
// products on one V_MFMA_F32_32X32X1_2B_F32, the bits of sixteen multiplications a block. Lane (r, h) brings input row r's
// scale and that of weight row r's block h of the two. It takes 64 cycles of the matrix cores for 128 of the vector ALU,
// eleven LDS reads a superblock and sixteen registers (a V_MFMA_F32_32X32X2_F32 a block, 64 cycles for 64, had made the 128 x 128
// tiles 6 % slower). 450 -> 314 vector instructions a superblock on the 128 x 128 tiles, 466 -> 333 on the 32 x 32 ones. us a call
// before and after, quantization and completion included: 4096 x 4096 by 40 / 96 / 200 / 333 / 512 / 2048 rows 25.9 / 29.4 / 43.1 / 50.8 /
// 53.8 / 133.5 -> 23.6 / 27.8 / 36.3 / 47.5 / 50.8 / 126.8, 7168 x 2048 by 700 67 -> 59, 129 280 x 7168 by 3 with its selection
// 216 -> 208. The kernels that call this are bounded to 256 registers: with more to spend the compiler keeps the products in
// accumulation registers and moves each out.
__device__ __forceinline__ v32f scale_products(float d_a, unsigned scale_bits)
{
    v32f zero;
#pragma unroll
    for (int i = 0; i < 32; ++i) zero[i] = 0.0f;
    return __builtin_amdgcn_mfma_f32_32x32x1f32(d_a, f16_bits_to_float(scale_bits), zero, 0, 0, 0);
}

// One superblock out of LDS: lane (r, h)'s weight row at `w_row` (272 bytes), its input row's codes, of which it holds
// sixteen bytes a block, at `a_row`, and that input row's scale, the same for both halves, at `scale_at` (scale_products takes it to
// the lanes that hold the row's sums).
__device__ __forceinline__ void q80_superblock(unsigned w_row, unsigned a_row, unsigned scale_at, unsigned h, float scale, double (&acc)[16])
{
    float total[16];
    uint4 lo[2], hi[2] = {};
    v4i tokens[2];
    auto read_block = [&](unsigned c) {
        const unsigned slot = c % 2u;
        const unsigned start_at = c % 2u == 0u ? 34u * c : 34u * c + 2u;      // the lane's window: + 16 h
        lo[slot] = read16(w_row + 16u * h + (start_at & ~15u));
        // (an even block's window is 20 bytes, an odd block's 16: what of it lies in the next piece)
        const unsigned behind = w_row + 16u * h + (start_at & ~15u) + 16u, words = (start_at & 15u) / 4u + (c % 2u == 0u ? 1u : 0u);
        if (words == 1u) hi[slot].x = lds_read_u32(behind);
        else if (words == 2u) {
            const uint2 two = lds_read_uint2(behind);
            hi[slot].x = two.x;
            hi[slot].y = two.y;
        } else if (words) hi[slot] = read16(behind);
        tokens[slot] = lds_read_v4i(a_row + 32u * c);
    };
    auto codes_of = [&](unsigned c) -> v4i {
        const unsigned slot = c % 2u;
        const unsigned start_at = c % 2u == 0u ? 34u * c : 34u * c + 2u, at = (start_at & 15u) / 4u;
        const unsigned q[8] = {lo[slot].x, lo[slot].y, lo[slot].z, lo[slot].w,
                               hi[slot].x, hi[slot].y, hi[slot].z, hi[slot].w};
        v4i codes;
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j)
            codes[j] = c % 2u == 0u ? (int)__builtin_amdgcn_alignbyte(q[at + j + 1u], q[at + j], 2u) : (int)q[at + j];
        return codes;
    };
    read_block(0u);
    const float d_a = __uint_as_float(lds_read_u32(scale_at));
    unsigned scale_bits = lds_read_u16(w_row + 34u * h);
    v32f step;
#pragma unroll
    for (unsigned c = 0; c < 8u; ++c) {
        const v4i codes = codes_of(c);
        if (c + 1u < 8u) read_block(c + 1u);
        __builtin_amdgcn_sched_barrier(0);
        const v16f dot = block_sums(tokens[c % 2u], codes);
        __builtin_amdgcn_sched_barrier(0);
        if (c % 2u == 0u) {
            step = scale_products(d_a, scale_bits);
            if (c < 6u) scale_bits = lds_read_u16(w_row + 34u * (c + 2u + h));
        }
        float value[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) value[i] = __builtin_fmaf(dot[i], scale, -67108864.0f * __uint_as_float(kStartBits));
        if (c % 2u == 0u) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float both = step[16u * (c % 2u) + i];
            total[i] = c == 0u ? both * value[i] : __builtin_fmaf(both, value[i], total[i]);
        }
        // (the compiler would sink all of it behind the last block, and keep every block's sums until then)
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(total[i]));
#endif
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] += (double)total[i];
}

constexpr unsigned kPlainWaves = 4u;
// LDS of a wave: its 32 weight rows' superblock, its 32 input rows' codes (both 272 bytes a row), their scales
constexpr unsigned kPlainAct = 32u * kStagedPitch, kPlainScales = 2u * kPlainAct, kPlainWindow = kPlainScales + 128u;
constexpr unsigned kPlainLdsBytes = kPlainWaves * kPlainWindow;        // (the partial tiles take their place in the end)

// 32 weight rows x 32 input rows a workgroup, a superblock in four a wave. Every lane used to load its own pieces of 16
// bytes, 33 instructions of 64 cache lines a superblock at two cycles a line: waves stood before the memory pipeline half
// their time and the vector ALU was 19 % busy. The lanes of a load take consecutive pieces of consecutive rows now, a
// superblock ahead, and the bytes pass through a window of LDS of the wave's own. 4096 x 4096 by 32 / 96 rows
// 17.0 / 25.6 -> 14.2 / 18.3 us, 2048 x 7168 by 32 / 256 21.2 / 34.1 -> 18.3 / 25.9. (Eight waves, two superblocks each, are
// 1 to 1.5 us behind: the reduction is longer and the device no fuller.)
__global__ __launch_bounds__(64 * kPlainWaves, 2) void dense_q8_0_kernel(DenseQ80Args g)
{
    extern __shared__ __align__(16) unsigned char dense_q8_0_plain_lds[];
    if (lds_address_of(dense_q8_0_plain_lds) != 0u) {   // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(g.status, 2);
        return;
    }
    choose_matrix(g);
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned r = lane & 31u, h = lane >> 5;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 32ull;
    const unsigned long long tok0 = (unsigned long long)blockIdx.y * 32ull;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < 32ull ? g.row_count - row0 : 32ull);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < 32ull ? g.input_rows - tok0 : 32ull);
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;
    const unsigned char *const weights = g.encoded + row0 * g.row_bytes, *const acts = g.act + tok0 * act_row_bytes;
    // pieces 64 k + lane of 32 rows x 17 and of 32 rows x 16 (a ragged edge repeats the last row)
    const unsigned char *weight_at[9], *act_at[8];
#pragma unroll
    for (unsigned k = 0; k < 9u; ++k) {
        const unsigned piece = k < 8u ? 64u * k + lane : 512u + r, row = piece / 17u;
        weight_at[k] = weights + (row < rows_here ? row : rows_here - 1u) * g.row_bytes + 16u * (piece - 17u * row);
    }
#pragma unroll
    for (unsigned k = 0; k < 8u; ++k) {
        const unsigned row = 4u * k + (lane >> 4);
        act_at[k] = acts + (row < toks_here ? row : toks_here - 1u) * act_row_bytes + 4u + 16u * (lane & 15u);
    }
    const unsigned char *const scale_from = acts + (r < toks_here ? r : toks_here - 1u) * act_row_bytes;
    struct {
        v4i weights[9], acts[8];
        unsigned scale;
    } ahead;
    typedef v4i v4i_dword __attribute__((aligned(4)));
    auto request = [&](unsigned sb) {
        const unsigned long long w = sb * 272ull, a = (unsigned long long)sb * kQ8KBytes;
#pragma unroll
        for (unsigned k = 0; k < 9u; ++k) ahead.weights[k] = *reinterpret_cast<const v4i_dword *>(weight_at[k] + w);
#pragma unroll
        for (unsigned k = 0; k < 8u; ++k) ahead.acts[k] = *reinterpret_cast<const v4i_dword *>(act_at[k] + a);
        ahead.scale = *reinterpret_cast<const unsigned *>(scale_from + a);
    };
    const unsigned window = kPlainWindow * wave;
    const float scale = sum_scale();
    double acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0;
    if (wave < g.blocks) request(wave);
    for (unsigned sb = wave; sb < g.blocks; sb += kPlainWaves) {
        // (LDS operations of one wave complete in order)
#pragma unroll
        for (unsigned k = 0; k < 8u; ++k) {
            lds_write_v4i(window + 1024u * k + 16u * lane, ahead.weights[k]);
            lds_write_v4i(window + kPlainAct + 4u * kStagedPitch * k + kStagedPitch * (lane >> 4) + 16u * (lane & 15u), ahead.acts[k]);
        }
        lds_write_v4i(window + 8192u + 16u * r, ahead.weights[8]);
        lds_write_u32(window + kPlainScales + 4u * r, ahead.scale);
        // the next superblock's bytes travel while this one is worked on
        request(sb + kPlainWaves < g.blocks ? sb + kPlainWaves : sb);
        wave_lds_fence();
        q80_superblock(window + r * kStagedPitch, window + kPlainAct + r * kStagedPitch + 16u * h, window + kPlainScales + 4u * r, h,
                       scale, acc);
        wave_lds_fence();
    }

    // (the partial tiles of waves 1 to 3 take the windows' place)
    __syncthreads();
    double *const partial = reinterpret_cast<double *>(dense_q8_0_plain_lds);
    if (wave) {
#pragma unroll
        for (int i = 0; i < 16; ++i) partial[((wave - 1u) * 16u + i) * 64u + lane] = acc[i];
    }
    __syncthreads();
    if (wave) return;
    // lane (r, h): weight row r against sixteen input rows; a store instruction writes 32
    // consecutive floats of two output rows
    const unsigned long long row = row0 + r;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const unsigned long long token = tok0 + 8u * (i >> 2) + 4u * h + (i & 3);
        double wide = acc[i];
#pragma unroll
        for (unsigned w = 0; w + 1u < kPlainWaves; ++w) wide += partial[(w * 16u + i) * 64u + lane];
        const float sum = (float)wide;
        if (row >= g.row_count || token >= g.input_rows) continue;
        const unsigned long long at = token * g.out_stride + row;
        const float value = g.additive ? sum + g.additive[at] : sum;
        if (!finite_f32(value)) raise_status(g.status, 1);
        else g.out[at] = g.output_bf16 ? bf16_round(value) : value;
    }
}

constexpr unsigned kSmallWaves = 8u;
// LDS of a wave: 16 weight rows' superblock, 16 input rows' codes (both 272 bytes a row), their scales
constexpr unsigned kSmallAct = 16u * kStagedPitch, kSmallScales = 2u * kSmallAct, kSmallWindow = kSmallScales + 64u;
constexpr unsigned kSmallLdsBytes = kSmallWaves * kSmallWindow;        // (the partial tiles take their place in the end)

// 16 weight rows x 16 input rows a workgroup, a superblock in eight a wave, on V_MFMA_I32_16X16X32_I8: twice the workgroups
// of the 32 x 32 tiles and no token slot wasted on a batch of sixteen. Loads in runs, a superblock ahead, through LDS as
// above. Lane (r, q) holds bytes 8 q .. 8 q + 7 of input row r's block (A) and of weight row r's block (B); accumulator
// i is weight row r against input row 4 q + i. 4096 x 4096 by 4 / 8 / 16 rows 10.2 / 14.4 / 12.8 us (the first two on
// matvec_block_kernel, the third on the 32 x 32 tiles) -> 7.9 / 8.1 / 8.9, 2048 x 7168 by 4 / 16 / 32 9.9 / 17.2 / 18.3 ->
// 8.7 / 10.2 / 10.0, 1024 x 4096 by 64 13.0 -> 7.4.
__global__ __launch_bounds__(64 * kSmallWaves) void dense_q8_0_small_kernel(DenseQ80Args g)
{
    typedef int v4s __attribute__((ext_vector_type(4)));
    typedef v4i v4i_dword __attribute__((aligned(4)));
    extern __shared__ __align__(16) unsigned char dense_q8_0_small_lds[];
    if (lds_address_of(dense_q8_0_small_lds) != 0u) {   // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(g.status, 2);
        publish_when_last(g.publication, g.status, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
        return;
    }
    choose_matrix(g);
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned r = lane & 15u, q = lane >> 4;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 16ull, tok0 = (unsigned long long)blockIdx.y * 16ull;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < 16ull ? g.row_count - row0 : 16ull);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < 16ull ? g.input_rows - tok0 : 16ull);
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;
    const unsigned char *const weights = g.encoded + row0 * g.row_bytes, *const acts = g.act + tok0 * act_row_bytes;
    // pieces 64 k + lane of 16 rows x 17 (a ragged edge repeats the last row)
    const unsigned char *weight_at[5];
#pragma unroll
    for (unsigned k = 0; k < 5u; ++k) {
        const unsigned piece = k < 4u ? 64u * k + lane : 256u + r, row = piece / 17u;
        weight_at[k] = weights + (row < rows_here ? row : rows_here - 1u) * g.row_bytes + 16u * (piece - 17u * row);
    }
    InputRows16 inputs(acts, act_row_bytes, toks_here, lane);
    v4i ahead[5];
    auto request = [&](unsigned sb) {
        const unsigned long long w = sb * 272ull;
#pragma unroll
        for (unsigned k = 0; k < 5u; ++k) ahead[k] = *reinterpret_cast<const v4i_dword *>(weight_at[k] + w);
        inputs.request(sb);
    };
    const unsigned window = kSmallWindow * wave;
    const unsigned w_row = window + r * kStagedPitch, a_row = window + kSmallAct + r * kStagedPitch + 8u * q;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (wave < g.blocks) request(wave);
    for (unsigned sb = wave; sb < g.blocks; sb += kSmallWaves) {
        // (LDS operations of one wave complete in order)
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) lds_write_v4i(window + 1024u * k + 16u * lane, ahead[k]);
        lds_write_v4i(window + 4096u + 16u * r, ahead[4]);
        inputs.write(window + kSmallAct, kStagedPitch, window + kSmallScales, lane);
        request(sb + kSmallWaves < g.blocks ? sb + kSmallWaves : sb);
        wave_lds_fence();
        const uint4 d4 = read16(window + kSmallScales + 16u * q);
        const float d_a[4] = {__uint_as_float(d4.x), __uint_as_float(d4.y), __uint_as_float(d4.z), __uint_as_float(d4.w)};
        float total[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (unsigned c = 0; c < 8u; ++c) {
            // (an even block's codes start two bytes into a dword)
            const unsigned at = w_row + ((34u * c + 2u) & ~3u) + 8u * q;
            unsigned words[3] = {lds_read_u32(at), lds_read_u32(at + 4u), c % 2u == 0u ? lds_read_u32(at + 8u) : 0u};
            if (c % 2u == 0u) {
                words[0] = __builtin_amdgcn_alignbyte(words[1], words[0], 2u);
                words[1] = __builtin_amdgcn_alignbyte(words[2], words[1], 2u);
            }
            const uint2 tokens = lds_read_uint2(a_row + 32u * c);
            const float d_w = f16_bits_to_float(lds_read_u16(w_row + 34u * c));
            const long a = (long)(((unsigned long long)tokens.y << 32) | tokens.x);
            const long b = (long)(((unsigned long long)words[1] << 32) | words[0]);
            const v4s dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4s{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) total[i] = __builtin_fmaf(d_w * d_a[i], (float)dot[i], total[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += (double)total[i];
        wave_lds_fence();
    }
    __syncthreads();
    double *const partial = reinterpret_cast<double *>(dense_q8_0_small_lds);
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
        for (unsigned w = 0; w + 1u < kSmallWaves; ++w) wide += partial[(w * 4u + i) * 64u + lane];
        const float sum = (float)wide;
        if (row >= g.row_count || token >= g.input_rows) continue;
        const unsigned long long at = token * g.out_stride + row;
        const float value = g.additive ? sum + g.additive[at] : sum;
        if (!finite_f32(value)) raise_status(g.status, 1);
        else store_published(g.publication, g.out + at, g.output_bf16 ? bf16_round(value) : value);
    }
    publish_when_last(g.publication, g.status, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
}

// The same product for batches that offer every compute unit a tile of 128 weight rows x 64
// input rows: the operands of one superblock pass through LDS. GLOBAL_LOAD_LDS instructions whose
// lanes walk consecutive 16-byte pieces of consecutive rows (a dozen cache lines an instruction
// where the kernel above touches up to 64) fill the other of two buffers while this one is
// multiplied; one barrier per superblock. A weight row keeps its 272 bytes and an input row's 256
// codes get the same pitch, its scale (the row's first 16 bytes) as a seventeenth piece behind
// them, so the 16-byte operand reads of 16 lanes fall on 16 different bank groups. The window of
// a block's codes is not 16-byte aligned in its row: a lane reads the two aligned pieces around
// it and picks its dwords (the offsets are compile-time constants).
//
// Eight waves, two per SIMD, each 32 weight rows x 32 input rows over the whole row width: no
// partial tiles. Here the input rows are the A operand and the weight rows the B operand, so lane
// (r, h) holds weight row r against input rows 8 (i / 4) + 4 h + i % 4: the block's scale is one
// value a lane (read from the row's bytes in LDS), and so is an input row's (scale_products).
//
// ROW_BLOCKS = 4: the tile above (512 lanes, 104 KB of LDS, a workgroup a compute unit);
// ROW_BLOCKS = 2: 64 weight rows, four waves, 70 KB, two workgroups a compute unit, for batches
// that have too few of the large tiles.
// TOKEN_BLOCKS = 1 (with ROW_BLOCKS = 8: 256 weight rows x 32 input rows, 153 KB): batches of up to
// 32 input rows against a matrix too large for the caches, an output head at decode width, where
// the second block of input rows would be padding and half of every wave's work with it.
constexpr unsigned staged_lds_bytes(unsigned row_blocks, unsigned token_blocks = 2u)
{
    return 2u * (32u * row_blocks + 32u * token_blocks) * kStagedPitch;
}


template <unsigned ROW_BLOCKS, unsigned TOKEN_BLOCKS = 2u>
__global__ __launch_bounds__(64 * ROW_BLOCKS * TOKEN_BLOCKS, 2) void dense_q8_0_staged_kernel(DenseQ80Args g)
{
    constexpr unsigned kStagedThreads = 64u * ROW_BLOCKS * TOKEN_BLOCKS, kStagedRows = 32u * ROW_BLOCKS;
    constexpr unsigned kStagedTokens = 32u * TOKEN_BLOCKS;
    constexpr unsigned kStagedActBytes = kStagedTokens * kStagedPitch;                  // one buffer
    constexpr unsigned kStagedWeightBytes = kStagedRows * kStagedPitch;                 // one buffer
    constexpr unsigned kStagedWeightBase = 0u;                                          // [buffer]
    constexpr unsigned kStagedActBase = kStagedWeightBase + 2u * kStagedWeightBytes;    // [buffer]
    constexpr unsigned kWeightRounds = kStagedRows * 17u / kStagedThreads;              // full rounds of copies
    constexpr unsigned kWeightRest = (kStagedRows * 17u - kWeightRounds * kStagedThreads) / 64u;   // waves of the last
    constexpr unsigned kActRounds = kStagedTokens * 17u / kStagedThreads;
    constexpr unsigned kActRest = (kStagedTokens * 17u - kActRounds * kStagedThreads) / 64u;
    constexpr unsigned kActTail = (kStagedTokens * 17u - kActRounds * kStagedThreads) % 64u;    // lanes of one more wave
    static_assert((kStagedRows * 17u) % 64u == 0u && (kActTail == 0u || kActTail == 32u), "whole or half waves copy");
    static_assert(kWeightRounds + 1u <= 10u && kActRounds + 1u <= 5u, "copy sources");
    extern __shared__ __align__(16) unsigned char dense_q8_0_lds[];
    if (lds_address_of(dense_q8_0_lds) != 0u) {   // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(g.status, 2);
        if constexpr (TOKEN_BLOCKS == 1u) publish_when_last(g.publication, g.status, blockIdx.x, gridDim.x);
        return;
    }
    choose_matrix(g);
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const unsigned r = lane & 31u, h = lane >> 5;
    const unsigned row_block = wave % ROW_BLOCKS, token_block = wave / ROW_BLOCKS;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * kStagedRows;
    const unsigned long long tok0 = (unsigned long long)blockIdx.y * kStagedTokens;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < kStagedRows ? g.row_count - row0 : kStagedRows);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < kStagedTokens ? g.input_rows - tok0 : kStagedTokens);
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;

    // ---- copy sources (a ragged edge repeats the tile's last row) ----
    // weights: piece q = tid + threads * k of the tile's rows x 17; input rows: piece q of 64 x 17,
    // the seventeenth being the 16 bytes at the row's start
    const unsigned char *weight_from[kWeightRounds + 1u], *act_from[kActRounds + 1u];
#pragma unroll
    for (unsigned k = 0; k < kWeightRounds + 1u; ++k) {
        unsigned q = tid + kStagedThreads * k;
        if (q >= kStagedRows * 17u) q = kStagedRows * 17u - 1u;            // (waves that do not copy this round)
        const unsigned row = q / 17u, piece = q - row * 17u;
        weight_from[k] = g.encoded + (row0 + (row < rows_here ? row : rows_here - 1u)) * g.row_bytes + 16u * piece;
    }
#pragma unroll
    for (unsigned k = 0; k < kActRounds + 1u; ++k) {
        unsigned q = tid + kStagedThreads * k;
        if (q >= kStagedTokens * 17u) q = kStagedTokens * 17u - 1u;
        const unsigned token = q / 17u, piece = q - token * 17u;
        act_from[k] = g.act + (tok0 + (token < toks_here ? token : toks_here - 1u)) * act_row_bytes +
                      (piece < 16u ? 4u + 16u * piece : 0u);
    }
    const unsigned last_block = g.blocks - 1u;
    auto copies = [&](unsigned sb) {
        const unsigned buffer = sb & 1u;
        const unsigned clamped = sb < last_block ? sb : last_block;
        const unsigned long long w_at = (unsigned long long)clamped * 272ull;
        const unsigned long long a_at = (unsigned long long)clamped * kQ8KBytes;
        const unsigned w_to = kStagedWeightBase + buffer * kStagedWeightBytes + 1024u * wave;
        const unsigned a_to = kStagedActBase + buffer * kStagedActBytes + 1024u * wave;
#pragma unroll
        for (unsigned k = 0; k < kWeightRounds; ++k)
            copy_to_lds_16(weight_from[k] + w_at,
                           (unsigned)__builtin_amdgcn_readfirstlane((int)(w_to + 16u * kStagedThreads * k)));
        if (wave < kWeightRest)
            copy_to_lds_16(weight_from[kWeightRounds] + w_at,
                           (unsigned)__builtin_amdgcn_readfirstlane((int)(w_to + 16u * kStagedThreads * kWeightRounds)));
#pragma unroll
        for (unsigned k = 0; k < kActRounds; ++k)
            copy_to_lds_16(act_from[k] + a_at,
                           (unsigned)__builtin_amdgcn_readfirstlane((int)(a_to + 16u * kStagedThreads * k)));
        if (wave < kActRest)
            copy_to_lds_16(act_from[kActRounds] + a_at,
                           (unsigned)__builtin_amdgcn_readfirstlane((int)(a_to + 16u * kStagedThreads * kActRounds)));
        else if (kActTail && wave == kActRest)
            copy_to_lds_16_first32(act_from[kActRounds] + a_at,
                                   (unsigned)__builtin_amdgcn_readfirstlane((int)(a_to + 16u * kStagedThreads * kActRounds)));
    };

    double acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0;

    copies(0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (unsigned sb = 0; sb < g.blocks; ++sb) {
        const unsigned buffer = sb & 1u;
        if (sb + 1u < g.blocks) copies(sb + 1u);
        const unsigned w_row = kStagedWeightBase + buffer * kStagedWeightBytes + (32u * row_block + r) * kStagedPitch;
        const unsigned a_tile = kStagedActBase + buffer * kStagedActBytes + 32u * token_block * kStagedPitch;

        const float d_a = __uint_as_float(lds_read_u32(a_tile + r * kStagedPitch + 256u));   // the lane's input row's scale
        float total[16];            // the superblock's chain of eight terms
#pragma unroll
        for (unsigned i = 0; i < 16u; ++i) total[i] = 0.0f;
        // Three stages in flight, or a wave would run its LDS reads, its matrix instruction and the
        // scaling of the results one after the other: in step k the operands of block k are
        // read, block k - 1 is multiplied and the results of block k - 2 are scaled (vector
        // instructions that issue while the matrix pipe works).
        uint4 lo[2], hi[2] = {};
        v4i tokens[2];
        unsigned scale_bits = 0u;   // of block c + h
        v16i dot[2];
        v32f step;                  // the products of the scales of two blocks (scale_products)
#pragma unroll
        for (unsigned k = 0; k < 10u; ++k) {
            if (k < 8u) {
                const unsigned c = k, slot = c % 2u;
                const unsigned start = c % 2u == 0u ? 34u * c : 34u * c + 2u;      // the lane's window: + 16 h
                lo[slot] = read16(w_row + 16u * h + (start & ~15u));
                // (an even block's window is 20 bytes, an odd block's 16: only block 7's fits one piece)
                hi[slot] = c % 2u == 0u || (start & 15u) ? read16(w_row + 16u * h + (start & ~15u) + 16u) : lo[slot];
                if (c % 2u == 0u) scale_bits = lds_read_u16(w_row + 34u * (c + h));
                tokens[slot] = lds_read_v4i(a_tile + r * kStagedPitch + 16u * (2u * c + h));
            }
            if (k >= 1u && k < 9u) {
                const unsigned c = k - 1u, slot = c % 2u;
                const unsigned start = c % 2u == 0u ? 34u * c : 34u * c + 2u;
                const unsigned at = (start & 15u) / 4u;
                const unsigned q[8] = {lo[slot].x, lo[slot].y, lo[slot].z, lo[slot].w,
                                       hi[slot].x, hi[slot].y, hi[slot].z, hi[slot].w};
                v4i codes;
                if (c % 2u == 0u) {
#pragma unroll
                    for (unsigned j = 0; j < 4u; ++j)
                        codes[j] = (int)__builtin_amdgcn_alignbyte(q[at + j + 1u], q[at + j], 2u);
                } else {
#pragma unroll
                    for (unsigned j = 0; j < 4u; ++j) codes[j] = (int)q[at + j];
                }
                v16i zero;
#pragma unroll
                for (int i = 0; i < 16; ++i) zero[i] = 0;
                dot[slot] = __builtin_amdgcn_mfma_i32_32x32x32_i8(tokens[slot], codes, zero, 0, 0, 0);
            }
            if (k >= 2u) {
                const unsigned slot = k % 2u;           // block k - 2
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    total[i] = __builtin_fmaf(step[16u * slot + i], (float)dot[slot][i], total[i]);
            }
            if (k % 2u == 1u && k < 9u) step = scale_products(d_a, scale_bits);      // of blocks k - 1 and k
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] += (double)total[i];
        // the next superblock's copies have landed and every wave is done with this one's buffers
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    // lane (r, h): weight row r of the wave's 32 against sixteen input rows; a store instruction
    // writes 32 consecutive floats of two output rows
    const unsigned long long row = row0 + 32u * row_block + r;
    bool bad = false;
#pragma unroll
    for (unsigned i = 0; i < 16u; ++i) {
        const unsigned long long token = tok0 + 32u * token_block + 8u * (i >> 2) + 4u * h + (i & 3u);
        if (row >= g.row_count || token >= g.input_rows) continue;
        const unsigned long long at = token * g.out_stride + row;
        const float sum = (float)acc[i];
        const float value = g.additive ? sum + g.additive[at] : sum;
        if (!finite_f32(value)) bad = true;
        else if (TOKEN_BLOCKS == 1u) store_published(g.publication, g.out + at, g.output_bf16 ? bf16_round(value) : value);
        else g.out[at] = g.output_bf16 ? bf16_round(value) : value;
    }
    if (bad) raise_status(g.status, 1);
    if constexpr (TOKEN_BLOCKS == 1u) publish_when_last(g.publication, g.status, blockIdx.x, gridDim.x);
}

constexpr unsigned kWideRows = 128u, kWideTokens = 128u, kWideThreads = 1024u;
constexpr unsigned kWideWeightBytes = kWideRows * kStagedPitch, kWideActBytes = kWideTokens * kStagedPitch;  // one buffer
constexpr unsigned kWideActBase = 2u * kWideWeightBytes, kWideScaleBase = kWideActBase + 2u * kWideActBytes;
constexpr unsigned kWideLdsBytes = kWideScaleBase + 2u * kWideTokens * 4u;

// The same product for batches that fill the device with tiles of 128 weight rows x 128 input rows.
// Behind one matrix instruction (32 cycles) sixteen results a lane are brought to float, multiplied by their scale and
// chained: the vector ALU has most of the work, and no wave may be alone with its waits. What this kernel does about it:
//  * kStartBits above in place of the conversions.
//  * A wave owns 32 weight rows x 32 input rows on 128 registers, so that sixteen of them, four a SIMD, cover each
//    other's waits and the rate of one wave's instructions (one in 5.5 cycles on this part; two waves issue 4-cycle
//    instructions in 5.0 cycles each, four in 4.4).
//  * Copies take a scalar base and a 32-bit offset a lane: a register and no addition each.
// 4096 x 4096 by 2048 rows 136 -> 129 us (532 TOP/s; eight waves of 32 x 64, two a SIMD, before). With
// scale_products 119 us. No pipe is full: the vector ALU is issued to 51 % of the time, the LDS is busy 32 %, nearly half of it bank
// conflicts (at a pitch of 272 bytes rows r and r + 16 start on one bank, which the reads of less than 16 bytes meet on), the matrix
// cores 25 %; a wave waits for data 42 % of its time, copies behind a full wait and a barrier a superblock, and for its turn to
// issue 34 %. Whole 16-byte reads of a window's end, before scale_products: 131 us.
__global__ __launch_bounds__(kWideThreads) void dense_q8_0_wide_kernel(DenseQ80Args g)
{
    extern __shared__ __align__(16) unsigned char dense_q8_0_lds[];
    if (lds_address_of(dense_q8_0_lds) != 0u) {   // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(g.status, 2);
        return;
    }
    choose_matrix(g);
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const unsigned r = lane & 31u, h = lane >> 5;
    const unsigned row_block = wave & 3u, token_block = wave >> 2;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * kWideRows;
    const unsigned long long tok0 = (unsigned long long)blockIdx.y * kWideTokens;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < kWideRows ? g.row_count - row0 : kWideRows);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < kWideTokens ? g.input_rows - tok0 : kWideTokens);
    const unsigned act_row_bytes = g.blocks * kQ8KBytes, row_bytes = (unsigned)g.row_bytes;

    // ---- copies: pieces q = tid + 1024 k of 128 rows x 17 (a ragged edge repeats the tile's last row;
    // an input row's seventeenth piece only keeps the pitch); the last 128 pieces of the weights by
    // waves 0 and 1, of the input rows by waves 2 and 3, the input rows' scales by waves 4 and 5 ----
    unsigned weight_at[3], act_at[3];
#pragma unroll
    for (unsigned k = 0; k < 3u; ++k) {
        const unsigned q = k < 2u ? tid + kWideThreads * k : 2048u + (tid & 127u);
        const unsigned row = q / 17u, piece = q - row * 17u;
        weight_at[k] = (row < rows_here ? row : rows_here - 1u) * row_bytes + 16u * piece;
        act_at[k] = (row < toks_here ? row : toks_here - 1u) * act_row_bytes + (piece < 16u ? 4u + 16u * piece : 0u);
    }
    const unsigned scale_token = tid & 127u;
    const unsigned scale_at = (scale_token < toks_here ? scale_token : toks_here - 1u) * act_row_bytes;
    const unsigned char *weights = g.encoded + row0 * g.row_bytes;
    const unsigned char *acts = g.act + tok0 * act_row_bytes;
    const unsigned wave_lds = (unsigned)__builtin_amdgcn_readfirstlane((int)(1024u * wave));
    const unsigned scale_lds = (unsigned)__builtin_amdgcn_readfirstlane((int)(kWideScaleBase + 256u * (wave & 1u)));
    const unsigned rest_lds = (unsigned)__builtin_amdgcn_readfirstlane((int)(2048u * 16u + 1024u * (wave & 1u)));
    auto copies = [&](unsigned sb) {
        const unsigned buffer = sb & 1u;
        const unsigned char *w = weights + (unsigned long long)sb * 272ull;
        const unsigned char *a = acts + (unsigned long long)sb * kQ8KBytes;
        const unsigned w_to = buffer * kWideWeightBytes, a_to = kWideActBase + buffer * kWideActBytes;
#pragma unroll
        for (unsigned k = 0; k < 2u; ++k) {
            copy_to_lds_16_at(w, weight_at[k], w_to + wave_lds + 16u * kWideThreads * k);
            copy_to_lds_16_at(a, act_at[k], a_to + wave_lds + 16u * kWideThreads * k);
        }
        if (wave < 2u) copy_to_lds_16_at(w, weight_at[2], w_to + rest_lds);
        else if (wave < 4u) copy_to_lds_16_at(a, act_at[2], a_to + rest_lds);
        else if (wave < 6u) copy_to_lds_4_at(a, scale_at, scale_lds + buffer * (kWideTokens * 4u));
    };

    const float scale = sum_scale();
    double acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0;
    copies(0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (unsigned sb = 0; sb < g.blocks; ++sb) {
        const unsigned buffer = sb & 1u;
        if (sb + 1u < g.blocks) copies(sb + 1u);
        q80_superblock(buffer * kWideWeightBytes + (32u * row_block + r) * kStagedPitch,
                       kWideActBase + buffer * kWideActBytes + (32u * token_block + r) * kStagedPitch + 16u * h,
                       kWideScaleBase + buffer * (kWideTokens * 4u) + (32u * token_block + r) * 4u, h, scale, acc);
        // the next superblock's copies have landed and every wave is done with this one's buffers
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    const unsigned long long row = row0 + 32u * row_block + r;
    if (row >= g.row_count) return;
    bool bad = false;
#pragma unroll
    for (unsigned i = 0; i < 16u; ++i) {
        const unsigned long long token = tok0 + 32u * token_block + 8u * (i >> 2) + 4u * h + (i & 3u);
        if (token >= g.input_rows) continue;
        const unsigned long long at = token * g.out_stride + row;
        const float sum = (float)acc[i];
        const float value = g.additive ? sum + g.additive[at] : sum;
        if (!finite_f32(value)) bad = true;
        else g.out[at] = g.output_bf16 ? bf16_round(value) : value;
    }
    if (bad) raise_status(g.status, 1);
}

}  // namespace

int launch_q8_0_rows_dense(const uint8_t *encoded, uint64_t row_count, uint64_t row_width,
                           uint64_t row_bytes, const void *act_q8k, uint64_t input_rows,
                           const float *additive, float *out, uint64_t out_stride, bool output_bf16,
                           int *status, hipStream_t stream, const uint8_t *encoded_second, float *out_second,
                           Publisher *publisher)
{
    const uint64_t matrices = encoded_second ? 2u : 1u;
    if (!row_count || !input_rows || row_width % 256u || row_width / 32u * 34u != row_bytes)
        return ST_BOUNDS;
    if ((((uintptr_t)encoded | (uintptr_t)encoded_second) & 3u) || ((uintptr_t)act_q8k & 3u)) return ST_INVALID_ARG;
    const bool aligned16 = !(((uintptr_t)encoded | (uintptr_t)encoded_second) & 15u);
    const uint64_t row_tiles = (row_count + 31u) / 32u;
    if (row_tiles > 0x7fffffffull || row_width / 256u > 0xffffffffull) return ST_BOUNDS;
    DenseQ80Args g{encoded, row_count, row_bytes, (unsigned)(row_width / 256u),
                   (const unsigned char *)act_q8k, input_rows, additive, out, out_stride,
                   output_bf16 ? 1 : 0, status, encoded_second, out_second, {}};
    if (matrices > 1u) publisher = nullptr;       // (workgroups are counted over one matrix)
    // Which tiles: the ones whose launch is the shortest. A pass over the row width takes a workgroup about as long
    // whatever the device's load, so a launch's time goes by its rounds over the compute units, or by its tiles where
    // many workgroups share one; either has a part that grows with the row (`long_rows`: 1 at 4096 columns). The numbers are
    // microseconds, fitted to calls of seventeen matrices of 1024 to 16384 rows of 256 to 14336 columns by 17 to 2048 rows, each on every
    // kind of tiles: the choice is 0.1 % behind the best one on average and 2.7 % at most, and 6 % at most for eleven other matrices
    // (1.3 and 24 before, by numbers that did not know the row's length and were older than scale_products). us a call before and
    // now: 4096 x 4096 by 1400 rows 118.3 and 113.5, 7168 x 7168 by 65 51.8 and 47.0, 2048 x 7168 by 333 52.6 and 48.6, 16384 x 2048 by 320
    // 70.1 and 62.1, 1024 x 4096 by 160 24.8 and 23.6.
    const uint64_t token_tiles32 = (input_rows + 31u) / 32u;
    const uint64_t token_tiles64 = (input_rows + 63u) / 64u;
    if (token_tiles32 > 65535ull) return ST_BOUNDS;
    const uint64_t units = (uint64_t)compute_units();
    // up to 32 input rows against a matrix with a 256-row tile for every compute unit (an output
    // head at decode width, 129 280 x 7168: 306 us on the 128 x 64 tiles, half of them padding;
    // memory time 173 us)
    if (aligned16 && input_rows <= 32u && units && matrices * ((row_count + 255u) / 256u) >= units) {
        YVEX_ALLOW_DYNAMIC_LDS((dense_q8_0_staged_kernel<8u, 1u>), staged_lds_bytes(8u, 1u));
        g.publication = take_publication(publisher, (row_count + 255u) / 256u);
        dense_q8_0_staged_kernel<8u, 1u><<<dim3((unsigned)((row_count + 255u) / 256u), 1, (unsigned)matrices), 512, staged_lds_bytes(8u, 1u),
                                           stream>>>(g);
        return check_launch("dense_q8_0_staged");
    }
    const uint64_t token_tiles16 = (input_rows + 15u) / 16u, small = matrices * ((row_count + 15u) / 16u) * token_tiles16;
    const uint64_t plain = matrices * row_tiles * token_tiles32;
    const double long_rows = (double)row_width / 4096.0;
    auto share = [&](uint64_t tiles) { return units && tiles > units ? (double)tiles / (double)units : 1.0; };
    auto rounds = [&](uint64_t tiles) { return units ? (double)((tiles + units - 1u) / units) : 1.0; };
    const double plain_cost = 6.9 + 7.4 * long_rows + (2.6 + 3.4 * long_rows) * (share(plain) - 1.0);
    const double small_cost = share(small) > 1.0 ? 3.8 + 2.9 * long_rows + (1.5 + 1.9 * long_rows) * share(small) : 1.3 + 5.3 * long_rows;
    const uint64_t tall = matrices * ((row_count + 127u) / 128u) * token_tiles64, low = matrices * ((row_count + 63u) / 64u) * token_tiles64;
    const uint64_t token_tiles128 = (input_rows + 127u) / 128u, wide = matrices * ((row_count + 127u) / 128u) * token_tiles128;
    // (two workgroups of the 64-row tiles share a compute unit: the second round costs little)
    const double low_rounds = rounds(low), low_second = low_rounds > 1.0 ? 2.1 + 5.2 * long_rows : 0.0;
    const double low_cost = 5.4 + 19.7 * long_rows + low_second + (low_rounds > 2.0 ? (1.5 + 11.3 * long_rows) * (low_rounds - 2.0) : 0.0);
    const double tall_cost = 5.2 + 30.7 * long_rows + (3.6 + 29.0 * long_rows) * (rounds(tall) - 1.0);
    const double wide_cost = 5.1 + 44.3 * long_rows + (5.8 + 39.3 * long_rows) * (rounds(wide) - 1.0);
    const bool staged = aligned16 && units;
    if (small_cost < plain_cost && (!staged || (small_cost < low_cost && small_cost <= tall_cost)) && token_tiles16 <= 65535u &&
        (row_count + 15u) / 16u <= 0x7fffffffull) {
        YVEX_ALLOW_DYNAMIC_LDS(dense_q8_0_small_kernel, kSmallLdsBytes);
        g.publication = take_publication(publisher, small);
        dense_q8_0_small_kernel<<<dim3((unsigned)((row_count + 15u) / 16u), (unsigned)token_tiles16, (unsigned)matrices),
                                  64 * kSmallWaves, kSmallLdsBytes, stream>>>(g);
        return check_launch("dense_q8_0_small");
    }
    if (staged) {
        // (32-bit offsets into a tile's rows)
        if (wide_cost < plain_cost && wide_cost <= low_cost && wide_cost <= tall_cost &&
            row_bytes <= (1ull << 24) && row_width / 256u * kQ8KBytes <= (1ull << 24)) {
            YVEX_ALLOW_DYNAMIC_LDS(dense_q8_0_wide_kernel, kWideLdsBytes);
            dense_q8_0_wide_kernel<<<dim3((unsigned)((row_count + 127u) / 128u), (unsigned)token_tiles128,
                                          (unsigned)matrices), kWideThreads, kWideLdsBytes, stream>>>(g);
            return check_launch("dense_q8_0_wide");
        }
        if (tall_cost < plain_cost && tall_cost <= low_cost) {
            YVEX_ALLOW_DYNAMIC_LDS(dense_q8_0_staged_kernel<4u>, staged_lds_bytes(4u));
            dense_q8_0_staged_kernel<4u><<<dim3((unsigned)((row_count + 127u) / 128u), (unsigned)token_tiles64, (unsigned)matrices), 512,
                                          staged_lds_bytes(4u), stream>>>(g);
            return check_launch("dense_q8_0_staged");
        }
        if (low_cost < plain_cost) {
            YVEX_ALLOW_DYNAMIC_LDS(dense_q8_0_staged_kernel<2u>, staged_lds_bytes(2u));
            dense_q8_0_staged_kernel<2u><<<dim3((unsigned)((row_count + 63u) / 64u), (unsigned)token_tiles64, (unsigned)matrices), 256,
                                          staged_lds_bytes(2u), stream>>>(g);
            return check_launch("dense_q8_0_staged");
        }
    }
    YVEX_ALLOW_DYNAMIC_LDS(dense_q8_0_kernel, kPlainLdsBytes);
    dense_q8_0_kernel<<<dim3((unsigned)row_tiles, (unsigned)token_tiles32, (unsigned)matrices), 64 * kPlainWaves, kPlainLdsBytes,
                        stream>>>(g);
    return check_launch("dense_q8_0");
}

}  // namespace yvex
