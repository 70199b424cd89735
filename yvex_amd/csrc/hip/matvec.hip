// Encoded matvec (dense projection / output head), gather and the int32 block-sum probe.
//
// One 64-lane wavefront owns one encoded weight row and up to T activation rows; lanes walk the
// row in 32-weight units, so one unit's packed bytes are decoded once and reused for every
// activation row of the tile. Q8_K activations go through v_dot4 integer dots whose exact sums
// are reduced across the eight lanes of a superblock before the single float scaling; F32
// activations use fused multiply-adds. Results are summed across the wave with shuffles.
//
// Behaviour restated from src/backend/cuda/kernels.cu:529-626 (matvec), :784-830 (gather) and
// src/backend/cuda/kernel_primitives.h:218-255,566-596 (row dots).
#include <type_traits>
#include "common.hpp"
#include "launch.hpp"
#include "units.hpp"
#include "route.hpp"
#include "publish.hpp"
#include "q8_0_rows.hpp"

namespace yvex {

struct MatvecArgs {
    const unsigned char *encoded;
    unsigned long long row_count, row_width, row_bytes;
    const void *input;
    unsigned long long input_rows, input_stride;
    const float *additive;
    float *out;
    unsigned long long out_stride;
    int output_bf16;
    int *status;
    double *parts;           // split projections: [split][input row][weight row] partial sums
    float *scores;           // join of a split projection: the router scores of the outputs as well
    int scoring;
    const unsigned char *encoded_second = nullptr;   // a second matrix of the same shape (blockIdx.z = 1)
    float *out_second = nullptr;
    Publication publication = {nullptr, nullptr, 0u, 0};
};

__device__ __forceinline__ void matvec_publish(const MatvecArgs &a, unsigned long long in,
                                               unsigned long long row, float sum)
{
    const unsigned long long at = in * a.out_stride + row;
    float value = a.additive ? sum + a.additive[at] : sum;
    if (!finite_f32(value)) raise_status(a.status, 1);
    else store_published(a.publication, a.out + at, a.output_bf16 ? bf16_round(value) : value);
}

// Slow exact path for a row whose F32 sum overflowed before opposite terms cancelled
// (kernels.cu:616-620): the whole wave recomputes it in double.
__device__ float matvec_recover_f64(const unsigned char *row, const float *x,
                                    unsigned long long width, unsigned qtype)
{
    double sum = 0.0;
    for (unsigned long long i = threadIdx.x & 63u; i < width; i += 64u)
        sum += (double)qtype_value(row, i, qtype) * (double)x[i];
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) sum += __shfl_xor(sum, offset, kWave);
    return (float)sum;
}

// U: 64-unit chunks of the row whose loads are issued together before the first of them is used.
// A wave walks one row front to back; with one chunk in flight it waits a full memory latency per
// chunk (weights, then the activation bytes that go with them), which bounds a long matrix such as
// an output head well below what the same loads reach when nothing waits on them.
// EVEN: every row starts on an even address (even base address and even row bytes).
// STAGE (one F32 input row): the workgroup copies the input row into LDS once, 16-byte pieces
// swizzled inside each 128-byte unit, and its four waves read their units from there. A lane owns
// 32 consecutive values, so read from global memory each of its eight 16-byte loads touches 64
// different cache lines, which the memory pipeline serves at about two cycles a line.
template <unsigned QT, bool Q8, int T, int U, bool EVEN, bool STAGE = false>
__global__ __launch_bounds__(256) void matvec_block_kernel(MatvecArgs a)
{
    __shared__ Iq2Tables tables;
    extern __shared__ __align__(16) float4 staged_row[];
    const unsigned long long in0 = (unsigned long long)blockIdx.y * T;
    if (blockIdx.z) {
        a.encoded = a.encoded_second;
        a.out = a.out_second;
    }
    if constexpr (STAGE) {
        const float4 *source = reinterpret_cast<const float4 *>((const float *)a.input + in0 * a.input_stride);
        const unsigned pieces = (unsigned)(a.row_width >> 2);
        for (unsigned p = threadIdx.x; p < pieces; p += 256u)
            staged_row[(p & ~7u) | ((p ^ (p >> 3)) & 7u)] = source[p];
    }
    if constexpr (QT == QT_IQ2_XXS) iq2_tables_fill(tables);
    if constexpr (QT == QT_IQ2_XXS || STAGE) __syncthreads();
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long row = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (row >= a.row_count) return;
    const unsigned char *wrow = a.encoded + row * a.row_bytes;
    const unsigned units = (unsigned)(a.row_width >> 5);
    const unsigned long long act_row_bytes = (a.row_width >> 8) * kQ8KBytes;
    // Q8_K activations against superblock formats: a superblock's float term is formed in the
    // order of the reference's device primitive and the terms of a row are added in double and
    // rounded once, as the CPU path adds a row's blocks (src/gguf/quant_compute.c:152-172): the
    // result is that path's, bit for bit. Q8_0 rows chain their eight terms of a superblock as
    // the primitive chains them (total = fmaf(d_b * d_a, float(dot_b), total), b = 0 .. 7, from
    // zero: kernel_primitives.h:342-359) across the eight lanes that hold the superblock's blocks.
    // F32 activations keep float partial sums, inside the tolerance of the dense projections.
    constexpr bool kWide = Q8 && (UnitTraits<QT>::kIntegerCombine || QT == QT_Q8_0);
    using Sum = typename std::conditional<kWide, double, float>::type;
    Sum acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = (Sum)0;

    // Every lane runs the same trip count so the superblock shuffles below stay converged.
    for (unsigned base = 0; base < units; base += 64u * U) {
        Unit unit[U];
        unsigned uu[U];
        bool live[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const unsigned u = base + 64u * j + lane;
            live[j] = u < units;
            uu[j] = live[j] ? u : units - 1u;
            unit_load<QT, EVEN ? 1 : -1>(tables, wrow, uu[j], unit[j]);
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            if (j > 0 && base + 64u * j >= units) break;      // wave-uniform: no chunk here
#pragma unroll
            for (int t = 0; t < T; ++t) {
                unsigned long long in = in0 + t;
                if (in >= a.input_rows) in = a.input_rows - 1ull;   // clamped rows are never written
                if constexpr (Q8) {
                    const unsigned char *act = (const unsigned char *)a.input + in * act_row_bytes +
                                               (unsigned long long)(uu[j] >> 3) * kQ8KBytes;
                    UnitSum s = unit_dot_q8<QT>(unit[j], act, uu[j] & 7u);
                    const float act_scale = *reinterpret_cast<const float *>(act);
                    if constexpr (UnitTraits<QT>::kIntegerCombine) {
                        if (!live[j]) s.dot = s.min = 0;
                        s.dot = group_sum_i32<8>(s.dot);
                        if constexpr (QT != QT_IQ2_XXS) s.min = group_sum_i32<8>(s.min);
                        if (live[j] && (uu[j] & 7u) == 0u)
                            acc[t] += (Sum)super_combine<QT>(wrow + (uu[j] >> 3) * UnitTraits<QT>::kSuperBytes,
                                                             act_scale, s);
                    } else {
                        // lane b of a group of eight holds block b. The start gives lane 0 its
                        // chain (block 0 onto zero); step k gives lane k the chain through block k
                        // from lane k - 1's value of the step before, so after seven steps the last
                        // lane holds the superblock's total. What a lane holds after its own step
                        // is read by nobody and may be anything (units past the row's end belong
                        // to no superblock: a row is whole superblocks)
                        const float scale = f16_bits_to_float((unsigned short)unit[j].scale_bits) * act_scale;
                        const float value = (float)s.dot;
                        float total = __builtin_fmaf(scale, value, 0.0f);
#pragma unroll
                        for (int step = 1; step < 8; ++step) {
                            const float before = __int_as_float(
                                __builtin_amdgcn_update_dpp(0, __float_as_int(total), 0x111, 0xf, 0xf, false));   // row_shr:1
                            total = __builtin_fmaf(scale, value, before);
                        }
                        acc[t] += (Sum)(live[j] && (lane & 7u) == 7u ? total : 0.0f);
                    }
                } else if constexpr (STAGE) {
                    float4 x4[8];
#pragma unroll
                    for (unsigned i = 0; i < 8u; ++i) x4[i] = staged_row[8u * uu[j] + (i ^ (uu[j] & 7u))];
                    const float v = unit_dot_f32_values<QT>(unit[j], wrow, uu[j], x4);
                    if (live[j]) acc[t] += v;
                } else {
                    const float *x = (const float *)a.input + in * a.input_stride + 32ull * uu[j];
                    const float v = unit_dot_f32<QT>(unit[j], wrow, uu[j], x);
                    if (live[j]) acc[t] += v;
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float sum;
        if constexpr (kWide) {
            sum = (float)wave_sum_f64(acc[t]);
        } else {
            sum = group_sum_f32<64>(acc[t]);
        }
        const unsigned long long in = in0 + t;
        if (in >= a.input_rows) continue;
        if constexpr (!Q8) {
            if (!finite_f32(sum) && *a.status == 0)
                sum = matvec_recover_f64(wrow, (const float *)a.input + in * a.input_stride,
                                         a.row_width, QT);
        }
        if (lane == 0u) matvec_publish(a, in, row, sum);
    }
}

// A few F32 input rows against Q8_0 rows on even addresses, quantized on the way (q8_0_rows.hpp). The first weight row's
// bytes are on their way while the input rows are quantized.
template <int T, int U>
__global__ __launch_bounds__(kHeldThreads) void matvec_q8_0_quantizing_kernel(MatvecArgs a)
{
    extern __shared__ __align__(16) unsigned char held[];
    const unsigned units = (unsigned)(a.row_width >> 5), input_rows = (unsigned)a.input_rows;
    HoldRows hold{(const float *)a.input, a.input_stride, units >> 3, input_rows * (units >> 3), a.status, {}};
    held_rows<T, U>(a.row_count, blockIdx.x, gridDim.x, units, held,
                    [&](unsigned long long row) { return a.encoded + row * a.row_bytes; }, hold,
                    [&](unsigned in, unsigned long long row, float sum) {
                        if (in < input_rows) matvec_publish(a, in, row, sum);
                    });
    publish_when_last(a.publication, a.status, blockIdx.x, gridDim.x);
}

// A unit against 32 int8 activations held in registers; `sums` = the two 16-value sums of the
// activations as Q8_K stores them (low and high half of the dword).
template <unsigned QT>
__device__ __forceinline__ UnitSum unit_dot_regs(const Unit &unit, const unsigned *a, unsigned sums)
{
    const int first = (int)(short)(sums & 0xffffu), second = (int)(short)(sums >> 16);
    UnitSum out;
    if constexpr (QT == QT_Q2_K) {
        int d1 = 0, d2 = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            d1 = dot4(unit.w[i], a[i], d1);
            d2 = dot4(unit.w[4 + i], a[4 + i], d2);
        }
        out.dot = unit.factor * d1 + unit.factor2 * d2;
        out.min = unit.min1 * first + unit.min2 * second;
    } else {
        int d = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) d = dot4(unit.w[i], a[i], d);
        out.dot = unit.factor * d;
        out.min = QT == QT_Q4_K ? unit.min1 * (first + second) : 0;
    }
    return out;
}

// A lane's half superblock (units 4 half .. 4 half + 3 of superblock sb) of a weight row that
// starts on a dword boundary. The 32 record bytes of an IQ2_XXS half start on a 2-byte boundary,
// and vector loads that are not dword-aligned run at less than half rate: the aligned dwords
// that hold them are loaded and shifted into place, and the superblock's fp16 scale comes out
// of the aligned dword that holds it (never a byte outside the row's own or its neighbours').
template <unsigned QT>
__device__ __forceinline__ void half_superblock_load(LaneChunk<QT> &chunk, const unsigned char *wrow,
                                                     unsigned sb, unsigned half)
{
    if constexpr (QT == QT_IQ2_XXS) {
        const unsigned char *b = wrow + sb * 66u;
        const unsigned char *p = b + 2u + 32u * half;
        const unsigned shift = (unsigned)(unsigned long long)p & 3u;       // 0 or 2
        const unsigned *at = reinterpret_cast<const unsigned *>(p - shift);
        unsigned raw[9];
#pragma unroll
        for (int i = 0; i < 8; ++i) raw[i] = at[i];
        raw[8] = at[shift ? 8 : 0];                       // (aligned records end with the eighth)
        const unsigned head = *reinterpret_cast<const unsigned *>(b - ((unsigned long long)b & 2ull));
#pragma unroll
        for (int i = 0; i < 8; ++i) chunk.q[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], shift);
        chunk.d16 = ((unsigned long long)b & 2ull) ? head >> 16 : head & 0xffffu;
    } else {
        chunk.load(wrow, 8u * sb + 4u * half);
    }
}

// One Q8_K input row against superblock-format weight rows, for matrices of a few megabytes
// whose launch is over before the memory system is busy: what counts is the number of memory
// round trips a wave waits for one after another. A lane owns half a superblock (four units)
// of its weight row and L lanes share the row, so a wave holds 64 / L rows; every byte the lane
// needs (weight record, superblock header, activation bytes, their scale and sums) is asked for
// by loads that depend on nothing, issued together, and (IQ2_XXS) the codebook tables are
// built in LDS while those are in flight: one round trip, where the general kernel above
// waits for several in turn (unit after unit, then the header for the lane that combines).
// The float term of a superblock and the double-precision row sum are the general kernel's.
template <unsigned QT, int L>
__global__ __launch_bounds__(256) void dense_row_q8k_kernel(MatvecArgs a)
{
    __shared__ Iq2Tables tables;
    constexpr unsigned kRows = 64u / L;
    const unsigned lane = threadIdx.x & 63u, slot = lane % L;
    unsigned long long row = ((unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6)) * kRows + lane / L;
    const bool row_live = row < a.row_count;
    if (!row_live) row = a.row_count - 1ull;          // (no early exit: the barrier below)
    const unsigned char *wrow = a.encoded + row * a.row_bytes;
    const unsigned halves = (unsigned)(a.row_width >> 7);
    // (asked for ahead of the weight bytes: loads come back in order, and the tables are to be
    // built while the weight bytes are on their way, not after them)
    unsigned digits = 0u;
    if constexpr (QT == QT_IQ2_XXS) digits = k_iq2_digits[threadIdx.x];
    double acc = 0.0;
    for (unsigned base = 0; base < halves; base += L) {
        // a superblock's two lanes are live or clamped together (halves and L are even)
        const bool live = base + slot < halves;
        const unsigned hs = live ? base + slot : halves - 1u;
        const unsigned sb = hs >> 1, half = hs & 1u;
        LaneChunk<QT> chunk;
        half_superblock_load<QT>(chunk, wrow, sb, half);
        const unsigned char *block = (const unsigned char *)a.input + (unsigned long long)sb * kQ8KBytes;
        const unsigned *values = reinterpret_cast<const unsigned *>(block + 4u + 128u * half);
        unsigned act[32], sums[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < 32; ++i) act[i] = values[i];
        if constexpr (QT != QT_IQ2_XXS) {
            const unsigned *s = reinterpret_cast<const unsigned *>(block + 260u + 16u * half);
#pragma unroll
            for (int i = 0; i < 4; ++i) sums[i] = s[i];
        }
        const float act_scale = *reinterpret_cast<const float *>(block);
        if constexpr (QT == QT_IQ2_XXS) {
            if (base == 0u) {                             // (the same trip for every thread)
                asm volatile("" : "+v"(digits));          // (the entry is not to be worked out, and waited for, ahead of the loads above)
                tables.magnitudes[threadIdx.x] = iq2_magnitude_of_digits(digits);   // 256 threads, 256 entries
                if (threadIdx.x < 128u) tables.signmask[threadIdx.x] = iq2_signmask_entry(threadIdx.x);
                __syncthreads();
            }
        }
        UnitSum total{0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            Unit unit;
            chunk.decode(tables, k, 8u * sb + 4u * half, unit);
            const UnitSum s = unit_dot_regs<QT>(unit, act + 8 * k, sums[k]);
            total.dot += s.dot;
            total.min += s.min;
        }
        total.dot += dpp_move<0xb1, 0xf>(total.dot);      // the superblock's other half
        if constexpr (QT != QT_IQ2_XXS) total.min += dpp_move<0xb1, 0xf>(total.min);
        const float term = chunk.combine(act_scale, total);
        if (live && half == 0u) acc += (double)term;
    }
    acc = group_sum_f64_last<L>(acc);
    if (row_live && slot == (unsigned)L - 1u) matvec_publish(a, 0ull, row, (float)acc);
    publish_when_last(a.publication, a.status, blockIdx.x, gridDim.x);
}

// The same for a few Q8_K input rows (rows of up to 8192 columns, which L lanes hold whole): the
// lane's four units are decoded once and stay in registers, and the input rows go by one after
// another, the next one's bytes asked for before the current one is multiplied.
struct RowActs {
    unsigned values[32];
    unsigned sums[4];
    float scale;
};

template <unsigned QT>
__device__ __forceinline__ void row_acts_load(RowActs &r, const unsigned char *block, unsigned half)
{
    const unsigned *values = reinterpret_cast<const unsigned *>(block + 4u + 128u * half);
#pragma unroll
    for (int i = 0; i < 32; ++i) r.values[i] = values[i];
    if constexpr (QT != QT_IQ2_XXS) {
        const unsigned *s = reinterpret_cast<const unsigned *>(block + 260u + 16u * half);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.sums[i] = s[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) r.sums[i] = 0u;
    }
    r.scale = *reinterpret_cast<const float *>(block);
}

template <unsigned QT, int L>
__global__ __launch_bounds__(256) void dense_fewrows_q8k_kernel(MatvecArgs a)
{
    __shared__ Iq2Tables tables;
    constexpr unsigned kRows = 64u / L;
    const unsigned lane = threadIdx.x & 63u, slot = lane % L;
    unsigned long long row = ((unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6)) * kRows + lane / L;
    const bool row_live = row < a.row_count;
    if (!row_live) row = a.row_count - 1ull;
    const unsigned char *wrow = a.encoded + row * a.row_bytes;
    const unsigned halves = (unsigned)(a.row_width >> 7);             // <= L
    const unsigned long long act_row_bytes = (a.row_width >> 8) * kQ8KBytes;
    unsigned digits = 0u;
    if constexpr (QT == QT_IQ2_XXS) digits = k_iq2_digits[threadIdx.x];
    const bool live = slot < halves;
    const unsigned hs = live ? slot : halves - 1u;
    const unsigned sb = hs >> 1, half = hs & 1u;
    LaneChunk<QT> chunk;
    half_superblock_load<QT>(chunk, wrow, sb, half);
    const unsigned char *block = (const unsigned char *)a.input + (unsigned long long)sb * kQ8KBytes;
    RowActs current;
    row_acts_load<QT>(current, block, half);
    if constexpr (QT == QT_IQ2_XXS) {
        asm volatile("" : "+v"(digits));
        tables.magnitudes[threadIdx.x] = iq2_magnitude_of_digits(digits);
        if (threadIdx.x < 128u) tables.signmask[threadIdx.x] = iq2_signmask_entry(threadIdx.x);
        __syncthreads();
    }
    Unit units[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) chunk.decode(tables, k, 8u * sb + 4u * half, units[k]);
    for (unsigned long long in = 0; in < a.input_rows; ++in) {
        RowActs next;
        const unsigned long long ahead = in + 1ull < a.input_rows ? in + 1ull : in;
        row_acts_load<QT>(next, block + ahead * act_row_bytes, half);
        UnitSum total{0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const UnitSum s = unit_dot_regs<QT>(units[k], current.values + 8 * k, current.sums[k]);
            total.dot += s.dot;
            total.min += s.min;
        }
        total.dot += dpp_move<0xb1, 0xf>(total.dot);
        if constexpr (QT != QT_IQ2_XXS) total.min += dpp_move<0xb1, 0xf>(total.min);
        const float term = chunk.combine(current.scale, total);
        const double sum = group_sum_f64_last<L>(live && half == 0u ? (double)term : 0.0);
        if (row_live && slot == (unsigned)L - 1u) matvec_publish(a, in, row, (float)sum);
        current = next;
    }
    publish_when_last(a.publication, a.status, blockIdx.x, gridDim.x);
}

// F32 / F16 / BF16 weight rows: lanes stride the row element-wise. Products and sums run in
// double, as the CPU row dot forms them (src/gguf/quant_compute.c:152-172: double(value) *
// double(x) added in double, rounded to float once); the product of two floats is exact in
// double, so only the order of the double additions differs from the serial loop, far below
// what the final rounding to float keeps.
template <int T>
__global__ __launch_bounds__(256) void matvec_scalar_kernel(MatvecArgs a, unsigned qtype)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long row = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    const unsigned long long in0 = (unsigned long long)blockIdx.y * T;
    if (row >= a.row_count) return;
    const unsigned char *wrow = a.encoded + row * a.row_bytes;
    double acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = 0.0;
    for (unsigned long long i = lane; i < a.row_width; i += 64u) {
        const float w = qtype_value(wrow, i, qtype);
        if (!finite_f32(w)) raise_status(a.status, 1);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            unsigned long long in = in0 + t;
            if (in >= a.input_rows) in = a.input_rows - 1ull;
            acc[t] += (double)w * (double)((const float *)a.input)[in * a.input_stride + i];
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        double sum = acc[t];
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) sum += __shfl_xor(sum, offset, kWave);
        const unsigned long long in = in0 + t;
        if (in >= a.input_rows) continue;
        if (lane == 0u) matvec_publish(a, in, row, (float)sum);
    }
}

// F32, F16 or BF16 weight rows against fewer than eight F32 input rows (the router and mixing
// projections of a batch of one to seven tokens; a projection or an output head kept in 16-bit
// floats): the lane-strided kernel above walks a row one load at a time, a wave a row: a
// 256 x 7168 F32 router took 90 us of memory round trips, a 129 280 x 7168 F16 head streamed at
// 1.1 TB/s. Here a workgroup owns
// one weight row, its 256 threads take 16-byte pieces of it side by side (a 4 KB stretch a
// step), DEPTH steps of weight and input loads are in flight before the first product, and the
// four waves' double-precision sums are joined through LDS in wave order. Products and sums in
// double as above.
// ROW_WAVES: waves that share a row. One (four rows a workgroup, no barrier) for matrices of many rows, where the device
// is full either way and a workgroup a row is a launch and a barrier a row; sixteen where a row has a piece for each of
// their threads: the products are double-precision and one wave issues an instruction in five cycles, so four waves, one a
// SIMD, took longer over a row than the memory (256 x 7168
// by 3 / 5 / 7 rows 7.1 / 8.8 / 9.3 -> 5.7 / 6.7 / 8.0 us, 24 x 16384 by 1 / 3 / 7 4.8 / 8.9 / 9.0 -> 4.2 / 6.7 / 6.8).
template <unsigned QT, int T, int DEPTH, unsigned ROW_WAVES>
__global__ __launch_bounds__(ROW_WAVES == 1u ? 256u : 64u * ROW_WAVES) void matvec_scalar_few_kernel(MatvecArgs a)
{
    constexpr bool WAVE_ROW = ROW_WAVES == 1u;
    constexpr unsigned kSpan = 64u * ROW_WAVES;             // threads that share a row
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    constexpr int kColumns = QT == QT_F32 ? 4 : 8;           // weights in a 16-byte piece
    constexpr int kInputs = kColumns / 4;                    // 16-byte pieces of an input row beside it
    __shared__ double partial[ROW_WAVES][T];
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned long long row = WAVE_ROW ? (unsigned long long)blockIdx.x * 4ull + wave : blockIdx.x;
    const unsigned long long in0 = (unsigned long long)blockIdx.y * T;
    if (WAVE_ROW && row >= a.row_count) return;
    const unsigned self = WAVE_ROW ? lane : threadIdx.x;
    const v4u *w4 = reinterpret_cast<const v4u *>(a.encoded + row * a.row_bytes);
    const v4f *x4[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const unsigned long long in = in0 + t < a.input_rows ? in0 + t : a.input_rows - 1ull;   // clamped rows are never written
        x4[t] = reinterpret_cast<const v4f *>((const float *)a.input + in * a.input_stride);
    }
    const unsigned pieces = (unsigned)(a.row_width / kColumns);
    double acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = 0.0;
    unsigned bad = 0u;
    for (unsigned base = 0; base < pieces; base += kSpan * DEPTH) {
        const unsigned first = base + self;
        // steps of this turn that hold a piece for some thread (the same for the whole
        // workgroup: a step with none is not loaded at all, a short row costs what it holds)
        const unsigned steps = (pieces - base + kSpan - 1u) / kSpan;
        v4u raw[DEPTH];
        v4f x[T][DEPTH][kInputs];
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if ((unsigned)u < steps) {
                const unsigned at = first + kSpan * u < pieces ? first + kSpan * u : pieces - 1u;
                raw[u] = w4[at];
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int j = 0; j < kInputs; ++j) x[t][u][j] = x4[t][at * kInputs + j];
            } else {
                raw[u] = v4u{0u, 0u, 0u, 0u};
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int j = 0; j < kInputs; ++j) x[t][u][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            // (a thread past the end of the row repeated the last piece: its inputs count as
            // zeros. A branch here would pull each step's loads behind it, one wait a step)
            const bool live = first + kSpan * u < pieces;
            float w[kColumns];
#pragma unroll
            for (int c = 0; c < kColumns; ++c) {
                if constexpr (QT == QT_F32) {
                    w[c] = __uint_as_float(raw[u][c]);
                } else {
                    const unsigned bits = (raw[u][c >> 1] >> (16 * (c & 1))) & 0xffffu;
                    w[c] = QT == QT_BF16 ? __uint_as_float(bits << 16) : f16_bits_to_float(bits);
                }
                bad |= (unsigned)!finite_f32(w[c]);
            }
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int c = 0; c < kColumns; ++c)
                    acc[t] += (double)w[c] * (double)(live ? x[t][u][c >> 2][c & 3] : 0.0f);
        }
    }
    if (bad) raise_status(a.status, 1);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        acc[t] = wave_sum_f64(acc[t]);
        if (!WAVE_ROW && lane == 0u) partial[wave][t] = acc[t];
    }
    if constexpr (WAVE_ROW) {
        if (lane != 0u) return;
#pragma unroll
        for (int t = 0; t < T; ++t)
            if (in0 + t < a.input_rows) matvec_publish(a, in0 + t, row, (float)acc[t]);
        return;
    }
    __syncthreads();
    const unsigned t = threadIdx.x;          // a thread an input row
    if (t >= (unsigned)T || in0 + t >= a.input_rows) return;
    double sum = partial[0][t];
#pragma unroll
    for (unsigned w = 1; w < ROW_WAVES; ++w) sum += partial[w][t];
    matvec_publish(a, in0 + t, row, (float)sum);
}

template <unsigned QT, unsigned ROW_WAVES>
static int launch_scalar_few_rows(const MatvecArgs &a, hipStream_t s)
{
    constexpr unsigned kThreads = ROW_WAVES == 1u ? 256u : 64u * ROW_WAVES;
    constexpr int kDeep = ROW_WAVES == 16u ? 4 : 8;
    const unsigned long long grid_x = ROW_WAVES == 1u ? (a.row_count + 3ull) / 4ull : a.row_count;
    if (a.input_rows == 1ull)
        matvec_scalar_few_kernel<QT, 1, kDeep, ROW_WAVES><<<dim3((unsigned)grid_x, 1), kThreads, 0, s>>>(a);
    else if (a.input_rows == 2ull)
        matvec_scalar_few_kernel<QT, 2, kDeep, ROW_WAVES><<<dim3((unsigned)grid_x, 1), kThreads, 0, s>>>(a);
    else if (ROW_WAVES == 16u && a.input_rows > 4ull && 2ull * a.row_count > (unsigned long long)compute_units()) {
        // (all of them a workgroup, and its weight row once, unless two workgroups a row have a compute unit each)
        if constexpr (ROW_WAVES == 16u) {
            if (a.input_rows == 5ull) matvec_scalar_few_kernel<QT, 5, 2, 16><<<(unsigned)grid_x, kThreads, 0, s>>>(a);
            else if (a.input_rows == 6ull) matvec_scalar_few_kernel<QT, 6, 2, 16><<<(unsigned)grid_x, kThreads, 0, s>>>(a);
            else if (a.input_rows == 7ull) matvec_scalar_few_kernel<QT, 7, 2, 16><<<(unsigned)grid_x, kThreads, 0, s>>>(a);
            else return ST_BOUNDS;
        }
    } else
        matvec_scalar_few_kernel<QT, 4, kDeep / 2, ROW_WAVES><<<dim3((unsigned)grid_x, (unsigned)((a.input_rows + 3ull) / 4ull)),
                                                                kThreads, 0, s>>>(a);
    return check_launch("matvec_scalar_few");
}

template <unsigned QT>
static int launch_scalar_few(const MatvecArgs &a, hipStream_t s)
{
    // (sixteen waves a compute unit either way from 4096 rows on)
    if (a.row_count >= 4096ull) return launch_scalar_few_rows<QT, 1>(a, s);
    // sixteen waves a row while every row has a compute unit and its columns are work for them (four and sixteen: 256 x
    // 7168 by 2 rows 4.8 and 5.3 us, by 3 6.5 and 5.8; 256 x 4096 by 5 5.4 and 6.9; 1000 x 4096 by 1 6.7 and 9.1)
    if constexpr (QT == QT_F32)
        if (a.row_count <= (unsigned long long)compute_units() &&
            (a.row_width >= 16384ull || (a.row_width >= 6144ull && a.input_rows >= 3ull)))
            return launch_scalar_few_rows<QT, 16>(a, s);
    return launch_scalar_few_rows<QT, 4>(a, s);
}

// F32 weight rows against a batch of F32 input rows (a router or mixing projection over a row
// batch) on the double-precision matrix cores: a workgroup of WAVES waves owns 16 weight rows x
// 16 input rows on V_MFMA_F64_16X16X4_F64 and its waves split the row width. Lane (i, q) loads
// four consecutive floats of weight row i and of input row i at offset 16 j + 4 q. A product of
// two floats is exact in double and the sums run in double, which is how the CPU row dot forms
// them (src/gguf/quant_compute.c:152-172); only the order of the double additions differs from
// its serial loop, so the float the sum rounds to is the CPU path's. The partial tiles of the
// waves (and of the workgroups that split the width: blockIdx.z, joined by a second launch in
// split order) are doubles, added in a fixed order.
// Four consecutive weights (column a multiple of four) of a row of F32, F16 or BF16 values, or of
// Q8_0 blocks (scale times code, exact in float: the value the CPU decoder forms,
// src/gguf/quant_block.c:715-881), as floats.
template <unsigned QT>
__device__ __forceinline__ float4 scalar_weights4(const unsigned char *row, unsigned long long column)
{
    if constexpr (QT == QT_F32) {
        return *reinterpret_cast<const float4 *>(row + 4ull * column);
    } else if constexpr (QT == QT_Q8_0) {
        const unsigned char *block = row + 34ull * (column >> 5);
        const float d = f16_bits_to_float(*reinterpret_cast<const unsigned short *>(block));
        const unsigned char *codes = block + 2u + (unsigned)(column & 31ull);      // on a 2-byte boundary
        const unsigned lo = *reinterpret_cast<const unsigned short *>(codes);
        const unsigned hi = *reinterpret_cast<const unsigned short *>(codes + 2);
        return make_float4(d * (float)(signed char)(lo & 255u), d * (float)(signed char)(lo >> 8),
                           d * (float)(signed char)(hi & 255u), d * (float)(signed char)(hi >> 8));
    } else {
        const uint2 v = *reinterpret_cast<const uint2 *>(row + 2ull * column);
        if constexpr (QT == QT_F16)
            return make_float4(f16_bits_to_float(v.x & 0xffffu), f16_bits_to_float(v.x >> 16),
                               f16_bits_to_float(v.y & 0xffffu), f16_bits_to_float(v.y >> 16));
        else
            return make_float4(bf16_bits_to_float(v.x & 0xffffu), bf16_bits_to_float(v.x >> 16),
                               bf16_bits_to_float(v.y & 0xffffu), bf16_bits_to_float(v.y >> 16));
    }
}

template <unsigned WAVES, unsigned QT = QT_F32>
__global__ __launch_bounds__(WAVES * 64) void matvec_f32_tile16_kernel(MatvecArgs a)
{
    typedef double v4d __attribute__((ext_vector_type(4)));
    __shared__ double partial[WAVES - 1u][4][64];
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned i16 = lane & 15u, q = lane >> 4;
    unsigned long long wrow = (unsigned long long)blockIdx.x * 16ull + i16;
    unsigned long long in = (unsigned long long)blockIdx.y * 16ull + i16;
    if (wrow >= a.row_count) wrow = a.row_count - 1ull;      // a ragged edge repeats the last row
    if (in >= a.input_rows) in = a.input_rows - 1ull;
    const unsigned long long share = a.row_width / ((unsigned long long)gridDim.z * WAVES);   // a multiple of 16
    const unsigned long long begin = ((unsigned long long)blockIdx.z * WAVES + wave) * share + 4u * q;
    const unsigned char *wp = a.encoded + wrow * a.row_bytes;       // columns from `begin` on
    const float *xp = (const float *)a.input + in * a.input_stride + begin;
    const unsigned steps = (unsigned)(share / 16ull);
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    unsigned bad = 0u;
    // four steps of loads stay in flight ahead of the matrix instructions that use them
    const unsigned groups = (steps + 3u) / 4u;
    float4 w[4], x[4];
#pragma unroll
    for (unsigned j = 0; j < 4u; ++j) {
        const unsigned at = 16u * (j < steps ? j : steps - 1u);
        w[j] = scalar_weights4<QT>(wp, begin + at);
        x[j] = *reinterpret_cast<const float4 *>(xp + at);
    }
    for (unsigned group = 0; group < groups; ++group) {
        float4 wn[4], xn[4];
        if (group + 1u < groups) {
#pragma unroll
            for (unsigned j = 0; j < 4u; ++j) {
                const unsigned step = 4u * (group + 1u) + j;
                const unsigned at = 16u * (step < steps ? step : steps - 1u);
                wn[j] = scalar_weights4<QT>(wp, begin + at);
                xn[j] = *reinterpret_cast<const float4 *>(xp + at);
            }
        }
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) {
            if (4u * group + j >= steps) break;
            bad |= (unsigned)!finite_f32(w[j].x) | (unsigned)!finite_f32(w[j].y) |
                   (unsigned)!finite_f32(w[j].z) | (unsigned)!finite_f32(w[j].w);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)w[j].x, (double)x[j].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)w[j].y, (double)x[j].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)w[j].z, (double)x[j].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)w[j].w, (double)x[j].w, acc, 0, 0, 0);
        }
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) {
            w[j] = wn[j];
            x[j] = xn[j];
        }
    }
    if (bad) raise_status(a.status, 1);
    if (wave) {
#pragma unroll
        for (int k = 0; k < 4; ++k) partial[wave - 1u][k][lane] = acc[k];
    }
    __syncthreads();
    if (wave) return;
    const unsigned long long out_in = (unsigned long long)blockIdx.y * 16ull + i16;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        // accumulator k of lane (i, q): weight row 4 k + q, input row i
        const unsigned long long row = (unsigned long long)blockIdx.x * 16ull + 4u * k + q;
        double sum = acc[k];
#pragma unroll
        for (unsigned wv = 0; wv + 1u < WAVES; ++wv) sum += partial[wv][k][lane];
        if (row >= a.row_count || out_in >= a.input_rows) continue;
        if (a.parts) {
            a.parts[((unsigned long long)blockIdx.z * a.input_rows + out_in) * a.row_count + row] = sum;
            continue;
        }
        matvec_publish(a, out_in, row, (float)sum);
    }
}

// The same product for a batch of input rows on tiles of 32 weight rows x INPUTS input rows whose waves split the row
// width (and workgroups do: blockIdx.z, as above). The matrix instructions bound it: 64 cycles each, 54 us of the
// device for 256 x 7168 by 1111 rows. So the operands must come at half the bytes and a quarter of the cache lines that
// a 16 x 16 tile asks for: a wave loads 32 columns of its tile's rows as consecutive 16-byte pieces, eight lanes a row,
// 32 columns ahead, passes them through a window of LDS of its own (144 bytes a row: the sixteen rows that a read
// touches lie on different banks) and needs no barrier before the sums are added.
// 256 x 7168 by 64 / 256 / 512 / 1111 / 2048 rows 18.7 / 38.6 / 62.6 / 136 / 168 us -> 14.0 / 25.0 / 40.8 / 87.0 / 131, with
// the join. A vector instruction and a matrix instruction on doubles never run together (SQ_VALU_MFMA_COEXEC_CYCLES is zero), so the
// vector instructions that are left count in full. Weights tested by one input tile's workgroups and conversions in batches:
// 256 x 7168 by 1111 / 1500 / 2048 rows of a layer 102 / 117 / 160 -> 100 / 110 / 151 us, 256 x 4096 and 24 x 16384 by 333
// 21.4 and 16.1 -> 20.0 and 15.2, level up to 96. (Two or three chunks ahead instead of one: registers of the second
// workgroup, 160 -> 181; the eight workgroups of an input tile on one XCD: level.)
constexpr unsigned kTile32Columns = 32u, kTile32Pitch = kTile32Columns * 4u + 16u, kTile32Waves = 8u;

template <unsigned QT, unsigned INPUTS>
__global__ __launch_bounds__(kTile32Waves * 64) void matvec_f32_tile32_kernel(MatvecArgs a)
{
    constexpr unsigned WAVES = kTile32Waves;
    typedef double v4d __attribute__((ext_vector_type(4)));
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr unsigned kRows = 32u + INPUTS, kWindow = kRows * kTile32Pitch, kTiles = INPUTS / 8u;
    constexpr unsigned kInputLoads = INPUTS / 8u;
    // Columns whose operands are converted together, ahead of eight matrix instructions that then follow one another: no
    // vector instruction issues while one of them runs, and between two of them a conversion and its wait states are a gap.
    constexpr unsigned kBatch = INPUTS == 16u ? 4u : 2u;
    static_assert((WAVES - 1u) * kTiles * 4u * 64u * 8u <= WAVES * kWindow, "the partial sums fit the windows");
    __shared__ __align__(16) unsigned char windows[WAVES * kWindow];
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned i16 = lane & 15u, q = lane >> 4;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 32ull, in0 = (unsigned long long)blockIdx.y * INPUTS;
    const unsigned weights_here = (unsigned)(a.row_count - row0 < 32ull ? a.row_count - row0 : 32ull);
    const unsigned inputs_here = (unsigned)(a.input_rows - in0 < INPUTS ? a.input_rows - in0 : INPUTS);
    unsigned char *const window = windows + wave * kWindow;
    // the lane's pieces: columns 4 (lane % 8) .. + 3 of rows lane / 8 + 8 k (a ragged edge repeats the last row)
    const unsigned piece = lane & 7u;
    const unsigned char *weight_at[4];
    const float *input_at[kInputLoads];
#pragma unroll
    for (unsigned k = 0; k < 4u; ++k) {
        const unsigned row = 8u * k + (lane >> 3);
        weight_at[k] = a.encoded + (row0 + (row < weights_here ? row : weights_here - 1u)) * a.row_bytes;
    }
#pragma unroll
    for (unsigned k = 0; k < kInputLoads; ++k) {
        const unsigned row = 8u * k + (lane >> 3);
        input_at[k] = (const float *)a.input + (in0 + (row < inputs_here ? row : inputs_here - 1u)) * a.input_stride + 4u * piece;
    }
    unsigned char *const to = window + (lane >> 3) * kTile32Pitch + 16u * piece;
    const unsigned char *const from = window + i16 * kTile32Pitch + 16u * q;
    const unsigned chunks = (unsigned)(a.row_width / kTile32Columns), shares = gridDim.z * WAVES;
    const unsigned share = blockIdx.z * WAVES + wave;
    const unsigned begin = (unsigned)((unsigned long long)chunks * share / shares);
    const unsigned end = (unsigned)((unsigned long long)chunks * (share + 1u) / shares);
    v4f weights[4], inputs[kInputLoads];
    unsigned bad = 0u;
    auto request = [&](unsigned chunk) {
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            const float4 w = scalar_weights4<QT>(weight_at[k], (unsigned long long)chunk * kTile32Columns + 4u * piece);
            weights[k] = v4f{w.x, w.y, w.z, w.w};
        }
#pragma unroll
        for (unsigned k = 0; k < kInputLoads; ++k)
            inputs[k] = *reinterpret_cast<const v4f *>(input_at[k] + (unsigned long long)chunk * kTile32Columns);
    };
    v4d acc[kTiles];
#pragma unroll
    for (unsigned t = 0; t < kTiles; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
    if (begin < end) request(begin);
    for (unsigned chunk = begin; chunk < end; ++chunk) {
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) *reinterpret_cast<v4f *>(to + 8u * k * kTile32Pitch) = weights[k];
        // (vector instructions take the time of the matrix cores here: one input tile's workgroups test the weights for all)
        if (blockIdx.y == 0u) {
#pragma unroll
            for (unsigned k = 0; k < 4u; ++k)
                bad |= (unsigned)!finite_f32(weights[k][0]) | (unsigned)!finite_f32(weights[k][1]) |
                       (unsigned)!finite_f32(weights[k][2]) | (unsigned)!finite_f32(weights[k][3]);
        }
#pragma unroll
        for (unsigned k = 0; k < kInputLoads; ++k) *reinterpret_cast<v4f *>(to + (32u + 8u * k) * kTile32Pitch) = inputs[k];
        request(chunk + 1u < end ? chunk + 1u : chunk);       // (the last turn's are not used)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (unsigned step = 0; step < kTile32Columns / 16u; ++step) {
            v4f w[2], x[INPUTS / 16u];
#pragma unroll
            for (unsigned m = 0; m < 2u; ++m) w[m] = *reinterpret_cast<const v4f *>(from + 16u * m * kTile32Pitch + 64u * step);
#pragma unroll
            for (unsigned n = 0; n < INPUTS / 16u; ++n)
                x[n] = *reinterpret_cast<const v4f *>(from + (32u + 16u * n) * kTile32Pitch + 64u * step);
#pragma unroll
            for (unsigned at = 0; at < 4u; at += kBatch) {
                double wide[kBatch][2], in[kBatch][INPUTS / 16u];
#pragma unroll
                for (unsigned c = 0; c < kBatch; ++c) {
#pragma unroll
                    for (unsigned m = 0; m < 2u; ++m) wide[c][m] = (double)w[m][at + c];
#pragma unroll
                    for (unsigned n = 0; n < INPUTS / 16u; ++n) in[c][n] = (double)x[n][at + c];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (unsigned c = 0; c < kBatch; ++c)
#pragma unroll
                    for (unsigned t = 0; t < kTiles; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wide[c][t & 1u], in[c][t >> 1], acc[t], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (bad) raise_status(a.status, 1);
    __syncthreads();
    double *const partial = reinterpret_cast<double *>(windows);
    if (wave) {
#pragma unroll
        for (unsigned t = 0; t < kTiles; ++t)
#pragma unroll
            for (unsigned k = 0; k < 4u; ++k) partial[(((wave - 1u) * kTiles + t) * 4u + k) * 64u + lane] = acc[t][k];
    }
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (unsigned t = 0; t < kTiles; ++t) {
        const unsigned long long in = in0 + 16u * (t >> 1) + i16;
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            // accumulator k of lane (i, q): weight row 4 k + q of the tile, input row i
            const unsigned long long row = row0 + 16u * (t & 1u) + 4u * k + q;
            double sum = acc[t][k];
#pragma unroll
            for (unsigned other = 0; other + 1u < WAVES; ++other) sum += partial[((other * kTiles + t) * 4u + k) * 64u + lane];
            if (row >= a.row_count || in >= a.input_rows) continue;
            if (a.parts) a.parts[((unsigned long long)blockIdx.z * a.input_rows + in) * a.row_count + row] = sum;
            else matvec_publish(a, in, row, (float)sum);
        }
    }
}

// Second launch of a split projection: the partial sums of one output added in split order.
__global__ __launch_bounds__(256) void matvec_f32_join_kernel(MatvecArgs a, unsigned splits)
{
    const unsigned long long outputs = a.input_rows * a.row_count;
    const unsigned long long at = (unsigned long long)blockIdx.x * 256ull + threadIdx.x;
    if (at >= outputs) return;
    const unsigned long long in = at / a.row_count, row = at % a.row_count;
    double sum = a.parts[at];
    for (unsigned z = 1; z < splits; ++z) sum += a.parts[z * outputs + at];
    matvec_publish(a, in, row, (float)sum);
    if (a.scores) {
        // the router's score of this logit: the routing launch behind this one then has no
        // double-precision exponentials left in its one workgroup
        const double s = route_score((double)(float)sum, a.scoring);
        const float published = (float)s;
        if (!(s == s) || !finite_f32(published)) raise_status(a.status, 1);
        a.scores[in * a.row_count + row] = published;
    }
}

// The second launch of a router's split projection: one workgroup joins a row's partial sums, scores
// them and routes the row, a thread an expert and then one wavefront (route.hpp). With the rows'
// routing in workgroups of their own the launch behind this one is left with the worklist; when its
// one routing workgroup took sixteen rows at a time, 96 rows cost 26 us there, 9 us now.
__global__ __launch_bounds__(256) void matvec_f32_join_route_kernel(
    MatvecArgs a, unsigned splits, const float *__restrict__ bias, unsigned topk, int normalize, double scaling,
    unsigned long long *__restrict__ selected, float *__restrict__ weights)
{
    __shared__ float scores[256];
    const unsigned experts = (unsigned)a.row_count, e = threadIdx.x;
    const unsigned long long in = blockIdx.x, outputs = a.input_rows * a.row_count, at = in * a.row_count + e;
    RouteInputs row;
    if (e < 64u)
#pragma unroll
        for (unsigned i = 0; i < 4u; ++i)          // the biases: on their way meanwhile
            row.bias[i] = bias ? bias[4u * e + i < experts ? 4u * e + i : experts - 1u] : 0.0f;
    if (e < experts) {
        double part[16], sum = 0.0;
#pragma unroll
        for (unsigned z = 0; z < 16u; ++z) part[z] = z < splits ? a.parts[z * outputs + at] : 0.0;
        sum = part[0];
#pragma unroll
        for (unsigned z = 1; z < 16u; ++z)
            if (z < splits) sum += part[z];
        for (unsigned z = 16u; z < splits; ++z) sum += a.parts[z * outputs + at];
        matvec_publish(a, in, e, (float)sum);
        const double s = route_score((double)(float)sum, a.scoring);
        const float published = (float)s;
        if (!(s == s) || !finite_f32(published)) raise_status(a.status, 1);
        scores[e] = published;
    }
    __syncthreads();
    if (e >= 64u) return;
#pragma unroll
    for (unsigned i = 0; i < 4u; ++i) row.value[i] = scores[4u * e + i < experts ? 4u * e + i : experts - 1u];
    route_row(row, true, in, e, experts, topk, a.scoring, normalize, scaling, selected, weights, a.status);
}

// int32 block sums of the Q8_K path, produced by the same unit code the matvec runs.
template <unsigned QT>
__global__ __launch_bounds__(256) void block_dots_kernel(
    const unsigned char *encoded, unsigned long long row_count, unsigned long long row_width,
    unsigned long long row_bytes, const unsigned char *input, unsigned long long input_rows,
    int *sums)
{
    __shared__ Iq2Tables tables;
    if constexpr (QT == QT_IQ2_XXS) {
        iq2_tables_fill(tables);
        __syncthreads();
    }
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long row = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    const unsigned long long in = blockIdx.y;
    if (row >= row_count || in >= input_rows) return;
    const unsigned char *wrow = encoded + row * row_bytes;
    const unsigned units = (unsigned)(row_width >> 5);
    const unsigned long long blocks = row_width >> 8;
    for (unsigned base = 0; base < units; base += 64u) {
        const unsigned u = base + lane;
        const bool live = u < units;
        const unsigned uu = live ? u : units - 1u;
        Unit unit;
        unit_load<QT>(tables, wrow, uu, unit);
        const unsigned char *act = input + (in * blocks + (uu >> 3)) * kQ8KBytes;
        UnitSum s = unit_dot_q8<QT>(unit, act, uu & 7u);
        if constexpr (UnitTraits<QT>::kIntegerCombine) {
            if (!live) s.dot = s.min = 0;
            s.dot = group_sum_i32<8>(s.dot);
            s.min = group_sum_i32<8>(s.min);
            if (live && (uu & 7u) == 0u) {
                int *o = sums + ((in * row_count + row) * blocks + (uu >> 3)) * 2ull;
                o[0] = s.dot;
                o[1] = s.min;
            }
        } else if (live) {
            sums[(in * row_count + row) * blocks * 8ull + uu] = s.dot;
        }
    }
}

// Serial double-precision row dot by one thread, element by element: the parity probe of the
// qtype decoders (src/backend/cuda/kernels.cu:112-124). Same order and arithmetic as the CPU row
// dot, so the two agree to the last bit wherever the decoders do.
__global__ void row_dot_serial_kernel(const unsigned char *__restrict__ encoded,
                                      const float *__restrict__ vector, unsigned long long elements,
                                      unsigned qtype, float *out)
{
    if (blockIdx.x != 0u || threadIdx.x != 0u) return;
    double sum = 0.0;
    for (unsigned long long index = 0; index < elements; ++index)
        sum += (double)qtype_value(encoded, index, qtype) * (double)vector[index];
    out[0] = (float)sum;
}

__global__ __launch_bounds__(256) void gather_kernel(
    const unsigned char *encoded, unsigned qtype, unsigned long long row_count,
    unsigned long long row_width, unsigned long long row_bytes, const unsigned *row_ids,
    unsigned long long selected, float *out, int *status)
{
    const unsigned long long index = (unsigned long long)blockIdx.x * 256ull + threadIdx.x;
    if (index >= selected * row_width) return;
    const unsigned long long s = index / row_width, column = index % row_width;
    const unsigned long long row = row_ids ? row_ids[s] : s;
    if (row >= row_count) {
        raise_status(status, 2);
        return;
    }
    const float value = qtype_value(encoded + row * row_bytes, column, qtype);
    if (!finite_f32(value)) raise_status(status, 1);
    else out[index] = value;
}

template <unsigned QT, bool Q8, bool EVEN>
static int launch_block_even(const MatvecArgs &a, hipStream_t stream)
{
    const unsigned long long grid_x = (a.row_count + 3ull) / 4ull;
    const unsigned grid_z = a.encoded_second ? 2u : 1u;
    if (grid_x > 0x7fffffffull) return ST_BOUNDS;
    if (a.input_rows == 1ull) {
        // Q8_K activations: four chunks (8192 columns) in flight for a matrix that takes many
        // rounds of waves, and for rows of more than one chunk, whose chunks would otherwise each
        // wait a memory round trip of their own
        const bool deep = Q8 && (a.row_count * a.row_bytes >= (64ull << 20) || a.row_width > 2048ull);
        // one F32 input row of up to 12 288 values (48 KB) is staged in LDS
        const bool stage = !Q8 && a.row_width <= 12288ull && !((uintptr_t)a.input & 15u);
        if (deep) matvec_block_kernel<QT, Q8, 1, Q8 ? 4 : 1, EVEN><<<dim3((unsigned)grid_x, 1, grid_z), 256, 0, stream>>>(a);
        else if (stage)
            matvec_block_kernel<QT, Q8, 1, 1, EVEN, !Q8><<<dim3((unsigned)grid_x, 1, grid_z), 256,
                                                            (size_t)a.row_width * 4u, stream>>>(a);
        else matvec_block_kernel<QT, Q8, 1, 1, EVEN><<<dim3((unsigned)grid_x, 1, grid_z), 256, 0, stream>>>(a);
    } else {
        const unsigned long long grid_y = (a.input_rows + 3ull) / 4ull;
        if (grid_y > 65535ull) return ST_BOUNDS;
        matvec_block_kernel<QT, Q8, 4, 1, EVEN><<<dim3((unsigned)grid_x, (unsigned)grid_y, grid_z), 256, 0, stream>>>(a);
    }
    return check_launch("matvec");
}

// Rows of up to 4096 columns, of which a workgroup has eight or more, end the operation by themselves; longer ones take a wave
// each, and the four of a workgroup are too little to wait for. us a call, published by the launch and behind it: 8192 x 4096 by
// 1 / 3 rows Q4_K 15.7 / 22.9 and 16.0 / 22.7, 65536 x 1024 by 1 / 3 17.9 / 30.8 and 18.4 / 31.0, 16384 x 4096 by 1 18.6 and 19.2; but 4096 x 7168 by
// 1 / 2 / 3 16.5 / 21.5 / 24.0 and 16.4 / 20.5 / 22.5, 1024 x 7168 by 1 13.9 and 13.8, IQ2_XXS 6144 x 7168 by 1 / 3 18.6 / 26.2 and 18.3 / 25.5.
constexpr uint64_t row_publishing_groups(int lanes_a_row) { return lanes_a_row < 64 ? kPublishingGroups : 0u; }

template <unsigned QT, int L>
static int launch_dense_row(MatvecArgs &a, hipStream_t stream, Publisher *publisher)
{
    const unsigned long long grid = (a.row_count + 4ull * (64u / L) - 1ull) / (4ull * (64u / L));
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    a.publication = take_publication(publisher, grid, row_publishing_groups(L));
    dense_row_q8k_kernel<QT, L><<<(unsigned)grid, 256, 0, stream>>>(a);
    return check_launch("matvec.row");
}

// One Q8_K input row against superblock-format rows on dword boundaries: the row kernel, whatever
// the size of the matrix (a 470 MB Q4_K matrix streams at 4.8 TB/s through it, at 2.4 TB/s
// through the general kernel, whose lanes wait for the superblock header on their own).
template <unsigned QT>
static bool dense_row_applies(const MatvecArgs &a)
{
    return UnitTraits<QT>::kIntegerCombine && a.input_rows == 1ull &&
           !((unsigned long long)a.encoded & 3ull) && !(a.row_bytes & 3ull);
}

template <unsigned QT, int L>
static int launch_dense_fewrows(MatvecArgs &a, hipStream_t stream, Publisher *publisher)
{
    const unsigned long long grid = (a.row_count + 4ull * (64u / L) - 1ull) / (4ull * (64u / L));
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    a.publication = take_publication(publisher, grid, row_publishing_groups(L));
    dense_fewrows_q8k_kernel<QT, L><<<(unsigned)grid, 256, 0, stream>>>(a);
    return check_launch("matvec.fewrows");
}

template <unsigned QT>
static bool dense_fewrows_applies(const MatvecArgs &a)
{
    // (measured against the general kernel on 2048 x 7168 and 7168 x 2048 matrices: ahead up to
    // a dozen input rows, and at any number below 32 where a row is 2048 columns or fewer)
    return UnitTraits<QT>::kIntegerCombine && a.input_rows >= 2ull && a.input_rows < 32ull &&
           (a.input_rows <= 12ull || a.row_width <= 2048ull) &&
           a.row_width <= 8192ull && a.row_count * a.row_bytes < (64ull << 20) &&
           !((unsigned long long)a.encoded & 3ull) && !(a.row_bytes & 3ull);
}

template <unsigned QT>
static int launch_dense_fewrows_width(MatvecArgs &a, hipStream_t stream, Publisher *publisher)
{
    const unsigned long long halves = a.row_width >> 7;
    if (halves <= 8ull) return launch_dense_fewrows<QT, 8>(a, stream, publisher);
    if (halves <= 16ull) return launch_dense_fewrows<QT, 16>(a, stream, publisher);
    if (halves <= 32ull) return launch_dense_fewrows<QT, 32>(a, stream, publisher);
    return launch_dense_fewrows<QT, 64>(a, stream, publisher);
}

template <unsigned QT>
static int launch_dense_row_width(MatvecArgs &a, hipStream_t stream, Publisher *publisher)
{
    const unsigned long long halves = a.row_width >> 7;
    if (halves <= 8ull) return launch_dense_row<QT, 8>(a, stream, publisher);
    if (halves <= 16ull) return launch_dense_row<QT, 16>(a, stream, publisher);
    if (halves <= 32ull) return launch_dense_row<QT, 32>(a, stream, publisher);
    return launch_dense_row<QT, 64>(a, stream, publisher);
}

template <unsigned QT, bool Q8>
static int launch_block(MatvecArgs &a, hipStream_t stream, Publisher *publisher)
{
    if constexpr (Q8 && UnitTraits<QT>::kIntegerCombine) {
        if (dense_row_applies<QT>(a)) return launch_dense_row_width<QT>(a, stream, publisher);
        if (dense_fewrows_applies<QT>(a)) return launch_dense_fewrows_width<QT>(a, stream, publisher);
    }
    const bool even = (((unsigned long long)a.encoded | a.row_bytes) & 1ull) == 0ull;
    return even ? launch_block_even<QT, Q8, true>(a, stream) : launch_block_even<QT, Q8, false>(a, stream);
}

template <unsigned QT>
static int launch_block_q(MatvecArgs &a, bool q8, hipStream_t stream, Publisher *publisher)
{
    return q8 ? launch_block<QT, true>(a, stream, publisher) : launch_block<QT, false>(a, stream, publisher);
}

}  // namespace yvex

using namespace yvex;

// How the tiles of 32 weight rows take a projection: input rows a tile, and workgroups that share a tile's row width.
struct ScalarTiles {
    unsigned inputs, splits;
    double us;
};

// The launch takes as long as the workgroups of the fullest compute unit: 65 us for 32 x 32 outputs of 7168 columns,
// 35 for 32 x 16. A split costs the join 0.3 us and its sums, written and read, 16 bytes an output at the
// 10 TB/s of the caches; the join itself is a launch. Measured, 256 weight rows: 1111 input rows in 1, 2, 3 and 4 splits 129, 101, 93
// and 89 us; 4096 columns by 96 in 4 and 8 splits of 16-row tiles 12.5 and 14.2, of 32-row tiles 17.2 and 14.6.
static ScalarTiles scalar_tiles(uint64_t row_count, uint64_t row_width, uint64_t input_rows,
                                unsigned least, unsigned most)
{
    const uint64_t cus = (uint64_t)compute_units(), rows = (row_count + 31u) / 32u, chunks = row_width / kTile32Columns;
    const double split_us = 0.3 + (double)row_count * (double)input_rows * 1.6e-6;
    ScalarTiles best{0u, 0u, 0.0};
    for (unsigned inputs = 16u; inputs <= 32u; inputs += 16u) {
        const uint64_t tiles = rows * ((input_rows + inputs - 1u) / inputs);
        const double chunk_us = inputs == 16u ? 35.0 / 28.0 : 65.0 / 28.0;      // of a wave: 28 are 7168 columns
        // (every wave has columns)
        for (unsigned z = least; z <= most && (z == least || (uint64_t)z * kTile32Waves <= chunks); ++z) {
            const uint64_t waves = (uint64_t)z * kTile32Waves;
            const double us = chunk_us * (double)((tiles * z + cus - 1u) / cus) * (double)((chunks + waves - 1u) / waves) +
                              (z > 1u ? 4.0 + split_us * z : 0.0);
            if (!best.inputs || us < best.us) best = ScalarTiles{inputs, z, us};
        }
    }
    return best;
}

template <unsigned QT>
static int launch_scalar_tiles(const MatvecArgs &a, ScalarTiles tiles, hipStream_t s)
{
    const uint64_t grid_x = (a.row_count + 31ull) / 32ull, grid_y = (a.input_rows + tiles.inputs - 1ull) / tiles.inputs;
    if (grid_x > 0x3fffffffull || (a.input_rows + 15ull) / 16ull > 65535ull) return ST_BOUNDS;
    const dim3 grid((unsigned)grid_x, (unsigned)grid_y, tiles.splits);
    if (tiles.inputs == 16u) matvec_f32_tile32_kernel<QT, 16><<<grid, 64u * kTile32Waves, 0, s>>>(a);
    else matvec_f32_tile32_kernel<QT, 32><<<grid, 64u * kTile32Waves, 0, s>>>(a);
    return check_launch("matvec_f32_tile32");
}

// Rows of F32, F16 or BF16 values against eight or more F32 input rows on the double-precision matrix cores:
// a small batch offers few tiles, so sixteen waves of a 16 x 16 tile split the row width, a larger one runs on the
// 32-row tiles.
template <unsigned QT>
static int launch_scalar_rows(const MatvecArgs &a, hipStream_t s)
{
    if (a.input_rows >= 256ull)
        return launch_scalar_tiles<QT>(a, scalar_tiles(a.row_count, a.row_width, a.input_rows, 1u, 1u), s);
    const unsigned long long grid_x = (a.row_count + 15ull) / 16ull, grid_y = (a.input_rows + 15ull) / 16ull;
    if (grid_x > 0x7fffffffull || grid_y > 65535ull) return ST_BOUNDS;
    matvec_f32_tile16_kernel<16, QT><<<dim3((unsigned)grid_x, (unsigned)grid_y), 1024, 0, s>>>(a);
    return check_launch("matvec_f32_tile16");
}

static bool q8_0_takes_matrix_cores(const uint8_t *encoded, uint64_t row_count, uint64_t row_bytes,
                                    uint64_t input_rows)
{
    const unsigned long long matrix_bytes = row_count * row_bytes;
    return !((uintptr_t)encoded & 3u) &&
           (input_rows >= (matrix_bytes < (2ull << 20) ? 12ull : 10ull) ||
            (input_rows >= 2ull && matrix_bytes >= (8ull << 20)));
}

static int launch_matvec(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                         uint64_t row_width, uint64_t row_bytes, const void *input,
                         int input_q8, uint64_t input_rows, uint64_t input_stride,
                         const float *additive, float *out, uint64_t out_stride,
                         int output_bf16, int *status, yvex_hip_stream stream, Publisher *publisher)
{
    unsigned block, bytes;
    if (!encoded || !input || !out || !status || !row_count || !row_width || !input_rows ||
        out_stride < row_count || (input_q8 != 0 && input_q8 != 1))
        return ST_INVALID_ARG;
    if (!qtype_geometry(qtype, block, bytes)) return ST_UNSUPPORTED;
    if (row_width % block || row_width / block * bytes != row_bytes) return ST_BOUNDS;
    if (row_width > 0xffffffffull * 32ull) return ST_BOUNDS;
    if (((uintptr_t)input & 3u) || ((uintptr_t)out & 3u)) return ST_INVALID_ARG;
    MatvecArgs a{encoded, row_count, row_width, row_bytes, input, input_rows, input_stride,
                 additive, out, out_stride, output_bf16, status, nullptr, nullptr, 0};
    hipStream_t s = as_stream(stream);
    const bool scalar = qtype == QT_F32 || qtype == QT_F16 || qtype == QT_BF16 || qtype == QT_I32;
    if (input_q8 && (scalar || row_width % 256u)) return ST_UNSUPPORTED;
    if (!input_q8) {
        if (input_stride < row_width) return ST_INVALID_ARG;
        if (!scalar && (((uintptr_t)input & 15u) || (input_stride & 3u))) return ST_INVALID_ARG;
    }
    // IQ2_XXS rows against a batch of Q8_K input rows: 16 x 16 tiles whose waves share the row width where the matrix is
    // small (dense_iq2.hip has the line), else the int8 matrix-core kernels of the
    // row-batch expert path, as one bucket that holds every input row (the reference turns its
    // tensor-core kernels on from 16 input rows, src/backend/cuda/private.h:461-464). The time of the sweep
    // below grows with the products, theirs stands while the tiles come out at one round, so below 32
    // input rows their line lies at a number of products (sweep and these, us): 7168 x 7168 by 8 31.7 and 32.0, by 12 45.1 and
    // 32.6; 32 768 x 4096 by 8 72 and 27, by 31 260 and 32; 129 280 x 7168 by 8 508 and 118, by 31
    // 1813 and 125. Same exact int32 superblock sums and the same float terms as the sweep, added in
    // double there and here: the same bits.
    const bool iq2_batch = input_rows >= 32ull || iq2_rows_small(row_count, row_width, input_rows) || (input_rows >= 8ull && row_width >= 512ull &&
                                                   row_count >= (73728ull + input_rows - 1ull) / input_rows);
    if (qtype == QT_IQ2_XXS && input_q8 && iq2_batch && !additive &&
        out_stride == row_count && row_count % 4ull == 0ull && !((uintptr_t)encoded & 3u) &&
        !(row_bytes & 3ull) && row_width / 32ull <= 64ull * 4ull && !((uintptr_t)out & 15u))
        return launch_iq2_rows_dense(encoded, row_count, row_width, row_bytes, input, input_rows, out,
                                     output_bf16 != 0, status, s, publisher);
    // Q4_K rows against two or more Q8_K input rows: matrix cores (the reference's threshold is 16
    // input rows; here the 16-token tiles beat the general kernel below from two rows on, 10.5 us
    // against 12.2 us at 2 and 19.7 us at 15 rows for 2048 x 7168; the few-rows kernel, where it
    // applies, is ahead of both at two and three rows: 6.0 and 7.1 us against 8.6)
    if (qtype == QT_Q4_K && input_q8 && input_rows >= 2ull && !((uintptr_t)encoded & 15u) &&
        !(input_rows < 4ull && dense_fewrows_applies<QT_Q4_K>(a)))
        return launch_q4k_rows_dense(encoded, row_count, row_width, row_bytes, input, input_rows, additive,
                                     out, out_stride, output_bf16 != 0, status, s, publisher);
    // Q8_0 rows against a batch of Q8_K input rows: matrix cores (the reference's threshold is 16 rows,
    // src/backend/cuda/private.h:461-464); the lane-strided kernel reads the matrix once per four input rows, which
    // matrices of under 8 MB bear up to nine (lane-strided and matrix cores: 1024 x 4096 by 4 / 8 / 10 / 12 rows 5.3 / 6.0 /
    // 7.0 / 7.2 and 6.5 / 6.7 / 6.9 / 7.1 us, 512 x 2048 by 10 4.4 and 4.7), larger ones not from two on (2048 x 4096 by 4 6.9
    // and 6.8, 4096 x 4096 by 2 / 8 9.8 / 14.7 and 7.7 / 8.1, 7168 x 7168 by 2 19.2 and 16.6)
    if (qtype == QT_Q8_0 && input_q8 && q8_0_takes_matrix_cores(encoded, row_count, row_bytes, input_rows))
        return launch_q8_0_rows_dense(encoded, row_count, row_width, row_bytes, input, input_rows, additive, out,
                                      out_stride, output_bf16 != 0, status, s, nullptr, nullptr, publisher);
    // F32 rows against a batch of F32 input rows: the double-precision matrix cores; rows of F16
    // and BF16 values take the same kernels (the conversion to double is exact for them as well),
    // and so do Q8_0 rows against F32 input rows (a caller that switched the Q8 activation policy
    // off: the decoded weight, scale times code, is exact in float; 4096 x 4096 by 2048 rows 20.9 ms
    // on the lane-strided kernel)
    if ((qtype == QT_F32 || qtype == QT_F16 || qtype == QT_BF16 || (qtype == QT_Q8_0 && !input_q8)) &&
        input_rows >= 8ull && !(((uintptr_t)encoded | (uintptr_t)input) & 15u) && !(input_stride & 3ull) &&
        row_width % (input_rows < 256ull ? 256ull : 64ull) == 0ull)
        return qtype == QT_F32 ? launch_scalar_rows<QT_F32>(a, s)
             : qtype == QT_F16 ? launch_scalar_rows<QT_F16>(a, s)
             : qtype == QT_BF16 ? launch_scalar_rows<QT_BF16>(a, s) : launch_scalar_rows<QT_Q8_0>(a, s);
    // (fewer than eight input rows, or a row width the matrix-core kernels do not take: 16-bit
    // rows have no other fast kernel and stay here at any number of input rows, four a workgroup)
    if (((qtype == QT_F32 && input_rows < 8ull) ||
         ((qtype == QT_F16 || qtype == QT_BF16) && (input_rows + 3ull) / 4ull <= 65535ull)) &&
        row_count <= 0x7fffffffull && !(((uintptr_t)encoded | (uintptr_t)input) & 15u) && !(input_stride & 3ull) &&
        !(row_bytes & 15ull)) {      // (whole 16-byte pieces a row: a multiple of 4 or 8 columns)
        if (qtype == QT_F32) return launch_scalar_few<QT_F32>(a, s);
        return qtype == QT_F16 ? launch_scalar_few<QT_F16>(a, s) : launch_scalar_few<QT_BF16>(a, s);
    }
    if (scalar) {
        const unsigned long long grid_x = (row_count + 3ull) / 4ull;
        if (grid_x > 0x7fffffffull) return ST_BOUNDS;
        if (input_rows == 1ull) {
            matvec_scalar_kernel<1><<<dim3((unsigned)grid_x, 1), 256, 0, s>>>(a, qtype);
        } else {
            const unsigned long long grid_y = (input_rows + 3ull) / 4ull;
            if (grid_y > 65535ull) return ST_BOUNDS;
            matvec_scalar_kernel<4><<<dim3((unsigned)grid_x, (unsigned)grid_y), 256, 0, s>>>(a, qtype);
        }
        return check_launch("matvec_scalar");
    }
    switch (qtype) {
    case QT_IQ2_XXS: return launch_block_q<QT_IQ2_XXS>(a, input_q8, s, publisher);
    case QT_Q8_0: return launch_block_q<QT_Q8_0>(a, input_q8, s, publisher);
    case QT_Q4_K: return launch_block_q<QT_Q4_K>(a, input_q8, s, publisher);
    case QT_Q2_K: return launch_block_q<QT_Q2_K>(a, input_q8, s, publisher);
    default: return ST_UNSUPPORTED;
    }
}

extern "C" int yvex_hip_matvec(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                               uint64_t row_width, uint64_t row_bytes, const void *input,
                               int input_q8, uint64_t input_rows, uint64_t input_stride,
                               const float *additive, float *out, uint64_t out_stride,
                               int output_bf16, int *status, yvex_hip_stream stream)
{
    return launch_matvec(encoded, qtype, row_count, row_width, row_bytes, input, input_q8, input_rows, input_stride,
                         additive, out, out_stride, output_bf16, status, stream, nullptr);
}

int yvex_hip_matvec_publishing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count, uint64_t row_width,
                               uint64_t row_bytes, const void *input, int input_q8, uint64_t input_rows,
                               uint64_t input_stride, const float *additive, float *out, uint64_t out_stride,
                               int output_bf16, int *status, const yvex_hip_publication *publication, int *published,
                               yvex_hip_stream stream)
{
    Publisher publisher = publisher_of(*publication);
    const int rc = launch_matvec(encoded, qtype, row_count, row_width, row_bytes, input, input_q8, input_rows, input_stride,
                                 additive, out, out_stride, output_bf16, status, stream, &publisher);
    *published = publisher.taken;
    return rc;
}

// Whether F32 input rows are multiplied by the launch that quantizes them. Every workgroup quantizes all of them, a
// block a wave at a time, so up to two rows, and as many blocks as the workgroup has waves or twice that while the rest of
// the launch is short. Two launches and one, us: 4096 x 4096 by 1 and 2 rows 9.8 and 7.2, 12.2 and 9.0 (by 3 12.4 and
// 11.9, by 4 12.7 and 12.8); 7168 x 7168 18.2 and 15.7, 22.5 and 18.5; 50 000 x 4096 57.9 and 45.7, 87 and 47;
// 129 280 x 7168 184.7 and 184.1, 206 and 196; 64 x 256 4.5 and 3.1; but 1024 x 7168 by 2 10.3 and 11.6, 2048 x 8192 by 1
// 9.7 and 10.2, 256 x 16384 11.3 and 13.8.
extern "C" int yvex_hip_matvec_quantizing_supported(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                                                    uint64_t row_width, uint64_t row_bytes, uint64_t input_rows)
{
    if (qtype != QT_Q8_0 || !input_rows || input_rows > 2u || !row_count || !row_width || row_width > 14336u ||
        row_width % 256u || row_width / 32u * 34u != row_bytes || ((uintptr_t)encoded & 1u))
        return 0;
    const uint64_t tasks = input_rows * (row_width / 256u);
    return (tasks <= 32u && row_width <= 7168u) || (tasks <= 56u && row_count >= 4096u);
}

template <int T>
static int launch_quantizing(MatvecArgs &a, hipStream_t s, Publisher *publisher)
{
    const unsigned long long groups = (a.row_count + kHeldWaves - 1ull) / kHeldWaves, most = (unsigned long long)compute_units();
    const unsigned grid = (unsigned)(groups < most ? groups : most);
    const unsigned lds = (unsigned)held_bytes(T, a.row_width / 256ull);
    // The launch ends the operation while a wave has up to eight rows: each row's store goes to memory ahead of the next
    // row's bytes and is waited for with them. us a call, published by the launch and behind it: 32 768 x 4096 by 1 / 2
    // rows 30.9 / 33.4 and 30.9 / 33.4, x 1024 17.5 / 21.8 and 18.2 / 22.7; 40 960 x 7168 61.7 / 66.9 and 61.0 / 65.8;
    // 129 280 x 4096 112.2 / 117.7 and 108.3 / 111.3, x 7168 188.4 / 204.2 and 184.4 / 195.8.
    a.publication = take_publication(publisher, groups, 8ull * most);
    if (a.row_width <= 2048ull) matvec_q8_0_quantizing_kernel<T, 1><<<grid, kHeldThreads, lds, s>>>(a);
    else if (a.row_width <= 4096ull) matvec_q8_0_quantizing_kernel<T, 2><<<grid, kHeldThreads, lds, s>>>(a);
    else matvec_q8_0_quantizing_kernel<T, 4><<<grid, kHeldThreads, lds, s>>>(a);
    return check_launch("matvec_quantizing");
}

static int launch_matvec_quantizing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                                          uint64_t row_width, uint64_t row_bytes, const float *input,
                                          uint64_t input_rows, uint64_t input_stride, const float *additive, float *out,
                                          uint64_t out_stride, int output_bf16, int *status, yvex_hip_stream stream, Publisher *publisher)
{
    if (!encoded || !input || !out || !status || out_stride < row_count || input_stride < row_width ||
        (((uintptr_t)input | (uintptr_t)out) & 3u))
        return ST_INVALID_ARG;
    if (!yvex_hip_matvec_quantizing_supported(encoded, qtype, row_count, row_width, row_bytes, input_rows))
        return ST_UNSUPPORTED;
    MatvecArgs a{encoded, row_count, row_width, row_bytes, input, input_rows, input_stride, additive, out, out_stride,
                 output_bf16, status, nullptr, nullptr, 0};
    return input_rows == 1u ? launch_quantizing<1>(a, as_stream(stream), publisher) : launch_quantizing<2>(a, as_stream(stream), publisher);
}

extern "C" int yvex_hip_matvec_quantizing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                                          uint64_t row_width, uint64_t row_bytes, const float *input,
                                          uint64_t input_rows, uint64_t input_stride, const float *additive, float *out,
                                          uint64_t out_stride, int output_bf16, int *status, yvex_hip_stream stream)
{
    return launch_matvec_quantizing(encoded, qtype, row_count, row_width, row_bytes, input, input_rows, input_stride, additive,
                                    out, out_stride, output_bf16, status, stream, nullptr);
}

int yvex_hip_matvec_quantizing_publishing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                                          uint64_t row_width, uint64_t row_bytes, const float *input,
                                          uint64_t input_rows, uint64_t input_stride, const float *additive, float *out,
                                          uint64_t out_stride, int output_bf16, int *status,
                                          const yvex_hip_publication *publication, int *published, yvex_hip_stream stream)
{
    Publisher publisher = publisher_of(*publication);
    const int rc = launch_matvec_quantizing(encoded, qtype, row_count, row_width, row_bytes, input, input_rows, input_stride,
                                            additive, out, out_stride, output_bf16, status, stream, &publisher);
    *published = publisher.taken;
    return rc;
}

// Two Q8_0 matrices of one shape against the same Q8_K input rows in one launch (a shared expert's gate
// and up projections): each offers too few workgroups for the device on its own (2048 x 4096 against
// 96 rows: 192 of them, 16 us a launch).
extern "C" int yvex_hip_matvec_q8_0_pair(const uint8_t *first, const uint8_t *second, uint64_t row_count,
                                         uint64_t row_width, uint64_t row_bytes, const void *input_q8k,
                                         uint64_t input_rows, float *out_first, float *out_second,
                                         int *status, yvex_hip_stream stream)
{
    if (!first || !second || !input_q8k || !out_first || !out_second || !status || !row_count || !row_width ||
        !input_rows || (((uintptr_t)input_q8k | (uintptr_t)out_first | (uintptr_t)out_second) & 3u))
        return ST_INVALID_ARG;
    if (row_width % 256u || row_width / 32u * 34u != row_bytes || row_width > 0xffffffffull * 32ull) return ST_BOUNDS;
    // (the kernels address both matrices the same way: the weaker alignment decides)
    const uint8_t *alignment = (const uint8_t *)((uintptr_t)first | (uintptr_t)second);
    if (q8_0_takes_matrix_cores(alignment, row_count, row_bytes, input_rows))
        return launch_q8_0_rows_dense(first, row_count, row_width, row_bytes, input_q8k, input_rows, nullptr,
                                      out_first, row_count, false, status, as_stream(stream), second, out_second);
    MatvecArgs a{first, row_count, row_width, row_bytes, input_q8k, input_rows, row_width, nullptr, out_first,
                 row_count, 0, status, nullptr, nullptr, 0, second, out_second};
    return ((uintptr_t)alignment & 1u) == 0u ? launch_block_even<QT_Q8_0, true, true>(a, as_stream(stream))
                                             : launch_block_even<QT_Q8_0, true, false>(a, as_stream(stream));
}

extern "C" int yvex_hip_block_dots_i32(const uint8_t *encoded, unsigned int qtype,
                                       uint64_t row_count, uint64_t row_width,
                                       uint64_t row_bytes, const uint8_t *input_q8,
                                       uint64_t input_rows, int32_t *sums, int *status,
                                       yvex_hip_stream stream)
{
    unsigned block, bytes;
    if (!encoded || !input_q8 || !sums || !status || !row_count || !row_width || !input_rows)
        return ST_INVALID_ARG;
    if (!qtype_geometry(qtype, block, bytes)) return ST_UNSUPPORTED;
    if (row_width % 256u || row_width / block * bytes != row_bytes) return ST_BOUNDS;
    if (((uintptr_t)input_q8 & 3u) || input_rows > 65535ull) return ST_INVALID_ARG;
    const unsigned long long grid_x = (row_count + 3ull) / 4ull;
    if (grid_x > 0x7fffffffull) return ST_BOUNDS;
    dim3 grid((unsigned)grid_x, (unsigned)input_rows);
    hipStream_t s = as_stream(stream);
    switch (qtype) {
    case QT_IQ2_XXS:
        block_dots_kernel<QT_IQ2_XXS><<<grid, 256, 0, s>>>(encoded, row_count, row_width,
                                                           row_bytes, input_q8, input_rows, sums);
        break;
    case QT_Q8_0:
        block_dots_kernel<QT_Q8_0><<<grid, 256, 0, s>>>(encoded, row_count, row_width, row_bytes,
                                                        input_q8, input_rows, sums);
        break;
    case QT_Q4_K:
        block_dots_kernel<QT_Q4_K><<<grid, 256, 0, s>>>(encoded, row_count, row_width, row_bytes,
                                                        input_q8, input_rows, sums);
        break;
    case QT_Q2_K:
        block_dots_kernel<QT_Q2_K><<<grid, 256, 0, s>>>(encoded, row_count, row_width, row_bytes,
                                                        input_q8, input_rows, sums);
        break;
    default: return ST_UNSUPPORTED;
    }
    return check_launch("block_dots");
}

extern "C" int yvex_hip_gather(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                               uint64_t row_width, uint64_t row_bytes, const uint32_t *row_ids,
                               uint64_t selected, float *out, int *status,
                               yvex_hip_stream stream)
{
    unsigned block, bytes;
    if (!encoded || !out || !status || !row_count || !row_width || !selected) return ST_INVALID_ARG;
    if (!qtype_geometry(qtype, block, bytes)) return ST_UNSUPPORTED;
    if (row_width % block || row_width / block * bytes != row_bytes) return ST_BOUNDS;
    if (selected > UINT64_MAX / row_width) return ST_BOUNDS;
    const unsigned long long grid = (selected * row_width + 255ull) / 256ull;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    gather_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        encoded, qtype, row_count, row_width, row_bytes, row_ids, selected, out, status);
    return check_launch("gather");
}

extern "C" int yvex_hip_row_dot(const uint8_t *encoded, unsigned int qtype, const float *vector,
                                uint64_t elements, float *out, yvex_hip_stream stream)
{
    unsigned block, bytes;
    if (!encoded || !vector || !out || !elements) return ST_INVALID_ARG;
    if (!qtype_geometry(qtype, block, bytes)) return ST_UNSUPPORTED;
    if (elements % block) return ST_BOUNDS;
    row_dot_serial_kernel<<<1, 1, 0, as_stream(stream)>>>(encoded, vector, elements, qtype, out);
    return check_launch("row_dot");
}

// Splits of the 16 x 16 tiles: 512 columns a split (128 a wave) where that gives 2 to 64 splits; a wider row takes
// the most splits up to 64 that leave every wave a multiple of 16 columns.
static unsigned f32_rows_column_splits(uint64_t row_width)
{
    if (row_width % 512u == 0u && row_width / 512u >= 2u && row_width / 512u <= 64u)
        return (unsigned)(row_width / 512u);
    if (row_width < 64u * 512u) return 0u;
    for (unsigned splits = 64u; splits >= 2u; --splits)
        if (row_width % (64ull * splits) == 0u) return splits;
    return 0u;
}

// The 16 x 16 tiles keep up to 16 input rows, and a decode batch whose workgroups, sixteen splits at most, have a compute
// unit each: 256 x 7168 by 10 rows 11.5 us (on the 32-row tiles 12.5), by 23 13.5 (12.9); 256 x 4096 by 32 10.4 (10.8), by
// 96 14.3 (12.3); 24 x 16384 by 32, 32 splits, 15.2 (14.4).
static bool f32_rows_wide(uint64_t row_count, uint64_t row_width, uint64_t input_rows)
{
    if (input_rows <= 16u || row_width % 128u) return false;
    const uint64_t splits = f32_rows_column_splits(row_width);
    return input_rows >= 256u || splits > 16u ||
           (row_count + 15u) / 16u * ((input_rows + 15u) / 16u) * splits > (uint64_t)compute_units();
}

// A batch of fewer tiles is always split (a router's second launch then routes its rows as well), a larger one where that
// is faster.
static ScalarTiles f32_rows_tiles(uint64_t row_count, uint64_t row_width, uint64_t input_rows)
{
    const bool few = input_rows < 256u || (row_count + 15u) / 16u * ((input_rows + 15u) / 16u) < 1024u;
    return scalar_tiles(row_count, row_width, input_rows, few ? 2u : 1u, 16u);
}

// Splits of an F32 projection over a row batch; 0 where it is one launch: a row of too few columns at decode width.
unsigned yvex::f32_rows_splits(uint64_t row_count, uint64_t row_width, uint64_t input_rows)
{
    if (input_rows < 8u || row_width % 128u) return 0u;
    const unsigned columns = f32_rows_column_splits(row_width);
    if (!f32_rows_wide(row_count, row_width, input_rows)) return columns;
    const unsigned splits = f32_rows_tiles(row_count, row_width, input_rows).splits;
    return splits > 1u ? splits : 0u;
}

extern "C" uint64_t yvex_hip_matvec_f32_scratch_bytes(uint64_t row_count, uint64_t row_width,
                                                      uint64_t input_rows)
{
    const unsigned splits = f32_rows_splits(row_count, row_width, input_rows);
    return splits ? (uint64_t)splits * input_rows * row_count * sizeof(double) : 0u;
}

// Whether the projection runs as partial tiles plus a join (two launches) or as one launch.
static bool f32_rows_split_applies(const float *weights, uint64_t row_count, uint64_t row_width,
                                   const float *input, uint64_t input_rows, uint64_t input_stride,
                                   const void *scratch, uint64_t scratch_bytes)
{
    const unsigned splits = f32_rows_splits(row_count, row_width, input_rows);
    const uint64_t need = yvex_hip_matvec_f32_scratch_bytes(row_count, row_width, input_rows);
    return splits && scratch && scratch_bytes >= need && !((uintptr_t)scratch & 7u) &&
           !(((uintptr_t)weights | (uintptr_t)input) & 15u) && !(input_stride & 3ull) && weights && input &&
           row_count && input_stride >= row_width;
}

extern "C" unsigned int yvex_hip_matvec_f32_rows_launches(const float *weights, uint64_t row_count,
                                                          uint64_t row_width, const float *input,
                                                          uint64_t input_rows, uint64_t input_stride,
                                                          const void *scratch, uint64_t scratch_bytes)
{
    return f32_rows_split_applies(weights, row_count, row_width, input, input_rows, input_stride, scratch,
                                  scratch_bytes) ? 2u : 1u;
}

static int launch_f32_rows_parts(const MatvecArgs &a, yvex_hip_stream stream);
static int launch_f32_rows_split(const MatvecArgs &a, yvex_hip_stream stream);

extern "C" int yvex_hip_matvec_f32_rows(const float *weights, uint64_t row_count, uint64_t row_width,
                                        const float *input, uint64_t input_rows, uint64_t input_stride,
                                        const float *additive, float *out, uint64_t out_stride,
                                        int output_bf16, void *scratch, uint64_t scratch_bytes,
                                        int *status, yvex_hip_stream stream)
{
    if (!f32_rows_split_applies(weights, row_count, row_width, input, input_rows, input_stride, scratch,
                                scratch_bytes) || !out || !status || out_stride < row_count)
        return yvex_hip_matvec((const uint8_t *)weights, QT_F32, row_count, row_width, row_width * 4u, input, 0,
                               input_rows, input_stride, additive, out, out_stride, output_bf16, status,
                               stream);
    MatvecArgs a{(const unsigned char *)weights, row_count, row_width, row_width * 4u, input, input_rows,
                 input_stride, additive, out, out_stride, output_bf16, status, (double *)scratch, nullptr, 0};
    return launch_f32_rows_split(a, stream);
}

// The split projection with the router's score of every output published beside it
// (`scores`, dense [input row][weight row]): the scores are computed by the join's many
// workgroups instead of the routing launch's one. Only where the split applies (two launches,
// as yvex_hip_matvec_f32_rows_launches says); anything else is refused.
extern "C" int yvex_hip_matvec_f32_rows_scored(const float *weights, uint64_t row_count, uint64_t row_width,
                                               const float *input, uint64_t input_rows,
                                               uint64_t input_stride, float *out, uint64_t out_stride,
                                               float *scores, int scoring, void *scratch,
                                               uint64_t scratch_bytes, int *status, yvex_hip_stream stream)
{
    if (!out || !scores || !status || out_stride < row_count || (scoring != 0 && scoring != 1) ||
        ((uintptr_t)out & 3u) || ((uintptr_t)scores & 3u))
        return ST_INVALID_ARG;
    if (!f32_rows_split_applies(weights, row_count, row_width, input, input_rows, input_stride, scratch,
                                scratch_bytes))
        return ST_UNSUPPORTED;
    MatvecArgs a{(const unsigned char *)weights, row_count, row_width, row_width * 4u, input, input_rows,
                 input_stride, nullptr, out, out_stride, 0, status, (double *)scratch, scores, scoring};
    return launch_f32_rows_split(a, stream);
}

// The router of a row batch: the split projection whose second launch routes as well. Selections,
// route weights and logits are those of yvex_hip_matvec_f32_rows followed by yvex_hip_moe_route_rows.
extern "C" int yvex_hip_matvec_f32_rows_routed(const float *weights, uint64_t row_count, uint64_t row_width,
                                               const float *input, uint64_t input_rows, uint64_t input_stride,
                                               float *logits, const float *bias, uint64_t topk, int scoring,
                                               int normalize, double scaling, uint64_t *selected,
                                               float *route_weights, void *scratch, uint64_t scratch_bytes,
                                               int *status, yvex_hip_stream stream)
{
    if (!logits || !selected || !route_weights || !status || (scoring != 0 && scoring != 1) || !topk ||
        topk > 16u || topk > row_count || ((uintptr_t)logits & 3u))
        return ST_INVALID_ARG;
    if (row_count > 256u ||
        !f32_rows_split_applies(weights, row_count, row_width, input, input_rows, input_stride, scratch,
                                scratch_bytes))
        return ST_UNSUPPORTED;
    MatvecArgs a{(const unsigned char *)weights, row_count, row_width, row_width * 4u, input, input_rows,
                 input_stride, nullptr, logits, row_count, 0, status, (double *)scratch, nullptr, scoring};
    int rc = launch_f32_rows_parts(a, stream);
    if (rc) return rc;
    matvec_f32_join_route_kernel<<<(unsigned)input_rows, 256, 0, as_stream(stream)>>>(
        a, f32_rows_splits(row_count, row_width, input_rows), bias, (unsigned)topk, normalize, scaling,
        (unsigned long long *)selected, route_weights);
    return check_launch("matvec_f32_rows.join_route");
}

static int launch_f32_rows_parts(const MatvecArgs &a, yvex_hip_stream stream)
{
    if (f32_rows_wide(a.row_count, a.row_width, a.input_rows))
        return launch_scalar_tiles<QT_F32>(a, f32_rows_tiles(a.row_count, a.row_width, a.input_rows), as_stream(stream));
    const uint64_t grid_x = (a.row_count + 15u) / 16u, grid_y = (a.input_rows + 15u) / 16u;
    if (grid_x > 0x7fffffffull || grid_y > 65535ull) return ST_BOUNDS;
    matvec_f32_tile16_kernel<4><<<dim3((unsigned)grid_x, (unsigned)grid_y,
                                       f32_rows_splits(a.row_count, a.row_width, a.input_rows)), 256, 0,
                                  as_stream(stream)>>>(a);
    return check_launch("matvec_f32_rows.parts");
}

int yvex::launch_f32_rows_parts(const float *weights, uint64_t row_count, uint64_t row_width, const float *input,
                                uint64_t input_rows, uint64_t input_stride, double *parts, int *status, hipStream_t stream)
{
    return ::launch_f32_rows_parts(MatvecArgs{(const unsigned char *)weights, row_count, row_width, row_width * 4u, input,
                                              input_rows, input_stride, nullptr, nullptr, row_count, 0, status, parts,
                                              nullptr, 0}, reinterpret_cast<yvex_hip_stream>(stream));
}

static int launch_f32_rows_split(const MatvecArgs &a, yvex_hip_stream stream)
{
    const uint64_t row_count = a.row_count, input_rows = a.input_rows;
    const unsigned splits = f32_rows_splits(row_count, a.row_width, input_rows);
    const uint64_t outputs = input_rows * row_count;
    if ((outputs + 255u) / 256u > 0x7fffffffull) return ST_BOUNDS;
    int rc = launch_f32_rows_parts(a, stream);
    if (rc) return rc;
    matvec_f32_join_kernel<<<(unsigned)((outputs + 255u) / 256u), 256, 0, as_stream(stream)>>>(a, splits);
    return check_launch("matvec_f32_rows.join");
}
