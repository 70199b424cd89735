// Residual-stream envelope around the expert math, for gfx950.
//
// A layer's input row holds `streams` residual streams of `width` values. Ingress collapses them
// into one row with sigmoid gates, builds the stream-mixing matrix (row softmax followed by
// alternating row and column normalisations), applies the weighted RMS norm and publishes bf16
// values; egress spreads the layer's output back over the streams. Behaviour restated from
// src/graph/numeric.c:630-877 (the arithmetic and its order), src/graph/moe.c:446-495 (how the
// MoE composes it) and src/backend/cuda/kernels.cu:867-910,1243-1428 (the device twins, which
// round the incoming residual to bf16 first).
//
// Both kernels are bound by reading the rows once; the gates and the mixing matrix are a few
// dozen double-precision operations per row.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace yvex {

constexpr unsigned kEnvelopeThreads = 256;
constexpr unsigned kEnvelopeMaxStreams = 7;       // (streams + 2) * streams <= 64 mixing rows
constexpr unsigned kEnvelopeMaxWidth = 16384;     // the reference's bound (src/graph/moe.c:453-455)
constexpr unsigned kEnvelopeLdsBytes = 147456;    // a row of floats and what else fits

__device__ __forceinline__ bool finite_f64(double v)
{
    return (__double_as_longlong(v) & 0x7ff0000000000000ll) != 0x7ff0000000000000ll;
}

// Sum over the workgroup, the same value in every thread: a butterfly inside each wavefront,
// then the wavefront totals in order. The order is fixed, so a row's result does not depend on
// where it runs.
template <unsigned WAVES>
__device__ __forceinline__ double workgroup_sum(double v, double *slots)
{
    v = wave_sum_f64(v);
    if ((threadIdx.x & 63u) == 0u) slots[threadIdx.x >> 6] = v;
    __syncthreads();
    double total = slots[0];
#pragma unroll
    for (unsigned w = 1; w < WAVES; ++w) total += slots[w];
    __syncthreads();
    return total;
}

__device__ __forceinline__ double sigmoid_f64(double value)
{
    const double e = exp(-fabs(value));
    return (value >= 0.0 ? 1.0 : e) / (1.0 + e);
}

__device__ __forceinline__ float4 bf16_round4(float4 v)
{
    return make_float4(bf16_round(v.x), bf16_round(v.y), bf16_round(v.z), bf16_round(v.w));
}

// Four values that bf16 holds, as it holds them, and back.
__device__ __forceinline__ uint2 bf16_pack4(float4 v)
{
    return make_uint2(__builtin_amdgcn_perm(__float_as_uint(v.y), __float_as_uint(v.x), 0x07060302u),
                      __builtin_amdgcn_perm(__float_as_uint(v.w), __float_as_uint(v.z), 0x07060302u));
}

__device__ __forceinline__ float4 bf16_unpack4(uint2 v)
{
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                       __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
}

// A coefficient vector (scale, base, norm) as the layer stores it, F32 or BF16 values, decoded
// where they are used (the reference decodes them into F32 buffers with launches of their own,
// src/backend/cuda/moe.c:1226-1240; the decoded value is the same float).
__device__ __forceinline__ float coefficient(const void *values, unsigned qtype, unsigned index)
{
    if (qtype == QT_F32) return static_cast<const float *>(values)[index];
    return __uint_as_float((unsigned)static_cast<const unsigned short *>(values)[index] << 16);
}

// Four consecutive coefficients from a 16-byte (F32) or 8-byte (BF16) aligned address.
__device__ __forceinline__ float4 coefficient4(const void *values, unsigned qtype, unsigned quad)
{
    if (qtype == QT_F32) return static_cast<const float4 *>(values)[quad];
    return bf16_unpack4(static_cast<const uint2 *>(values)[quad]);
}

// Alternating row and column normalisations of a 4 x 4 matrix, one element a lane (4 row + column,
// repeated in each group of sixteen lanes). The totals are two additions each way inside the row of
// sixteen lanes, on the vector ALU; sums of four floats of a matrix whose elements lie within a
// factor of 2^29 are exact in double, so the order of the additions does not show. Gathering the
// four elements with lane permutes through LDS, one waited for after another, took 0.4 us a turn
// (twenty of them: 8 of the 18 us of a one-row launch); 0.15 us now.
__device__ __forceinline__ float sinkhorn4(float m, unsigned iterations, double epsilon, bool &bad)
{
    for (unsigned it = 0; it < iterations; ++it) {
        if (it != 0u) {
            double across = (double)m;
            across += dpp_f64<0xb1>(across);       // quad_perm [1, 0, 3, 2]
            across += dpp_f64<0x4e>(across);       // quad_perm [2, 3, 0, 1]
            bad |= !finite_f64(across);
            m = (float)((double)m / (across + epsilon));
        }
        double down = (double)m;
        down += dpp_f64<0x128>(down);              // row_ror 8, row_ror 4
        down += dpp_f64<0x124>(down);
        bad |= !finite_f64(down);
        m = (float)((double)m / (down + epsilon));
    }
    return m;
}

// One workgroup per row. The row is passed over twice (mean square, then the gated sum of the streams); four 16-byte
// loads per thread are in flight, because a row is a short stream and a loop that waits for each load in turn spends its
// time on latency; long rows take 1024 threads for the same reason. Rows whose width is not a multiple of four take the
// scalar loops.
// SPLIT, where a batch leaves every row two compute units: a second workgroup forms the mean square as well and then the
// mixing matrix, whose chain of divisions so runs beside the second pass and not ahead of the sum that ends it, and the
// first pass leaves the rounded values in LDS for the second (`held`: unless the row is too long). Which thread adds which
// squares is the same either way, so a row's results do not depend on its batch. Four streams of 4096 values, where a
// one-row launch is 2.6 us of getting there and back and then waits of one workgroup for itself, by 1 / 96 / 128 rows
// 9.6 / 11.0 / 11.4 -> 7.7 / 9.8 / 10.4 us, of 7168 values 13.7 / 15.4 / 16.0 -> 10.7 / 13.7 / 15.2. Where two workgroups
// have to share a compute unit the second pass over the row costs what it gave: 160 rows 11.8 and 14.7, 16.6 and 24.4.
// With `parts` the mixing projection's sums arrive as its `splits` partial sums (doubles, [split][row][mixing row]), requested ahead
// of the row and put into LDS behind it; whoever uses a sum adds its parts in their order, as matvec_f32_join_kernel
// does, whose launch is not needed then: 6.5 us a layer of 96 rows, 4.7 of 333.
constexpr unsigned kPartsAThread = 4u;    // 63 mixing rows in 64 splits, or in 16 of an expanded row under 8192 values

template <unsigned THREADS, bool SPLIT>
__global__ __launch_bounds__(THREADS) void mhc_ingress_kernel(
    const float *__restrict__ rows, const float *__restrict__ mixes, const void *__restrict__ scale_values,
    const void *__restrict__ base_values, const void *__restrict__ norm, unsigned scale_qtype,
    unsigned base_qtype, unsigned norm_qtype, unsigned streams, unsigned width,
    unsigned iterations, double rms_epsilon, double mhc_epsilon, double post_multiplier,
    float *__restrict__ normalized, float *__restrict__ post, float *__restrict__ combination,
    int quads, int held, const double *__restrict__ parts, unsigned splits, unsigned parts_at, int *status)
{
    __shared__ float base[64], scale[3];      // (streams + 2) * streams <= 63 mixing rows
    extern __shared__ __align__(16) float collapsed[];   // width values; behind them, where held, the row as bf16
    __shared__ double slots[THREADS / 64u];
    __shared__ double gate[8];
    constexpr unsigned kBatch = 4, kAhead = SPLIT ? 8 : 4;   // (two workgroups share a compute unit on fewer registers)
    constexpr unsigned kWorkers = THREADS - 64u;             // the second pass leaves the first wavefront out
    const unsigned tid = threadIdx.x;
    const unsigned long long row = SPLIT ? blockIdx.x >> 1 : blockIdx.x;
    const bool mixes_only = SPLIT && (blockIdx.x & 1u) != 0u, mixes_here = !SPLIT || mixes_only;
    const unsigned expanded = streams * width, mixing_rows = (streams + 2u) * streams;
    const float *in = rows + row * expanded;
    const float *mix = parts ? nullptr : mixes + row * mixing_rows;
    bool bad = false;    // quads: width is a multiple of four and every row starts 16-byte aligned
    double *const parts_held = reinterpret_cast<double *>(collapsed + parts_at);
    double part[kPartsAThread];
    if (parts) {
        const unsigned long long row_count = SPLIT ? gridDim.x >> 1 : gridDim.x;
#pragma unroll
        for (unsigned k = 0; k < kPartsAThread; ++k) {
            const unsigned at = tid + k * THREADS, z = at / mixing_rows;
            part[k] = z < splits ? parts[(z * row_count + row) * mixing_rows + (at - z * mixing_rows)] : 0.0;
        }
    }
    auto mix_of = [&](unsigned index) {
        if (!parts) return mix[index];
        double sum = parts_held[index];
        for (unsigned z = 1; z < splits; ++z) sum += parts_held[z * mixing_rows + index];
        bad |= !finite_f32((float)sum);
        return (float)sum;
    };

    // mean square of the bf16-rounded residual (a value that is not finite makes the sum not finite)
    double squares = 0.0;
    uint2 *const row_held = reinterpret_cast<uint2 *>(collapsed + width);
    const bool hold = SPLIT && held != 0 && !mixes_only;
    if (quads) {
        const float4 *in4 = reinterpret_cast<const float4 *>(in);
        const unsigned count = expanded >> 2;
        for (unsigned first = tid; first < count; first += THREADS * kAhead) {
            float4 v[kAhead];
#pragma unroll
            for (unsigned u = 0; u < kAhead; ++u) {
                const unsigned at = first + u * THREADS;
                v[u] = at < count ? in4[at] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
#pragma unroll
            for (unsigned u = 0; u < kAhead; ++u) {
                if (SPLIT && first - tid + u * THREADS >= count) break;
                const float4 r = bf16_round4(v[u]);
                squares += (double)r.x * (double)r.x;
                squares += (double)r.y * (double)r.y;
                squares += (double)r.z * (double)r.z;
                squares += (double)r.w * (double)r.w;
                if (hold && first + u * THREADS < count) row_held[first + u * THREADS] = bf16_pack4(r);
            }
        }
    } else {
        for (unsigned lane = tid; lane < expanded; lane += THREADS) {
            const float v = bf16_round(in[lane]);
            squares += (double)v * (double)v;
        }
    }
    bad |= !finite_f64(squares);
    if (tid < mixing_rows) {
        base[tid] = coefficient(base_values, base_qtype, tid);
        bad |= !finite_f32(base[tid]) || (!parts && !finite_f32(mix[tid]));
    }
    if (parts) {
#pragma unroll
        for (unsigned k = 0; k < kPartsAThread; ++k)
            if (tid + k * THREADS < splits * mixing_rows) parts_held[tid + k * THREADS] = part[k];
    }
    if (tid < 3u) {
        scale[tid] = coefficient(scale_values, scale_qtype, tid);
        bad |= !finite_f32(scale[tid]);
    }
    // (the barriers inside the sum publish base, scale and the partial sums to the threads that read them below)
    const double inverse = 1.0 / sqrt(workgroup_sum<THREADS / 64u>(squares, slots) / (double)expanded + rms_epsilon);
    bad |= !finite_f64(inverse);

    // (the two sigmoids of a stream in different wavefronts)
    if (!mixes_only && tid < streams) {
        const double pre = sigmoid_f64((double)mix_of(tid) * inverse * (double)scale[0] + (double)base[tid]);
        gate[tid] = pre + mhc_epsilon;
    } else if (!mixes_only && tid >= 64u && tid < 64u + streams) {
        const unsigned s = tid - 64u;
        post[row * streams + s] = (float)(post_multiplier * sigmoid_f64(
            (double)mix_of(streams + s) * inverse * (double)scale[1] + (double)base[streams + s]));
    }
    __syncthreads();

    // The mixing matrix lives in the first wavefront, one element per lane, and never touches
    // memory: a row (or column) total is gathered with lane reads in index order, so every lane
    // of the row forms the same double-precision sum the serial code forms. It is a chain of
    // dependent divisions several microseconds long, so the other wavefronts run the second pass
    // over the row meanwhile.
    const unsigned cells = streams * streams;
    if (mixes_here && tid < 64u) {
        // (four streams: every group of sixteen lanes holds the matrix)
        const unsigned held = streams == 4u ? tid & 15u : tid;
        const bool cell = held < cells;
        const unsigned r = cell ? held / streams : 0u, c = cell ? held % streams : 0u;
        const unsigned index = 2u * streams + (cell ? held : 0u);
        float m = (float)((double)mix_of(index) * inverse * (double)scale[2] + (double)base[index]);
        double maximum = -__builtin_inf(), total = 0.0;
        for (unsigned k = 0; k < streams; ++k)
            maximum = fmax(maximum, (double)__shfl(m, (int)(r * streams + k), kWave));
        const double mine = exp((double)m - maximum);          // an exponential a lane; a row's are added in their order
        for (unsigned k = 0; k < streams; ++k) total += __shfl(mine, (int)(r * streams + k), kWave);
        bad |= cell && (!finite_f64(total) || !(total > 0.0));
        m = (float)((double)(float)mine / total + mhc_epsilon);
        if (streams == 4u) m = sinkhorn4(m, iterations, mhc_epsilon, bad);
        else for (unsigned it = 0; it < iterations; ++it) {
            if (it != 0u) {
                double across = 0.0;
                for (unsigned k = 0; k < streams; ++k) across += (double)__shfl(m, (int)(r * streams + k), kWave);
                bad |= cell && !finite_f64(across);
                m = (float)((double)m / (across + mhc_epsilon));
            }
            double down = 0.0;
            for (unsigned k = 0; k < streams; ++k) down += (double)__shfl(m, (int)(k * streams + c), kWave);
            bad |= cell && !finite_f64(down);
            m = (float)((double)m / (down + mhc_epsilon));
        }
        if (tid < cells) combination[row * cells + tid] = m;
    }
    if (mixes_only) {
        if (bad) raise_status(status, 1);
        return;
    }

    // collapsed row: float accumulation over the streams in order, then bf16
    double collapsed_squares = 0.0;
    if (tid < 64u) {
        // busy with the mixing matrix above
    } else if (quads && streams <= kBatch) {
        const float4 *in4 = reinterpret_cast<const float4 *>(in);
        const unsigned count = width >> 2;
        for (unsigned at = tid - 64u; at < count; at += kWorkers) {
            float4 v[kBatch];
            if (hold) {
#pragma unroll
                for (unsigned s = 0; s < kBatch; ++s) v[s] = bf16_unpack4(row_held[s < streams ? s * count + at : at]);
            } else {
#pragma unroll
                for (unsigned s = 0; s < kBatch; ++s)
                    v[s] = s < streams ? in4[s * count + at] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
                for (unsigned s = 0; s < kBatch; ++s) v[s] = bf16_round4(v[s]);
            }
            float4 total = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (unsigned s = 0; s < kBatch; ++s) {
                if (s < streams) {
                    total.x += (float)(gate[s] * (double)v[s].x);
                    total.y += (float)(gate[s] * (double)v[s].y);
                    total.z += (float)(gate[s] * (double)v[s].z);
                    total.w += (float)(gate[s] * (double)v[s].w);
                }
            }
            bad |= !finite_f32(total.x) || !finite_f32(total.y) || !finite_f32(total.z) || !finite_f32(total.w);
            const float4 published = bf16_round4(total);
            reinterpret_cast<float4 *>(collapsed)[at] = published;
            collapsed_squares += (double)published.x * (double)published.x;
            collapsed_squares += (double)published.y * (double)published.y;
            collapsed_squares += (double)published.z * (double)published.z;
            collapsed_squares += (double)published.w * (double)published.w;
        }
    } else {
        for (unsigned lane = tid - 64u; lane < width; lane += kWorkers) {
            float total = 0.0f;
            for (unsigned s = 0; s < streams; ++s)
                total += (float)(gate[s] * (double)bf16_round(in[s * width + lane]));
            bad |= !finite_f32(total);
            const float published = bf16_round(total);
            collapsed[lane] = published;
            collapsed_squares += (double)published * (double)published;
        }
    }

    // weighted RMS norm of the collapsed row, published as bf16 (the barriers inside the sum
    // order the collapsed values before any thread reads them)
    const double mean = workgroup_sum<THREADS / 64u>(collapsed_squares, slots) / (double)width;
    const double norm_inverse = 1.0 / sqrt(mean + rms_epsilon);
    bad |= !finite_f64(norm_inverse);
    if (quads && streams <= kBatch) {
        float4 *out4 = reinterpret_cast<float4 *>(normalized + row * width);
        const unsigned count = width >> 2;
        for (unsigned at = tid; at < count; at += THREADS) {
            const float4 w = coefficient4(norm, norm_qtype, at), v = reinterpret_cast<const float4 *>(collapsed)[at];
            const float in_lane[4] = {v.x, v.y, v.z, v.w}, weight[4] = {w.x, w.y, w.z, w.w};
            float value[4];
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) {
                double d = (double)in_lane[i] * norm_inverse;
                d *= (double)weight[i];
                value[i] = (float)d;
                bad |= !finite_f32(weight[i]) || !finite_f64(d) || !finite_f32(value[i]);
            }
            out4[at] = bf16_round4(make_float4(value[0], value[1], value[2], value[3]));
        }
    } else {
        for (unsigned lane = tid; lane < width; lane += THREADS) {
            const float weight = coefficient(norm, norm_qtype, lane);
            double v = (double)collapsed[lane] * norm_inverse;
            v *= (double)weight;
            const float value = (float)v;
            bad |= !finite_f32(weight) || !finite_f64(v) || !finite_f32(value);
            normalized[row * width + lane] = bf16_round(value);
        }
    }
    if (bad) raise_status(status, 1);
}

// One thread per (row, four lanes): the lanes' values in every stream are read once and every
// target stream's outputs are formed from them.
template <unsigned LANES>
__global__ __launch_bounds__(kEnvelopeThreads) void mhc_egress_kernel(
    const float *__restrict__ core, const float *__restrict__ rows, const float *__restrict__ post,
    const float *__restrict__ combination, unsigned long long row_count, unsigned streams,
    unsigned width, unsigned blocks_per_row, float *__restrict__ output, int *status)
{
    using Pack = typename std::conditional<LANES == 4u, float4, float>::type;
    const unsigned long long row = blockIdx.x / blocks_per_row;
    const unsigned lane = ((blockIdx.x % blocks_per_row) * kEnvelopeThreads + threadIdx.x) * LANES;
    if (row >= row_count || lane >= width) return;
    const unsigned expanded = streams * width;
    const float *in = rows + row * expanded;
    const float *mixing = combination + row * streams * streams;
    Pack loaded[kEnvelopeMaxStreams + 1u];
    loaded[kEnvelopeMaxStreams] = *reinterpret_cast<const Pack *>(core + row * width + lane);
#pragma unroll
    for (unsigned s = 0; s < kEnvelopeMaxStreams; ++s)
        if (s < streams) loaded[s] = *reinterpret_cast<const Pack *>(in + s * width + lane);
    double value[LANES], residual[kEnvelopeMaxStreams][LANES];
#pragma unroll
    for (unsigned i = 0; i < LANES; ++i) {
        value[i] = (double)reinterpret_cast<const float *>(&loaded[kEnvelopeMaxStreams])[i];
#pragma unroll
        for (unsigned s = 0; s < kEnvelopeMaxStreams; ++s)
            residual[s][i] = s < streams ? (double)bf16_round(reinterpret_cast<const float *>(&loaded[s])[i]) : 0.0;
    }
    bool bad = false;
    for (unsigned target = 0; target < streams; ++target) {
        const double gain = (double)post[row * streams + target];
        double weight[kEnvelopeMaxStreams];
#pragma unroll
        for (unsigned s = 0; s < kEnvelopeMaxStreams; ++s)
            weight[s] = s < streams ? (double)mixing[s * streams + target] : 0.0;
        Pack packed;
#pragma unroll
        for (unsigned i = 0; i < LANES; ++i) {
            double total = gain * value[i];
#pragma unroll
            for (unsigned s = 0; s < kEnvelopeMaxStreams; ++s)
                if (s < streams) total += weight[s] * residual[s][i];
            const float published = (float)total;
            bad |= !finite_f64(total) || !finite_f32(published);
            reinterpret_cast<float *>(&packed)[i] = bf16_round(published);
        }
        *reinterpret_cast<Pack *>(output + row * expanded + target * width + lane) = packed;
    }
    if (bad) raise_status(status, 1);
}

// The rank-ordered sum of the pairs' outputs, the shared expert and the egress in one pass over a
// row's columns (yvex_hip_moe_reduce_combine followed by yvex_hip_mhc_egress, the same operations in
// the same order): the combined row never goes to memory, and a decode batch has a launch less.
// A thread has one column: a few hundred instructions follow its loads, most of them double-precision, and a wave
// issues one in five cycles at best, so four columns a thread kept the few waves of a decode batch busy for longer than the
// memory took, and 87 registers kept a larger batch to five waves a SIMD. 4096 columns, six ranks, by 1 / 96 / 333 / 700 /
// 1111 / 2048 rows 7.5 / 13.8 / 30.7 / 50.6 / 70.7 / 114.5 us with four columns, 3.8 / 10.2 / 25.2 / 47.2 / 69.9 / 117.1 with one;
// eight ranks of 7168 columns by 2048 rows 209 and 213. The 2 % that 16-byte loads are ahead by at 2048 rows are not worth a
// second kernel. STREAMING: kPairsStreaming.
template <unsigned STREAMS, bool STREAMING>
__global__ __launch_bounds__(kEnvelopeThreads) void combine_egress_kernel(
    const float *__restrict__ pair_outputs, unsigned topk, const float *__restrict__ shared,
    const float *__restrict__ rows, const float *__restrict__ post, const float *__restrict__ combination,
    unsigned long long row_count, unsigned width, unsigned blocks_per_row, float *__restrict__ output, int *status)
{
    const unsigned long long row = blockIdx.x / blocks_per_row;
    const unsigned column = (blockIdx.x % blocks_per_row) * kEnvelopeThreads + threadIdx.x;
    if (row >= row_count || column >= width) return;
    const unsigned expanded = STREAMS * width;
    const float *in = rows + row * expanded + column;
    float residual[STREAMS];
#pragma unroll
    for (unsigned s = 0; s < STREAMS; ++s) residual[s] = in[s * width];
    const float base = shared[row * width + column];
    double gain[STREAMS], weight[STREAMS][STREAMS];
#pragma unroll
    for (unsigned t = 0; t < STREAMS; ++t) {
        gain[t] = (double)post[row * STREAMS + t];
#pragma unroll
        for (unsigned s = 0; s < STREAMS; ++s) weight[s][t] = (double)combination[(row * STREAMS + s) * STREAMS + t];
    }
    // ranks in order, four of them in flight
    float total = 0.0f;
    const float *source = pair_outputs + row * topk * width + column;
    for (unsigned rank = 0; rank < topk; rank += 4u) {
        float part[4];
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            const float *const from = source + (unsigned long long)(rank + k < topk ? rank + k : topk - 1u) * width;
            part[k] = STREAMING ? __builtin_nontemporal_load(from) : *from;
        }
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            if (rank + k >= topk) break;
            total += part[k];
        }
    }
    const float combined = bf16_round(total + base);
    bool bad = !finite_f32(total) || !finite_f32(combined);
    const double value = (double)combined;
#pragma unroll
    for (unsigned t = 0; t < STREAMS; ++t) {
        double sum = gain[t] * value;
#pragma unroll
        for (unsigned s = 0; s < STREAMS; ++s) sum += weight[s][t] * (double)bf16_round(residual[s]);
        const float published = (float)sum;
        bad |= !finite_f64(sum) || !finite_f32(published);
        output[row * expanded + t * width + column] = bf16_round(published);
    }
    if (bad) raise_status(status, 1);
}

}  // namespace yvex

using namespace yvex;

static bool envelope_shape_ok(uint64_t row_count, uint64_t streams, uint64_t width)
{
    return row_count && streams && streams <= kEnvelopeMaxStreams && width && width <= kEnvelopeMaxWidth &&
           row_count <= 0x7fffffffull / ((width + kEnvelopeThreads - 1u) / kEnvelopeThreads);
}

// The mixing projection that the ingress joins: its F32 weight rows, and scratch memory for the partial sums.
struct IngressProjection {
    const float *weights;
    void *scratch;
    uint64_t scratch_bytes;
};

static int launch_mhc_ingress(const float *rows, const float *mixes, const void *scale, unsigned scale_qtype,
                              const void *base, unsigned base_qtype, const void *norm, unsigned norm_qtype,
                              uint64_t row_count, uint64_t streams, uint64_t width, uint64_t iterations,
                              double rms_epsilon, double mhc_epsilon, double post_multiplier,
                              float *normalized, float *post, float *combination, int *status,
                              yvex_hip_stream stream, const IngressProjection *projection = nullptr)
{
    if (!rows || (!mixes && !projection) || !scale || !base || !norm || !normalized || !post || !combination || !status)
        return ST_INVALID_ARG;
    const unsigned qtypes[3] = {scale_qtype, base_qtype, norm_qtype};
    const void *const vectors[3] = {scale, base, norm};
    for (int k = 0; k < 3; ++k) {
        if (qtypes[k] != QT_F32 && qtypes[k] != QT_BF16) return ST_UNSUPPORTED;
        if ((uintptr_t)vectors[k] & (qtypes[k] == QT_F32 ? 3u : 1u)) return ST_INVALID_ARG;
    }
    if (!envelope_shape_ok(row_count, streams, width) || !iterations || iterations > 0xffffffffull)
        return ST_BOUNDS;
    if (!(rms_epsilon > 0.0) || !(mhc_epsilon > 0.0) || !(post_multiplier > 0.0) ||
        rms_epsilon > 1.0e300 || mhc_epsilon > 1.0e300 || post_multiplier > 1.0e300)
        return ST_INVALID_ARG;
    static std::once_flag once;
    static bool prepared = false;
    std::call_once(once, [] {
        prepared = true;
        for (const void *kernel : {(const void *)mhc_ingress_kernel<256, false>, (const void *)mhc_ingress_kernel<256, true>,
                                   (const void *)mhc_ingress_kernel<1024, false>, (const void *)mhc_ingress_kernel<1024, true>})
            prepared = prepared && hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)kEnvelopeLdsBytes) == hipSuccess;
        if (!prepared) (void)hipGetLastError();
    });
    if (!prepared) {
        set_last_error_text("mhc_ingress: the collapsed row does not fit in LDS");
        return ST_BACKEND;
    }
    const int quads = width % 4u == 0u && !(((uintptr_t)rows | (uintptr_t)normalized) & 15u) &&
                      !((uintptr_t)norm & (norm_qtype == QT_F32 ? 15u : 7u));
    const bool split = 2u * row_count <= (uint64_t)compute_units(), wide = streams * width >= 8192u;
    unsigned splits = 0u, parts_bytes = 0u;
    if (projection) {
        const uint64_t mixing_rows = (streams + 2u) * streams, expanded = streams * width;
        splits = f32_rows_splits(mixing_rows, expanded, row_count);
        if (yvex_hip_matvec_f32_rows_launches(projection->weights, mixing_rows, expanded, rows, row_count, expanded,
                                              projection->scratch, projection->scratch_bytes) != 2u)
            return ST_UNSUPPORTED;
        if (splits * mixing_rows > kPartsAThread * (wide ? 1024u : 256u)) return ST_BOUNDS;    // (never: kPartsAThread)
        parts_bytes = (unsigned)(splits * mixing_rows * sizeof(double));
    }
    // The collapsed row and the partial sums always fit; the row itself is held where there is room for it besides.
    static_assert(kEnvelopeMaxWidth * sizeof(float) + kPartsAThread * 1024u * sizeof(double) <= kEnvelopeLdsBytes,
                  "the collapsed row and the partial sums");
    const unsigned collapsed_bytes = (unsigned)(width * sizeof(float)), row_bytes = (unsigned)(2u * streams * width);
    const int held = split && quads && streams <= 4u && collapsed_bytes + row_bytes + parts_bytes <= kEnvelopeLdsBytes;
    const unsigned parts_at = (collapsed_bytes + (held ? row_bytes : 0u) + 7u) & ~7u, lds = parts_at + parts_bytes;
    if (projection) {
        const uint64_t mixing_rows = (streams + 2u) * streams, expanded = streams * width;
        const int rc = launch_f32_rows_parts(projection->weights, mixing_rows, expanded, rows, row_count, expanded,
                                             (double *)projection->scratch, status, as_stream(stream));
        if (rc) return rc;
    }
    const auto kernel = wide ? (split ? mhc_ingress_kernel<1024, true> : mhc_ingress_kernel<1024, false>)
                             : (split ? mhc_ingress_kernel<256, true> : mhc_ingress_kernel<256, false>);
    kernel<<<(unsigned)(split ? 2u * row_count : row_count), wide ? 1024 : 256, lds, as_stream(stream)>>>(
        rows, mixes, scale, base, norm, scale_qtype, base_qtype, norm_qtype, (unsigned)streams, (unsigned)width,
        (unsigned)iterations, rms_epsilon, mhc_epsilon, post_multiplier, normalized, post, combination, quads, held,
        projection ? (const double *)projection->scratch : nullptr, splits, parts_at / 4u, status);
    return check_launch("mhc_ingress");
}

extern "C" int yvex_hip_mhc_ingress(const float *rows, const float *mixes, const float *scale,
                                    const float *base, const float *norm, uint64_t row_count,
                                    uint64_t streams, uint64_t width, uint64_t iterations,
                                    double rms_epsilon, double mhc_epsilon, double post_multiplier,
                                    float *normalized, float *post, float *combination, int *status,
                                    yvex_hip_stream stream)
{
    return launch_mhc_ingress(rows, mixes, scale, QT_F32, base, QT_F32, norm, QT_F32, row_count, streams, width,
                              iterations, rms_epsilon, mhc_epsilon, post_multiplier, normalized, post,
                              combination, status, stream);
}

extern "C" int yvex_hip_mhc_ingress_encoded(const float *rows, const float *mixes, const void *scale,
                                            unsigned int scale_qtype, const void *base,
                                            unsigned int base_qtype, const void *norm,
                                            unsigned int norm_qtype, uint64_t row_count, uint64_t streams,
                                            uint64_t width, uint64_t iterations, double rms_epsilon,
                                            double mhc_epsilon, double post_multiplier, float *normalized,
                                            float *post, float *combination, int *status,
                                            yvex_hip_stream stream)
{
    return launch_mhc_ingress(rows, mixes, scale, scale_qtype, base, base_qtype, norm, norm_qtype, row_count,
                              streams, width, iterations, rms_epsilon, mhc_epsilon, post_multiplier, normalized,
                              post, combination, status, stream);
}

extern "C" int yvex_hip_mhc_ingress_projecting(const float *rows, const float *function, const void *scale,
                                               unsigned int scale_qtype, const void *base,
                                               unsigned int base_qtype, const void *norm,
                                               unsigned int norm_qtype, uint64_t row_count, uint64_t streams,
                                               uint64_t width, uint64_t iterations, double rms_epsilon,
                                               double mhc_epsilon, double post_multiplier, float *normalized,
                                               float *post, float *combination, void *scratch,
                                               uint64_t scratch_bytes, int *status, yvex_hip_stream stream)
{
    const IngressProjection projection{function, scratch, scratch_bytes};
    return launch_mhc_ingress(rows, nullptr, scale, scale_qtype, base, base_qtype, norm, norm_qtype, row_count, streams,
                              width, iterations, rms_epsilon, mhc_epsilon, post_multiplier, normalized, post,
                              combination, status, stream, &projection);
}

extern "C" int yvex_hip_mhc_egress(const float *core, const float *rows, const float *post,
                                   const float *combination, uint64_t row_count, uint64_t streams,
                                   uint64_t width, float *output, int *status, yvex_hip_stream stream)
{
    if (!core || !rows || !post || !combination || !output || !status || output == rows)
        return ST_INVALID_ARG;
    if (!envelope_shape_ok(row_count, streams, width)) return ST_BOUNDS;
    const bool quads = width % 4u == 0u && !(((uintptr_t)core | (uintptr_t)rows | (uintptr_t)output) & 15u);
    const uint64_t threads = quads ? width / 4u : width;
    const unsigned blocks_per_row = (unsigned)((threads + kEnvelopeThreads - 1u) / kEnvelopeThreads);
    if (quads)
        mhc_egress_kernel<4><<<(unsigned)(row_count * blocks_per_row), kEnvelopeThreads, 0, as_stream(stream)>>>(
            core, rows, post, combination, row_count, (unsigned)streams, (unsigned)width, blocks_per_row,
            output, status);
    else
        mhc_egress_kernel<1><<<(unsigned)(row_count * blocks_per_row), kEnvelopeThreads, 0, as_stream(stream)>>>(
            core, rows, post, combination, row_count, (unsigned)streams, (unsigned)width, blocks_per_row,
            output, status);
    return check_launch("mhc_egress");
}

// From here on pair outputs, which nobody reads again, are loaded past the caches: six ranks of 4096 columns by 300 / 500 / 700 / 1111 / 1500 /
// 2048 rows (29 to 201 MB) 17.1 / 25.5 / 34.5 / 51.9 / 68.7 / 92.7 us so, 16.5 / 25.7 / 35.7 / 55.2 / 72.8 / 95.0 through them, and the ingress of the
// layer behind 1 to 2 us less, whose rows stay in the caches.
constexpr uint64_t kPairsStreaming = 64ull << 20;

// Four streams, widths of whole 16-byte pieces; UNSUPPORTED otherwise (the two launches serve those).
extern "C" int yvex_hip_moe_combine_egress(const float *pair_outputs, uint64_t row_count, uint64_t topk,
                                           uint64_t streams, uint64_t width, const float *shared, const float *rows,
                                           const float *post, const float *combination, float *output, int *status,
                                           yvex_hip_stream stream)
{
    if (!pair_outputs || !shared || !rows || !post || !combination || !output || !status || output == rows || !topk ||
        topk > 0xffffu)
        return ST_INVALID_ARG;
    if (!envelope_shape_ok(row_count, streams, width)) return ST_BOUNDS;
    if (streams != 4u || width % 4u ||
        (((uintptr_t)pair_outputs | (uintptr_t)shared | (uintptr_t)rows | (uintptr_t)output) & 15u))
        return ST_UNSUPPORTED;
    const unsigned blocks_per_row = (unsigned)((width + kEnvelopeThreads - 1u) / kEnvelopeThreads);
    const auto kernel = row_count * topk * width * sizeof(float) > kPairsStreaming ? combine_egress_kernel<4, true> : combine_egress_kernel<4, false>;
    kernel<<<(unsigned)(row_count * blocks_per_row), kEnvelopeThreads, 0, as_stream(stream)>>>(
        pair_outputs, (unsigned)topk, shared, rows, post, combination, row_count, (unsigned)width, blocks_per_row,
        output, status);
    return check_launch("moe_combine_egress");
}
