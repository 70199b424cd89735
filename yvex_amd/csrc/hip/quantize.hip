// Q8_K activation quantizer for gfx950: a 64-lane wavefront four blocks of 256 values, or one where other work rides along (q8k.hpp).
#include "common.hpp"
#include "q8k.hpp"
#include "q8_0_rows.hpp"
#include "launch.hpp"
#include "grouped.hpp"

namespace yvex {

__global__ __launch_bounds__(256) void q8k_quantize_kernel(
    const float *__restrict__ values, unsigned long long rows, unsigned long long blocks,
    unsigned long long input_stride, unsigned char *__restrict__ encoded, int *status)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long tasks = rows * blocks;
    const unsigned long long task = ((unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6)) * 4ull + (lane >> 4);
    const unsigned long long held = task < tasks ? task : tasks - 1ull;
    // (rows end to end, as the layers' are, need no row number)
    const float *x = values + held * 256ull;
    if (input_stride != blocks * 256ull) {
        const unsigned long long row = held / blocks;
        x = values + row * input_stride + (held - row * blocks) * 256ull;
    }
    float v[4][4];
#pragma unroll
    for (unsigned k = 0; k < 4u; ++k) __builtin_memcpy(v[k], x + 4u * (lane & 15u) + 64u * k, 16);
    q8k_quantize_four(v, encoded + held * kQ8KBytes, lane, task < tasks, status);
}

// The same for a layer's intermediate rows where a shared expert's gate and up sums come from dense
// projections: behind the routed pairs' rows the shared rows' values are formed on the way in, the
// clamped SwiGLU product rounded to bfloat16 (what yvex_hip_moe_swiglu_rows stores). A launch and a
// round trip of the rows through memory less.
// Four routed blocks a wavefront as above, behind the workgroups of the shared ones, a block a wavefront: one product in
// five hundred takes the path in double, and a wavefront of four blocks meets it twice (96 rows 5.5 -> 6.9 us so).
__global__ __launch_bounds__(256) void q8k_quantize_swiglu_kernel(
    const float *__restrict__ values, unsigned long long rows, unsigned long long blocks,
    unsigned char *__restrict__ encoded, const float *__restrict__ gate, const float *__restrict__ up,
    unsigned long long shared_rows, double limit, unsigned char *__restrict__ shared_encoded, int *status)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long shared_tasks = shared_rows * blocks, shared_groups = (shared_tasks + 3ull) / 4ull;
    if (blockIdx.x >= shared_groups) {
        const unsigned long long tasks = rows * blocks;
        const unsigned long long task = ((blockIdx.x - shared_groups) * 4ull + (threadIdx.x >> 6)) * 4ull + (lane >> 4);
        const unsigned long long held = task < tasks ? task : tasks - 1ull;
        const float4 *const x = reinterpret_cast<const float4 *>(values + held * 256ull) + (lane & 15u);
        float v[4][4];
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) {
            const float4 x4 = x[16u * k];
            v[k][0] = x4.x, v[k][1] = x4.y, v[k][2] = x4.z, v[k][3] = x4.w;
        }
        q8k_quantize_four(v, encoded + held * kQ8KBytes, lane, task < tasks, status);
        return;
    }
    const unsigned long long shared_task = blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (shared_task >= shared_tasks) return;
    const float4 g = *reinterpret_cast<const float4 *>(gate + shared_task * 256ull + lane * 4u);
    const float4 u = *reinterpret_cast<const float4 *>(up + shared_task * 256ull + lane * 4u);
    const float v[4] = {swiglu_bf16_fast(g.x, u.x, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.y, u.y, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.z, u.z, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.w, u.w, 1.0f, limit, (float)limit)};
    q8k_quantize_values(v, shared_encoded + shared_task * kQ8KBytes, lane, status);
}

// One or two shared rows of which a Q8_0 projection is wanted: the products of their gate and up sums, quantized by every
// workgroup of the projection for itself.
struct HoldSwiglu {
    const float *gate, *up;
    unsigned tasks;
    double limit;
    int *status;
    float4 g, u;
    __device__ __forceinline__ void request(unsigned task)
    {
        const unsigned at = (task < tasks ? task : tasks - 1u) * 64u + (threadIdx.x & 63u);
        g = reinterpret_cast<const float4 *>(gate)[at];
        u = reinterpret_cast<const float4 *>(up)[at];
    }
    __device__ __forceinline__ void finish(unsigned wave, unsigned char *held)
    {
        for (unsigned task = wave; task < tasks; task += kHeldWaves) {
            const float v[4] = {swiglu_bf16_fast(g.x, u.x, 1.0f, limit, (float)limit),
                                swiglu_bf16_fast(g.y, u.y, 1.0f, limit, (float)limit),
                                swiglu_bf16_fast(g.z, u.z, 1.0f, limit, (float)limit),
                                swiglu_bf16_fast(g.w, u.w, 1.0f, limit, (float)limit)};
            hold_block(v, held + task * kHeldBlock, threadIdx.x & 63u, status);
            if (task + kHeldWaves < tasks) request(task + kHeldWaves);
        }
    }
};

// The routed rows quantized, sixteen blocks a workgroup, and beside them the shared expert's down projection of one or
// two rows from its gate and up sums: a launch less, and the quantized shared rows stay out of memory. Six
// routed rows of 2048 columns and one shared row against 4096 x 2048: 5.0 and 4.8 us for the two launches, 6.2 for this one.
template <int T>
__global__ __launch_bounds__(kHeldThreads) void q8k_quantize_swiglu_projecting_kernel(
    const float *__restrict__ values, unsigned tasks, unsigned blocks, unsigned char *__restrict__ encoded,
    const float *__restrict__ gate, const float *__restrict__ up, unsigned shared_rows, double limit,
    const unsigned char *__restrict__ down, unsigned long long row_count, unsigned long long row_bytes,
    float *__restrict__ out, int *status)
{
    extern __shared__ __align__(16) unsigned char held[];
    const unsigned lane = threadIdx.x & 63u, before = (tasks + kHeldWaves - 1u) / kHeldWaves;
    if (blockIdx.x < before) {
        const unsigned task = blockIdx.x * kHeldWaves + (threadIdx.x >> 6);
        if (task < tasks)
            q8k_quantize_block(values + task * 256ull + lane * 4u, encoded + (unsigned long long)task * kQ8KBytes, lane, status);
        return;
    }
    HoldSwiglu hold{gate, up, shared_rows * blocks, limit, status, {}, {}};
    held_rows<T, 1>(row_count, blockIdx.x - before, gridDim.x - before, 8u * blocks, held,
                    [&](unsigned long long row) { return down + row * row_bytes; }, hold,
                    [&](unsigned in, unsigned long long row, float sum) {
                        if (in >= shared_rows) return;
                        if (!finite_f32(sum)) raise_status(status, 1);
                        else out[in * row_count + row] = bf16_round(sum);
                    });
}

// Rows of a split input laid end to end, each value rounded to bf16 as the reference's split
// projection rounds it (src/backend/cuda/kernels.cu:736-782).
__global__ __launch_bounds__(256) void concat_rows_bf16_kernel(
    const float *__restrict__ head, const float *__restrict__ tail, unsigned long long rows,
    unsigned head_width, unsigned tail_width, float *__restrict__ out, int *status)
{
    const unsigned width = head_width + tail_width;
    const unsigned long long index = (unsigned long long)blockIdx.x * 256ull + threadIdx.x;
    if (index >= rows * width) return;
    const unsigned long long row = index / width;
    const unsigned column = (unsigned)(index % width);
    const float value = bf16_round(column < head_width ? head[row * head_width + column]
                                                       : tail[row * tail_width + (column - head_width)]);
    if (!finite_f32(value)) raise_status(status, 1);
    out[index] = value;
}

}  // namespace yvex

using namespace yvex;

extern "C" int yvex_hip_q8k_quantize(const float *values, uint64_t rows, uint64_t width,
                                     uint64_t input_stride, uint8_t *encoded, int *status,
                                     yvex_hip_stream stream)
{
    if (!values || !encoded || !status || !rows || !width || width % 256u ||
        input_stride < width || ((uintptr_t)encoded & 3u) || ((uintptr_t)values & 3u))
        return ST_INVALID_ARG;
    const uint64_t blocks = width / 256u;
    if (rows > UINT64_MAX / blocks) return ST_BOUNDS;
    const uint64_t tasks = rows * blocks, grid = (tasks + 15u) / 16u;
    if (grid > 0x1fffffffull) return ST_BOUNDS;
    q8k_quantize_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        values, rows, blocks, input_stride, encoded, status);
    return check_launch("q8k_quantize");
}

extern "C" int yvex_hip_q8k_quantize_swiglu(const float *values, uint64_t rows, uint64_t width, uint8_t *encoded,
                                            const float *gate, const float *up, uint64_t shared_rows,
                                            double limit, uint8_t *shared_encoded, int *status,
                                            yvex_hip_stream stream)
{
    if (!values || !encoded || !gate || !up || !shared_encoded || !status || !rows || !shared_rows || !width ||
        width % 256u || !(limit > 0.0) || ((uintptr_t)encoded & 3u) || ((uintptr_t)shared_encoded & 3u) ||
        (((uintptr_t)values | (uintptr_t)gate | (uintptr_t)up) & 15u))
        return ST_INVALID_ARG;
    const uint64_t blocks = width / 256u;
    if (rows > 0xffffffffull || shared_rows > 0xffffffffull) return ST_BOUNDS;
    const uint64_t grid = (rows * blocks + 15u) / 16u + (shared_rows * blocks + 3u) / 4u;
    if (grid > 0x1fffffffull) return ST_BOUNDS;
    q8k_quantize_swiglu_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        values, rows, blocks, encoded, gate, up, shared_rows, limit, shared_encoded, status);
    return check_launch("q8k_quantize_swiglu");
}

extern "C" int yvex_hip_q8k_quantize_swiglu_projecting_supported(const uint8_t *down, uint64_t row_count, uint64_t row_bytes,
                                                                 uint64_t shared_rows, uint64_t width)
{
    return down && !((uintptr_t)down & 1u) && shared_rows && shared_rows <= 2u && width && width % 256u == 0u &&
           width <= 14336u && shared_rows * (width / 256u) <= 56u && row_bytes == width / 32u * 34u && row_count &&
           row_count <= 0xffffffffull;
}

extern "C" int yvex_hip_q8k_quantize_swiglu_projecting(const float *values, uint64_t rows, uint64_t width, uint8_t *encoded,
                                                       const float *gate, const float *up, uint64_t shared_rows,
                                                       double limit, const uint8_t *down, uint64_t row_count,
                                                       uint64_t row_bytes, float *out, int *status, yvex_hip_stream stream)
{
    if (!values || !encoded || !gate || !up || !out || !status || !rows || !(limit > 0.0) || ((uintptr_t)encoded & 3u) ||
        ((uintptr_t)out & 3u) || (((uintptr_t)values | (uintptr_t)gate | (uintptr_t)up) & 15u))
        return ST_INVALID_ARG;
    if (!yvex_hip_q8k_quantize_swiglu_projecting_supported(down, row_count, row_bytes, shared_rows, width))
        return ST_UNSUPPORTED;
    const uint64_t blocks = width / 256u;
    if (rows > 0xffffffffull / blocks) return ST_BOUNDS;
    const uint64_t groups = (row_count + kHeldWaves - 1u) / kHeldWaves, most = (uint64_t)compute_units();
    const uint64_t grid = (rows * blocks + kHeldWaves - 1u) / kHeldWaves + (groups < most ? groups : most);
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    const auto kernel = shared_rows == 1u ? q8k_quantize_swiglu_projecting_kernel<1> : q8k_quantize_swiglu_projecting_kernel<2>;
    kernel<<<(unsigned)grid, kHeldThreads, (size_t)held_bytes(shared_rows, blocks), as_stream(stream)>>>(
        values, (unsigned)(rows * blocks), (unsigned)blocks, encoded, gate, up, (unsigned)shared_rows, limit, down, row_count,
        row_bytes, out, status);
    return check_launch("q8k_quantize_swiglu_projecting");
}

extern "C" int yvex_hip_concat_rows_bf16(const float *head, const float *tail, uint64_t rows,
                                         uint64_t head_width, uint64_t tail_width, float *out,
                                         int *status, yvex_hip_stream stream)
{
    if (!head || !tail || !out || !status || !rows || !head_width || !tail_width) return ST_INVALID_ARG;
    if (head_width + tail_width > 0xffffffffull || rows > UINT64_MAX / (head_width + tail_width))
        return ST_BOUNDS;
    const uint64_t grid = (rows * (head_width + tail_width) + 255u) / 256u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    concat_rows_bf16_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        head, tail, rows, (unsigned)head_width, (unsigned)tail_width, out, status);
    return check_launch("concat_rows_bf16");
}
