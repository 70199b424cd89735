// Q8_K activation quantizer for gfx950: one 64-lane wavefront per 256-value block (q8k.hpp).
#include "common.hpp"
#include "q8k.hpp"
#include "launch.hpp"
#include "grouped.hpp"

namespace yvex {

__global__ __launch_bounds__(256) void q8k_quantize_kernel(
    const float *__restrict__ values, unsigned long long rows, unsigned long long blocks,
    unsigned long long input_stride, unsigned char *__restrict__ encoded, int *status)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long task = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (task >= rows * blocks) return;
    const unsigned long long row = task / blocks, block = task % blocks;
    q8k_quantize_block(values + row * input_stride + block * 256ull + lane * 4u, encoded + task * kQ8KBytes,
                       lane, status);
}

// The same for a layer's intermediate rows where a shared expert's gate and up sums come from dense
// projections: behind the routed pairs' rows the shared rows' values are formed on the way in, the
// clamped SwiGLU product rounded to bfloat16 (what yvex_hip_moe_swiglu_rows stores). A launch and a
// round trip of the rows through memory less.
__global__ __launch_bounds__(256) void q8k_quantize_swiglu_kernel(
    const float *__restrict__ values, unsigned long long rows, unsigned long long blocks,
    unsigned char *__restrict__ encoded, const float *__restrict__ gate, const float *__restrict__ up,
    unsigned long long shared_rows, double limit, unsigned char *__restrict__ shared_encoded, int *status)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long task = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (task < rows * blocks) {
        q8k_quantize_block(values + task * 256ull + lane * 4u, encoded + task * kQ8KBytes, lane, status);
        return;
    }
    const unsigned long long shared_task = task - rows * blocks;
    if (shared_task >= shared_rows * blocks) return;
    const float4 g = *reinterpret_cast<const float4 *>(gate + shared_task * 256ull + lane * 4u);
    const float4 u = *reinterpret_cast<const float4 *>(up + shared_task * 256ull + lane * 4u);
    const float v[4] = {swiglu_bf16_fast(g.x, u.x, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.y, u.y, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.z, u.z, 1.0f, limit, (float)limit),
                        swiglu_bf16_fast(g.w, u.w, 1.0f, limit, (float)limit)};
    q8k_quantize_values(v, shared_encoded + shared_task * kQ8KBytes, lane, status);
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
    const uint64_t tasks = rows * blocks, grid = (tasks + 3u) / 4u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
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
    const uint64_t grid = ((rows + shared_rows) * blocks + 3u) / 4u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    q8k_quantize_swiglu_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        values, rows, blocks, encoded, gate, up, shared_rows, limit, shared_encoded, status);
    return check_launch("q8k_quantize_swiglu");
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
