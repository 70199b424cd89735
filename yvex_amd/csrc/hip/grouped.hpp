// Problem description shared by the grouped expert kernels (decode-width sweeps and the MFMA
// row-batch kernel): one set of expert matrices, the activation rows and the expert-major worklist.
#pragma once

#include "common.hpp"
#include "exp_negative.hpp"
#include "launch.hpp"
#include "lds_copy.hpp"

namespace yvex {

constexpr int kPass = 2;          // pairs of one bucket handled per sweep over the expert's bytes
constexpr int kUnitsPerLane = 4;  // a sweep lane owns half a superblock: 128 columns

// One set of expert matrices plus the pairs that use it.
struct GroupedProblem {
    const unsigned char *gate, *up;          // up == nullptr: plain projection (down)
    unsigned long long row_bytes, expert_bytes, up_row_bytes, up_expert_bytes;
    const void *activations;                 // Q8_K rows or F32 rows
    unsigned long long act_stride;           // bytes between activation rows
    int act_by_ordered_pair;                 // 1: activation row = ordered position (down)
    const unsigned long long *order, *expert_ids, *bucket_offsets, *bucket_populations;
    const unsigned long long *sweep_offsets, *counts;
    const float *route_weights;
    unsigned pairs, topk, experts;
    float *out;                              // [ordered or source pair][out_rows]
    int out_by_source_pair;
    unsigned sweeps;                         // single known bucket: ceil(pairs / kPass), else 0
};

struct GroupedArgs {
    GroupedProblem problem[2];               // [0] routed experts, [1] optional shared expert
    unsigned problems;
    unsigned width;                          // reduction width (activation row length)
    unsigned out_rows;                       // rows of the weight matrix per expert
    unsigned item_rows;                      // weight rows (row pairs when fused) per work item
    double limit;
    int *status;
    int image;                               // weights are the IQ2_XXS sweep image (72 B a superblock)
};

// The same value from fp32 arithmetic when that provably rounds to the same bfloat16. For
// |gate| <= 16 the fp32 result is within about 24 units in the last place of the exact one (the
// rounded product gate * log2(e) and the rounded constant contribute up to 19 of them, exp2,
// reciprocal, 1 + t and the multiplications the rest), so unless its low 16 bits sit within 64
// of the rounding midpoint the two roundings agree. Otherwise, and for non-finite or vanishing
// values, the double path decides.
__device__ __forceinline__ float swiglu_bf16(float g, float u, float route_weight, double limit);
__device__ __forceinline__ float swiglu_bf16_fast(float g, float u, float route_weight,
                                                  double limit, float limit_f32)
{
    const float gv = fminf(g, limit_f32);
    const float uv = fmaxf(-limit_f32, fminf(u, limit_f32));
    const float t = __builtin_amdgcn_exp2f(-fabsf(gv) * 1.44269504088896340736f);
    const float r = __builtin_amdgcn_rcpf(1.0f + t);
    const float silu = gv >= 0.0f ? gv * r : gv * t * r;
    const float v = silu * uv * route_weight;
    const unsigned bits = __float_as_uint(v), low = bits & 0xffffu;
    // (one branch: the tests are combined without short circuits)
    const bool finite = finite_f32(v), large = fabsf(v) > 1.0e-30f, inside = fabsf(gv) <= 16.0f;
    const bool clear = (low < 0x8000u - 64u) | (low > 0x8000u + 64u);
    const bool safe = ((double)limit_f32 == limit) & finite & large & inside & clear;
    if (safe) return bf16_round(v);
    return swiglu_bf16(g, u, route_weight, limit);
}

// SiLU-gated product in double, as src/graph/moe.c:605-611 orders it.
__device__ __forceinline__ float swiglu_bf16(float g, float u, float route_weight, double limit)
{
    const double gv = fmin((double)g, limit);
    const double uv = fmax(-limit, fmin((double)u, limit));
    const double t = exp_of_negative(-fabs(gv));
    const double silu = gv >= 0.0 ? gv / (1.0 + t) : gv * t / (1.0 + t);
    return bf16_round((float)(silu * uv * (double)route_weight));
}

// Geometry of a matrix given as the IQ2_XXS sweep image.
static inline int check_image_matrix(unsigned qtype, uint64_t width, uint64_t row_bytes, const void *base,
                                     uint64_t expert_bytes)
{
    if (qtype != QT_IQ2_XXS) return ST_UNSUPPORTED;
    if (!width || width % 256u || width / 256u * 72u != row_bytes) return ST_BOUNDS;
    if (((uintptr_t)base & 3u) || (expert_bytes & 3u)) return ST_INVALID_ARG;
    return ST_OK;
}

static inline int check_matrix(unsigned qtype, uint64_t width, uint64_t row_bytes)
{
    unsigned block, bytes;
    if (!qtype_geometry(qtype, block, bytes) || block < 32u) return ST_UNSUPPORTED;
    if (!width || width % 256u || width / block * bytes != row_bytes) return ST_BOUNDS;
    if (width / 32u > 64u * kUnitsPerLane) return ST_UNSUPPORTED;   // one wave spans a row
    return ST_OK;
}

struct WorklistView {
    const uint64_t *order, *expert_ids, *bucket_offsets, *bucket_populations, *sweep_offsets, *counts;
};

static inline void fill_up_problem(GroupedProblem &p, const yvex_hip_expert_weights *w,
                            const void *activations, int act_q8, const float *route_weights,
                            const WorklistView &wl, uint64_t pairs, uint64_t topk, uint64_t experts,
                            float *out)
{
    p.gate = w->gate;
    p.up = w->up;
    p.row_bytes = w->gate_row_bytes;
    p.expert_bytes = w->gate_expert_bytes;
    p.up_row_bytes = w->up_row_bytes;
    p.up_expert_bytes = w->up_expert_bytes;
    p.activations = activations;
    p.act_stride = act_q8 ? w->hidden / 256u * kQ8KBytes : w->hidden * sizeof(float);
    p.act_by_ordered_pair = 0;
    p.order = (const unsigned long long *)wl.order;
    p.expert_ids = (const unsigned long long *)wl.expert_ids;
    p.bucket_offsets = (const unsigned long long *)wl.bucket_offsets;
    p.bucket_populations = (const unsigned long long *)wl.bucket_populations;
    p.sweep_offsets = (const unsigned long long *)wl.sweep_offsets;
    p.counts = (const unsigned long long *)wl.counts;
    p.route_weights = route_weights;
    p.pairs = (unsigned)pairs;
    p.topk = (unsigned)topk;
    p.experts = (unsigned)experts;
    p.out = out;
    p.out_by_source_pair = 0;
    p.sweeps = wl.expert_ids ? 0u : (unsigned)((pairs + kPass - 1u) / kPass);
}

static inline void fill_down_problem(GroupedProblem &p, const yvex_hip_expert_weights *w,
                              const void *intermediate, int act_q8, const WorklistView &wl,
                              uint64_t pairs, uint64_t experts, float *out)
{
    p.gate = w->down;
    p.up = nullptr;
    p.row_bytes = w->down_row_bytes;
    p.expert_bytes = w->down_expert_bytes;
    p.up_row_bytes = p.up_expert_bytes = 0;
    p.activations = intermediate;
    p.act_stride = act_q8 ? w->intermediate / 256u * kQ8KBytes : w->intermediate * sizeof(float);
    p.act_by_ordered_pair = 1;
    p.order = (const unsigned long long *)wl.order;
    p.expert_ids = (const unsigned long long *)wl.expert_ids;
    p.bucket_offsets = (const unsigned long long *)wl.bucket_offsets;
    p.bucket_populations = (const unsigned long long *)wl.bucket_populations;
    p.sweep_offsets = (const unsigned long long *)wl.sweep_offsets;
    p.counts = (const unsigned long long *)wl.counts;
    p.route_weights = nullptr;
    p.pairs = (unsigned)pairs;
    p.topk = 1u;
    p.experts = (unsigned)experts;
    p.out = out;
    p.out_by_source_pair = 1;
    p.sweeps = wl.expert_ids ? 0u : (unsigned)((pairs + kPass - 1u) / kPass);
}

// Specialised IQ2_XXS x Q8_K decode sweeps (sweep_iq2.hip): reduction widths whose rows span 16
// to 64 lanes of 128 columns each.
bool iq2_sweep_supported(unsigned qtype, unsigned width, unsigned out_rows, unsigned long long pairs, bool image);
int launch_iq2_sweep(const GroupedArgs &a, unsigned qtype, bool fused, bool image, hipStream_t stream);

// Pairs behind a bucket's whole 64-pair tiles that are the few-pair kernels' (rows16.hip), by the same rule there and
// in the 64-pair kernels. A tile of theirs takes `few`. Where that leaves the 64-pair kernels with nothing but a few
// buckets' single tiles, two tiles of theirs take those too: a launch of the 64-pair kernels is one tile's time however
// few it holds (54 us of gate/up and 28 us of Q2_K down rows at width 4096 for one bucket or sixteen), a bucket in two
// tiles 2.6 and 1.5 us of the whole device. Two tiles in every bucket of 256 are the slower way: 665 us
// against 600 (width 4096, 24 pairs), 1148 against 935 (7168, fourteen); and beside a launch that is long anyway
// they gain nothing (1111 uneven rows of Q4_K 2570 us without, 2650 with). Taken again with products of the scales on the matrix
// cores in the 64-pair kernels: 420 even rows of 7168 by eight of 256 Q4_K experts 1657 us so, 1815 with two tiles in up to 64
// buckets or all; of 4096 by six in the model file's formats 666 so, 694 with a bucket never in two; uneven ones within 1 % (2.5 % at 1600
// rows of Q4_K, two tiles in every bucket). Every thread of a block calls this, a thread a
// bucket, those without one with 0; `lds` is the address of four words of LDS that hold nothing (the kernels leave no
// room for static LDS).
constexpr unsigned kFewPairSeconds = 16u;
__device__ __forceinline__ unsigned few_pair_limit(unsigned few, unsigned long long population, unsigned lds)
{
    const unsigned seconds = (unsigned)__popcll(__ballot(population > few && population <= 2u * few));
    const unsigned members = __ballot(population > 2u * few) ? kFewPairSeconds + 1u : seconds, wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0u && wave < 4u) lds_write_u32(lds + 4u * wave, members);
    __syncthreads();
    const unsigned all = lds_read_u32(lds) + lds_read_u32(lds + 4u) + lds_read_u32(lds + 8u) + lds_read_u32(lds + 12u);
    return all <= kFewPairSeconds ? 2u * few : few;
}

// Row-batch expert kernels on the int8 matrix cores (rows_q4k.hip): Q4_K weights, fused gate/up
// or a plain projection; Q2_K weights, a plain projection (the down experts). A bucket's last tile is left to
// the kernels below where few_pair_limit says so. `beside`, or null: a matrix alone of the same formats and sizes, in the
// same launch.
int launch_q4k_rows_grouped(const GroupedProblem &problem, unsigned qtype, bool fused, uint64_t width,
                            uint64_t out_rows, unsigned few, const GroupedProblem *beside, double limit, int *status,
                            hipStream_t stream);

// The same problems where few pairs meet (rows16.hip): IQ2_XXS (canonical bytes, or the sweep image) and
// Q4_K rows, fused gate/up or plain; Q2_K rows, plain. The first: pairs of a full tile, 0 for a problem
// the kernels do not serve. The second serves whole buckets (`behind` 0), or what a bucket holds
// behind whole tiles of `behind` pairs where few_pair_limit admits that; a plain projection's sums are rounded
// to bfloat16 where `round` says so.
unsigned rows16_tokens(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, uint64_t width,
                       uint64_t out_rows);
// Whether a matrix alone comes out at one round of the kernels' waves.
bool rows16_one_round(const GroupedProblem &problem, unsigned qtype, bool fused, unsigned tokens, uint64_t out_rows);
int launch_rows16_grouped(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, unsigned width,
                          unsigned out_rows, unsigned behind, bool round, double limit, int *status, hipStream_t stream);

static inline bool same_shape(const yvex_hip_expert_weights *a, const yvex_hip_expert_weights *b)
{
    return a->gate_qtype == b->gate_qtype && a->up_qtype == b->up_qtype &&
           a->down_qtype == b->down_qtype && a->hidden == b->hidden &&
           a->intermediate == b->intermediate;
}


}  // namespace yvex
