// MoE routing, expert-major worklist, and the decode-width grouped expert kernels for gfx950.
//
// The grouped kernels walk buckets (one expert plus the ordered (row, rank) pairs routed to it)
// so an expert's packed bytes are streamed from HBM once per bucket and reused for every pair in
// it. Lanes own fixed column ranges of the activation rows and keep them in registers; weight
// rows stream through with unaligned 16-byte loads; integer superblock sums are exact.
//
// Behaviour restated from src/backend/cuda/moe_kernels.cu:180-291 (routing), :294-402
// (worklist), :431-616 (grouped up/down, reduce, combine) and src/graph/moe.c:497-622.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "units.hpp"
#include "grouped.hpp"
#include "q8k.hpp"
#include "route.hpp"
#include "q8_0_rows.hpp"

namespace yvex {

// ---- routing --------------------------------------------------------------------------------

// The scores alone, as the token-local operation publishes them beside the logits
// (src/backend/cuda/moe_kernels.cu:29-55).
__global__ __launch_bounds__(256) void route_scores_kernel(
    const float *__restrict__ logits, unsigned count, int scoring, float *__restrict__ scores, int *status)
{
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= count) return;
    const double s = route_score((double)logits[i], scoring);
    const float published = (float)s;
    if (!(s == s) || !finite_f32(published)) raise_status(status, 1);
    scores[i] = published;
}

__global__ __launch_bounds__(256) void route_rows_kernel(
    const float *__restrict__ logits, const float *__restrict__ bias, unsigned long long rows,
    unsigned experts, unsigned topk, int scoring, int normalize, double scaling,
    unsigned long long *__restrict__ selected, float *__restrict__ weights, int *status)
{
    const unsigned long long row = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (row >= rows) return;
    RouteInputs in;
    route_inputs_load(in, logits, bias, row, threadIdx.x & 63u, experts);
    route_row(in, false, row, threadIdx.x & 63u, experts, topk, scoring, normalize, scaling, selected,
              weights, status);
}

// Hash router (src/backend/cuda/moe_kernels.cu:222-245, src/graph/moe.c:539-582): a row's experts
// are the first topk ordinals of its token's row of an I32 table; weights as for the learned
// router. One wavefront per row, lane r holds rank r. An ordinal outside the expert range, a
// repeated one or a token outside the table is a contract violation (status 2).
__global__ __launch_bounds__(256) void route_hash_rows_kernel(
    const float *__restrict__ logits, const unsigned char *__restrict__ table,
    const unsigned *__restrict__ token_ids, unsigned long long rows, unsigned experts, unsigned topk,
    unsigned long long table_rows, unsigned long long table_row_bytes, int single_row, int scoring,
    int normalize, double scaling, unsigned long long *__restrict__ selected,
    float *__restrict__ weights, int *status)
{
    const unsigned lane = threadIdx.x & 63u;
    const unsigned long long row = (unsigned long long)blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (row >= rows) return;
    const unsigned long long token = token_ids[row];
    if (token >= table_rows) {
        if (lane == 0u) raise_status(status, 2);
        return;
    }
    const int *ordinals = reinterpret_cast<const int *>(table + (single_row ? 0ull : token * table_row_bytes));
    const int mine = lane < topk ? ordinals[lane] : -1;
    const bool live = lane < topk;
    bool bad = live && (mine < 0 || (unsigned)mine >= experts);
    float score = 0.0f;
    if (live && !bad) {
        const double s = route_score((double)logits[row * experts + (unsigned)mine], scoring);
        score = (float)s;
        if (!(s == s) || !finite_f32(score)) raise_status(status, 1);
    }
    double total = 0.0;
    for (unsigned rank = 0; rank < topk; ++rank) {
        const int other = __shfl(mine, (int)rank, kWave);
        bad |= live && rank < lane && other == mine;
        total += (double)__shfl(score, (int)rank, kWave);      // rank order, in double
    }
    if (bad) raise_status(status, 2);
    if (normalize && !(total > 0.0 && total < 1.0e300)) raise_status(status, 1);
    if (live) {
        double value = (double)score;
        if (normalize) value /= total;
        value *= scaling;
        const float w = (float)value;
        if (!finite_f32(w)) raise_status(status, 1);
        weights[row * topk + lane] = w;
        selected[row * topk + lane] = bad ? 0ull : (unsigned long long)mine;
    }
}

// ---- worklist -------------------------------------------------------------------------------
//
// A row never routes to the same expert twice, so each expert's pairs are a set of rows: one bit
// per (expert, row) in LDS. Bucket order is expert order, order inside a bucket is row order,
// which is exactly the stable counting sort of pairs by expert (src/graph/worklist.c:380-393).

constexpr unsigned kWorklistMaxRows = 4096u;
constexpr uint64_t kWorklistMaxPairs = 0x7fffffffull;    // (counted in 32 bits)

__host__ __device__ constexpr unsigned worklist_pitch(unsigned rows) { return (rows + 31u) / 32u | 1u; }

// The whole worklist by one workgroup of 1024 threads; shared_words is its dynamic LDS (worklist_lds_bytes). `routed`: the
// selections in LDS, from a workgroup that has routed the rows itself and need not wait for its stores to come back.
// LARGE: for more rows than kPrepareMaxRoutedRows. One workgroup's round trips to memory, and its stores of single words, bound it there:
// 16 384 stores that touch a line each are 8 us. So the selections are read once and kept, four threads count an expert's
// words, and the order is put together in LDS (`ordered`, where it fits) and stored in lines. A decode batch
// has no use for that, and its launch fetches every instruction to run it once: 96 rows 6.2 us without, 6.7 with.
// With rows of pairs by a multiplication as well 2048 rows of eight experts 21 -> 15 us, 1111 rows 13 -> 10. (The odd pitch and the counts
// below a word: 2048 rows 39 -> 22 us before, 4096 rows 872 -> 112.)
template <bool LARGE>
__device__ __forceinline__ void worklist_block(
    const unsigned long long *__restrict__ selected, unsigned pairs, unsigned topk,
    unsigned experts, unsigned long long *__restrict__ order,
    unsigned long long *__restrict__ expert_ids, unsigned long long *__restrict__ bucket_offsets,
    unsigned long long *__restrict__ bucket_populations,
    unsigned long long *__restrict__ sweep_offsets, unsigned long long *__restrict__ counts,
    int *status, unsigned *shared_words, bool with_below, bool with_ordered = false, const unsigned *routed = nullptr)
{
    const unsigned rows = pairs / topk;
    // p / topk, exact while p * topk < 2^32 (so for 4096 rows of 256 choices). In place of two divisions a pair: the
    // preparation of 1 / 96 / 333 rows 9.1 / 6.0 / 7.3 -> 8.8 / 5.7 / 6.4 us. More choices a row repeat an expert and are
    // refused below; there a row may come out one too high, and the last one's would be another expert's word of the bitmap.
    const unsigned inverse = topk == 1u ? 0u : 0xffffffffu / topk + 1u;
    auto row_of = [&](unsigned p) { return inverse ? min(__umulhi(p, inverse), rows - 1u) : p; };
    const unsigned words = (rows + 31u) / 32u;            // bitmap words per expert
    const unsigned pitch = worklist_pitch(rows);          // odd: the experts' words in different banks
    unsigned *bitmap = shared_words;                       // [experts][pitch]
    unsigned *population = bitmap + experts * pitch;       // [experts]
    unsigned *offset = population + experts;               // [experts + 1]
    unsigned *slot = offset + experts + 1u;                // [experts] bucket index or ~0
    __shared__ unsigned bad;
    const unsigned tid = threadIdx.x;
    for (unsigned i = tid; i < experts * pitch; i += blockDim.x) bitmap[i] = 0u;
    if (tid == 0u) {
        bad = 0u;
        slot[experts + 1536u] = 0u;   // running maximum of the populations (scan[1536])
    }
    __syncthreads();
    // A thread's first selections in registers (2048 rows of eight experts have sixteen), the others four at a time, twice
    constexpr unsigned kKept = LARGE ? 16u : 0u, kInFlight = 4u, threads = 1024u;
    auto selection = [&](unsigned p) { return routed ? (unsigned long long)routed[p] : selected[p]; };
    auto mark = [&](unsigned p, unsigned e) {
        if (e >= experts) {
            bad = 1u;
            return;
        }
        const unsigned row = row_of(p);
        const unsigned old = atomicOr(&bitmap[e * pitch + (row >> 5)], 1u << (row & 31u));
        if (old & (1u << (row & 31u))) bad = 1u;   // duplicate expert inside one row
    };
    auto expert_of = [](unsigned long long chosen) { return chosen > 0xffffffffull ? 0xffffffffu : (unsigned)chosen; };
    unsigned kept[LARGE ? kKept : 1u];
    if constexpr (LARGE) {
        unsigned long long chosen[kKept];
#pragma unroll
        for (unsigned k = 0; k < kKept; ++k) {
            if ((k / kInFlight * kInFlight) * threads >= pairs) break;
            const unsigned p = tid + k * threads;
            chosen[k] = selection(p < pairs ? p : pairs - 1u);
        }
#pragma unroll
        for (unsigned k = 0; k < kKept; ++k) {
            if ((k / kInFlight * kInFlight) * threads >= pairs) break;
            kept[k] = expert_of(chosen[k]);
            if (tid + k * threads < pairs) mark(tid + k * threads, kept[k]);
        }
    }
    auto each_behind = [&](auto &&with) {
        for (unsigned first = kKept * threads + tid; first < pairs; first += kInFlight * threads) {
            unsigned long long chosen[kInFlight];
#pragma unroll
            for (unsigned k = 0; k < kInFlight; ++k) {
                const unsigned p = first + k * threads;
                chosen[k] = selection(p < pairs ? p : first);
            }
#pragma unroll
            for (unsigned k = 0; k < kInFlight; ++k)
                if (first + k * threads < pairs) with(first + k * threads, expert_of(chosen[k]));
        }
    };
    each_behind(mark);
    __syncthreads();
    // rows below each bitmap word that chose the expert (16 bits: at most 4096 rows), kept when
    // the table fits beside the bitmap
    unsigned short *below = reinterpret_cast<unsigned short *>(slot + experts + 1537u);
    [[maybe_unused]] unsigned short *const ordered = below + experts * words;      // [pairs], behind the table
    if constexpr (LARGE) {
        unsigned *const part = slot + experts + 64u;       // [4][256], in what the scan leaves free
        const unsigned e = tid & 255u, from = words * (tid >> 8) / 4u, to = words * ((tid >> 8) + 1u) / 4u;
        unsigned n = 0u;
        if (e < experts) {
#pragma unroll 4
            for (unsigned w = from; w < to; ++w) n += __popc(bitmap[e * pitch + w]);
            part[tid] = n;
        }
        __syncthreads();
        if (e < experts) {
            unsigned before = 0u;
            for (unsigned other = e; other < tid; other += 256u) before += part[other];
            if (tid >= 768u) population[e] = before + n;
            if (with_below) {
#pragma unroll 4
                for (unsigned w = from; w < to; ++w) {
                    below[w * experts + e] = (unsigned short)before;
                    before += __popc(bitmap[e * pitch + w]);
                }
            }
        }
    } else {
        for (unsigned e = tid; e < experts; e += threads) {
            unsigned n = 0u;
            for (unsigned w = 0; w < words; ++w) {
                if (with_below) below[w * experts + e] = (unsigned short)n;
                n += __popc(bitmap[e * pitch + w]);
            }
            population[e] = n;
        }
    }
    __syncthreads();
    // Inclusive prefix sums over the experts (<= 256: the first four wavefronts) of population,
    // sweep count and occupancy: a scan inside each wavefront, the wavefronts' totals
    // through LDS (one barrier); every expert then publishes its own bucket.
    unsigned *scan = slot + experts;                       // [4][3] wavefront totals; [1536] running maximum
    const unsigned n_mine = tid < experts ? population[tid] : 0u;
    unsigned sum_n = n_mine, sum_sweeps = (n_mine + (unsigned)kPass - 1u) / (unsigned)kPass,
             sum_used = n_mine ? 1u : 0u;
    if (tid < 256u) {
        sum_n = wave_inclusive_sum_u32(sum_n);
        sum_sweeps = wave_inclusive_sum_u32(sum_sweeps);
        sum_used = wave_inclusive_sum_u32(sum_used);
        if ((tid & 63u) == 63u) {
            scan[3u * (tid >> 6)] = sum_n;
            scan[3u * (tid >> 6) + 1u] = sum_sweeps;
            scan[3u * (tid >> 6) + 2u] = sum_used;
        }
    }
    __syncthreads();
    unsigned total_pairs = 0u, total_sweeps = 0u, bucket_count = 0u;
    for (unsigned w = 0; w < 4u; ++w) {
        const unsigned a = scan[3u * w], b = scan[3u * w + 1u], c = scan[3u * w + 2u];
        if (w < (tid >> 6)) {
            sum_n += a;
            sum_sweeps += b;
            sum_used += c;
        }
        total_pairs += a;
        total_sweeps += b;
        bucket_count += c;
    }
    if (tid < experts) {
        const unsigned n = n_mine;
        const unsigned cursor = sum_n - n;
        const unsigned sweeps_before = sum_sweeps - (n + (unsigned)kPass - 1u) / (unsigned)kPass;
        const unsigned bucket = sum_used - (n ? 1u : 0u);
        offset[tid] = cursor;
        if (n) {
            expert_ids[bucket] = tid;
            bucket_offsets[bucket] = cursor;
            bucket_populations[bucket] = n;
            sweep_offsets[bucket] = sweeps_before;
        }
        if (tid >= bucket_count) {                         // unused tail of the bucket arrays
            expert_ids[tid] = 0ull;
            bucket_populations[tid] = 0ull;
            bucket_offsets[tid + 1u] = total_pairs;
            sweep_offsets[tid + 1u] = total_sweeps;
        }
    }
    if (tid == 0u) {
        offset[experts] = total_pairs;
        bucket_offsets[bucket_count] = total_pairs;
        sweep_offsets[bucket_count] = total_sweeps;
        counts[0] = bucket_count;
        counts[2] = total_pairs;
        counts[3] = total_sweeps;
        if (total_pairs != pairs) bad = 1u;
    }
    // largest population: one atomic per wave after a wave-wide maximum
    {
        const unsigned n = wave_max_u32(tid < experts ? population[tid] : 0u);
        if ((tid & 63u) == 0u && tid < 256u) atomicMax(&scan[1536u], n);
    }
    __syncthreads();
    if (tid == 0u) counts[1] = scan[1536u];
    // every pair finds its own place: its bucket's start plus the rows below its own that chose
    // the same expert (pairs of a bucket stay in row order, which is the stable order)
    auto place = [&](unsigned p, unsigned e) {
        if (e >= experts) return;
        const unsigned row = row_of(p), w = row >> 5;
        const unsigned *mine = bitmap + e * pitch;
        unsigned before = __popc(mine[w] & ((1u << (row & 31u)) - 1u));
        if (with_below) before += below[w * experts + e];
        else
            for (unsigned other = 0; other < w; ++other) before += __popc(mine[other]);
        if (LARGE && with_ordered) ordered[offset[e] + before] = (unsigned short)p;
        else order[offset[e] + before] = p;
    };
    if constexpr (LARGE) {
#pragma unroll
        for (unsigned k = 0; k < kKept; ++k) {
            if ((k / kInFlight * kInFlight) * threads >= pairs) break;
            if (tid + k * threads < pairs) place(tid + k * threads, kept[k]);
        }
    }
    each_behind(place);
    if (LARGE && with_ordered) {
        __syncthreads();
        // (a batch that is refused below leaves places unwritten: every pair number is one all the same)
        for (unsigned at = tid; at < pairs; at += threads) order[at] = ordered[at] < pairs ? ordered[at] : 0u;
    }
    __syncthreads();
    if (tid == 0u && bad) raise_status(status, 2);
}

__global__ __launch_bounds__(1024) void worklist_kernel(
    const unsigned long long *__restrict__ selected, unsigned pairs, unsigned topk,
    unsigned experts, unsigned long long *__restrict__ order,
    unsigned long long *__restrict__ expert_ids, unsigned long long *__restrict__ bucket_offsets,
    unsigned long long *__restrict__ bucket_populations,
    unsigned long long *__restrict__ sweep_offsets, unsigned long long *__restrict__ counts,
    int *status, int with_below)
{
    extern __shared__ unsigned shared_words[];
    worklist_block<false>(selected, pairs, topk, experts, order, expert_ids, bucket_offsets, bucket_populations,
                          sweep_offsets, counts, status, shared_words, with_below != 0);
}

// A large batch's worklist by the first workgroup and, beside it, the input rows' Q8_K blocks by the others, four a
// wavefront: neither waits for the other, and the one workgroup takes as long as all the others. (Of the same LDS as the first, one
// a compute unit, so its waves go on from block to block and ask ahead.) In a layer of 7168 columns, eight of 256 experts,
// 2048 rows 21.2 and 13.9 us -> 22.5, 1111 rows 14.0 and 8.6 -> 17.9.
__global__ __launch_bounds__(1024) void worklist_quantize_kernel(
    const unsigned long long *__restrict__ selected, unsigned pairs, unsigned topk,
    unsigned experts, unsigned long long *__restrict__ order,
    unsigned long long *__restrict__ expert_ids, unsigned long long *__restrict__ bucket_offsets,
    unsigned long long *__restrict__ bucket_populations,
    unsigned long long *__restrict__ sweep_offsets, unsigned long long *__restrict__ counts,
    int *status, int with_below, int with_ordered, const float *__restrict__ values, unsigned tasks,
    unsigned char *__restrict__ encoded)
{
    extern __shared__ unsigned shared_words[];
    if (blockIdx.x == 0u) {
        worklist_block<true>(selected, pairs, topk, experts, order, expert_ids, bucket_offsets, bucket_populations,
                             sweep_offsets, counts, status, shared_words, with_below != 0, with_ordered != 0);
        return;
    }
    const unsigned lane = threadIdx.x & 63u, stride = (gridDim.x - 1u) * 64u;
    unsigned task = (blockIdx.x - 1u) * 64u + 4u * (threadIdx.x >> 6) + (lane >> 4);
    float v[4][4], ahead[4][4];
    auto request = [&](unsigned wanted, float (&to)[4][4]) {
        const unsigned held = wanted < tasks ? wanted : tasks - 1u;
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k) __builtin_memcpy(to[k], values + held * 256ull + 4u * (lane & 15u) + 64u * k, 16);
    };
    request(task, v);
    for (unsigned first = (blockIdx.x - 1u) * 64u; first < tasks; first += stride, task += stride) {
        request(task + stride, ahead);
        q8k_quantize_four(v, encoded + (task < tasks ? task : tasks - 1u) * (unsigned long long)kQ8KBytes, lane, task < tasks, status);
#pragma unroll
        for (unsigned k = 0; k < 4u; ++k)
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) v[k][i] = ahead[k][i];
    }
}

// A decode batch's preparation in one launch instead of three: workgroup 0 routes the rows (one
// wavefront a row, sixteen at a time) and then builds the worklist from what it wrote; every
// other workgroup quantizes sixteen Q8_K blocks of the input rows, which depend on neither.
constexpr unsigned kPrepareMaxRows = 128u;
// Rows that are routed already leave the worklist: as long as its bitmap is small enough for the
// quantizing workgroups, which get the same LDS, to share a compute unit.
constexpr unsigned kPrepareMaxRoutedRows = YVEX_HIP_PREPARE_ROUTED_MAX_ROWS;

// T: a decode batch of one or two rows whose shared expert holds Q8_0 matrices takes their products with the input rows
// along (the workgroups behind those that quantize): the routing that the launch waits for occupies one workgroup. One
// row of 4096 columns, two matrices of 2048 rows: 8.4 and 6.7 us for the two launches, 9.6 for this one.
struct PairRows {
    const unsigned char *first, *second;
    unsigned long long row_count, row_bytes;
    float *out_first, *out_second;
};

// ROUTES: from logits or scores; otherwise the router's own launch has routed the rows.
template <int T, bool ROUTES>
__global__ __launch_bounds__(1024) void decode_prepare_kernel(
    const float *__restrict__ logits, const float *__restrict__ bias, unsigned rows, unsigned experts,
    unsigned topk, int scoring, int normalize, double scaling, unsigned long long *selected,
    float *__restrict__ weights, unsigned long long *__restrict__ order,
    unsigned long long *__restrict__ expert_ids, unsigned long long *__restrict__ bucket_offsets,
    unsigned long long *__restrict__ bucket_populations, unsigned long long *__restrict__ sweep_offsets,
    unsigned long long *__restrict__ counts, const float *__restrict__ values, unsigned blocks,
    unsigned long long input_stride, unsigned char *__restrict__ encoded, int *status,
    const float *__restrict__ scores, PairRows pair)
{
    extern __shared__ __align__(16) unsigned shared_words[];
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if constexpr (T != 0) {
        const unsigned before = 1u + (rows * blocks + 15u) / 16u;       // the routing and the quantizing workgroups
        if (blockIdx.x >= before) {
            HoldRows hold{values, input_stride, blocks, rows * blocks, status, {}};
            held_rows<T, 2>(2ull * pair.row_count, blockIdx.x - before, gridDim.x - before, 8u * blocks,
                            reinterpret_cast<unsigned char *>(shared_words),
                            [&](unsigned long long row) {
                                return row < pair.row_count ? pair.first + row * pair.row_bytes
                                                            : pair.second + (row - pair.row_count) * pair.row_bytes;
                            },
                            hold,
                            [&](unsigned in, unsigned long long row, float sum) {
                                if (in >= rows) return;
                                float *const out = row < pair.row_count ? pair.out_first + in * pair.row_count + row
                                                                        : pair.out_second + (in - 1ull) * pair.row_count + row;
                                if (!finite_f32(sum)) raise_status(status, 1);
                                else *out = sum;
                            });
            return;
        }
    }
    if (blockIdx.x != 0u) {
        const unsigned task = (blockIdx.x - 1u) * 16u + wave;
        if (task >= rows * blocks) return;
        const unsigned row = task / blocks, block = task % blocks;
        q8k_quantize_block(values + (unsigned long long)row * input_stride + block * 256u + lane * 4u,
                           encoded + (unsigned long long)task * kQ8KBytes, lane, status);
        return;
    }
    // Sixteen rows at a time: the scores of their experts, a thread each (four double-precision scores a lane of the
    // wavefront that routes the row were a microsecond), then a wavefront a row. 5 rows of 256 experts
    // 12.4 -> 10.3 us; the launch behind a router that routes, without this code, on 32 registers and not 118, 5.9 -> 5.4.
    if constexpr (ROUTES) {
        __shared__ float scored[16u * 256u];
        __shared__ unsigned chosen[kPrepareMaxRows * 16u];
        const float *values_in = scores ? scores : logits;
        for (unsigned base = 0; base < rows; base += 16u) {
            const unsigned here = rows - base < 16u ? rows - base : 16u, row = base + wave;
            RouteInputs inputs;
            route_inputs_load(inputs, values_in, bias, row < rows ? row : rows - 1u, lane, experts);
            if (!scores) {
                for (unsigned i = threadIdx.x; i < here * experts; i += 1024u)
                    scored[i] = (float)route_score((double)logits[(unsigned long long)base * experts + i], scoring);
                __syncthreads();
#pragma unroll
                for (unsigned i = 0; i < 4u; ++i)
                    inputs.value[i] = scored[(wave < here ? wave : 0u) * experts + (lane * 4u + i < experts ? lane * 4u + i : experts - 1u)];
            }
            if (wave < here)
                route_row(inputs, true, row, lane, experts, topk, scoring, normalize, scaling, selected, weights, status,
                          chosen + row * topk);
            __syncthreads();   // the selections are read by other waves below, the scores overwritten
        }
        worklist_block<false>(selected, rows * topk, topk, experts, order, expert_ids, bucket_offsets, bucket_populations,
                       sweep_offsets, counts, status, shared_words, true, false, chosen);
        return;
    }
    worklist_block<false>(selected, rows * topk, topk, experts, order, expert_ids, bucket_offsets,
                   bucket_populations, sweep_offsets, counts, status, shared_words, true);
}

// ---- grouped expert projections ---------------------------------------------------------------
//
// Persistent kernel: one 512-thread workgroup per compute unit builds the conflict-free lookup
// tables once, then each of its waves walks a strided list of work items. An item is
// (bucket, tile of weight rows, sweep): a bucket's expert bytes stream from HBM once per sweep
// and every sweep serves up to kPass pairs of the bucket.

constexpr int kRowsInFlight = 1;  // weight-row groups a wave decodes back to back
constexpr int kGroupedThreads = 512;     // two waves per SIMD: with three, a sweep's activation columns spill out of 168 registers
constexpr int kGroupedWaves = kGroupedThreads / 64;
constexpr unsigned kItemRowsMax = 16u;   // gate/up row pairs per item when the SwiGLU is fused

struct LaneGeometry {
    unsigned rows_per_wave, reduce_width, sub, seg, unit0, super;
    bool lane_live;
    unsigned wave;
};

// One sweep of a wave over the item's weight rows [row_begin, row_end) with N live pairs.
// Each iteration handles kRows row groups; the packed bytes of the next iteration are requested
// before the current one is decoded, so HBM latency hides behind the decode.
template <unsigned QT, bool Q8, bool FUSED_UP, int N, typename Tables>
__device__ __forceinline__ void grouped_sweep(
    const GroupedArgs &a, const GroupedProblem &pr, const Tables &tables, const LaneGeometry &g,
    const unsigned char *gate_e, const unsigned char *up_e, unsigned long long first_ordered,
    unsigned row_begin, unsigned row_end, float *park, float *terms)
{
    constexpr int kStreams = FUSED_UP ? 2 : 1;
    constexpr int kRows = Q8 ? kRowsInFlight : 1;
    // ---- the sweep's activation rows: this lane's 128 columns stay in registers (Q8_K) ----
    unsigned act[N][Q8 ? kUnitsPerLane * 8 : 1];
    float act_scale[N];
    int act_bsum[N][(QT == QT_Q4_K || QT == QT_Q2_K) ? 8 : 1];
    const unsigned char *act_row[N];
    float route_weight[N];
    unsigned long long out_index[N];
#pragma unroll
    for (int p = 0; p < N; ++p) {
        const unsigned long long ordered = first_ordered + p;
        const unsigned long long source = pr.order ? pr.order[ordered] : ordered;
        const unsigned long long arow = pr.act_by_ordered_pair ? ordered : source / pr.topk;
        act_row[p] = (const unsigned char *)pr.activations + arow * pr.act_stride;
        route_weight[p] = pr.route_weights ? pr.route_weights[source] : 1.0f;
        out_index[p] = pr.out_by_source_pair ? source : ordered;
        act_scale[p] = 0.0f;
        if constexpr (Q8) {
            const unsigned char *blk = act_row[p] + (unsigned long long)g.super * kQ8KBytes;
            act_scale[p] = *reinterpret_cast<const float *>(blk);
            const unsigned char *q = blk + 4u + 32u * (g.unit0 & 7u);   // 4-byte aligned payload
#pragma unroll
            for (int k = 0; k < kUnitsPerLane * 2; ++k) {
                uint4 v;
                __builtin_memcpy(&v, q + 16 * k, 16);
                act[p][4 * k] = v.x;
                act[p][4 * k + 1] = v.y;
                act[p][4 * k + 2] = v.z;
                act[p][4 * k + 3] = v.w;
            }
            if constexpr (QT == QT_Q4_K || QT == QT_Q2_K) {
                const short *bs = reinterpret_cast<const short *>(blk + 260u) + 2u * (g.unit0 & 7u);
#pragma unroll
                for (int i = 0; i < 8; ++i) act_bsum[p][i] = bs[i];
            }
        }
    }

    const unsigned stride = kRows * g.rows_per_wave;
    LaneChunk<QT> next[kRows][kStreams];
    auto request = [&](unsigned base) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const unsigned want = base + r * g.rows_per_wave + g.sub;
            const unsigned safe_row = (g.lane_live && want < row_end) ? want : row_begin;
            next[r][0].load(gate_e + (unsigned long long)safe_row * pr.row_bytes, g.unit0);
            if constexpr (FUSED_UP)
                next[r][1].load(up_e + (unsigned long long)safe_row * pr.up_row_bytes, g.unit0);
        }
    };
    request(row_begin);

    for (unsigned base = row_begin; base < row_end; base += stride) {
        LaneChunk<QT> chunk[kRows][kStreams];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int w = 0; w < kStreams; ++w) chunk[r][w] = next[r][w];
        if (base + stride < row_end) request(base + stride);

        float sums[kRows][kStreams][N];
        double wide[Q8 ? 1 : kRows][Q8 ? 1 : kStreams][Q8 ? 1 : N];   // F32 activations: the lane's sums in double
        unsigned row[kRows];
        bool row_live[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            row[r] = base + r * g.rows_per_wave + g.sub;
            row_live[r] = g.lane_live && row[r] < row_end;
#pragma unroll
            for (int w = 0; w < kStreams; ++w) {
                const LaneChunk<QT> &c = chunk[r][w];
                int whole_dot[N], whole_min[N];
                int unit_dots[N][UnitTraits<QT>::kIntegerCombine ? 1 : kUnitsPerLane];   // Q8_0: a dot per 32-value block
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    whole_dot[p] = whole_min[p] = 0;
                    sums[r][w][p] = 0.0f;
                    if constexpr (!Q8) wide[r][w][p] = 0.0;
                }
#pragma unroll
                for (int k = 0; k < kUnitsPerLane; ++k) {
                    Unit unit;
                    c.decode(tables, k, g.unit0, unit);
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        if constexpr (Q8) {
                            const unsigned *av = &act[p][8 * k];
                            int d = 0, d2 = 0;
                            if constexpr (QT == QT_Q2_K) {
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    d = dot4(unit.w[i], av[i], d);
                                    d2 = dot4(unit.w[4 + i], av[4 + i], d2);
                                }
                                d = __mul24(unit.factor, d) + __mul24(unit.factor2, d2);
                            } else {
#pragma unroll
                                for (int i = 0; i < 8; ++i) d = dot4(unit.w[i], av[i], d);
                                if constexpr (QT != QT_Q8_0) d = __mul24(d, unit.factor);
                            }
                            if constexpr (UnitTraits<QT>::kIntegerCombine) {
                                whole_dot[p] += d;
                                if constexpr (QT == QT_Q4_K || QT == QT_Q2_K)
                                    whole_min[p] += unit.min1 * act_bsum[p][2 * k] +
                                                    unit.min2 * act_bsum[p][2 * k + 1];
                            } else {
                                unit_dots[p][k] = d;
                            }
                        } else {
                            const float *x = reinterpret_cast<const float *>(act_row[p]) +
                                             32ull * (g.unit0 + k);
                            wide[r][w][p] = chunk_unit_dot_f64<QT>(c, k, unit, x, wide[r][w][p]);
                        }
                    }
                }
                if constexpr (Q8 && UnitTraits<QT>::kIntegerCombine) {
                    // two neighbouring lanes hold the halves of one superblock: finish the exact
                    // integer sum; both compute the float value, the odd lane contributes zero
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        UnitSum t;
                        t.dot = group_sum_i32<2>(whole_dot[p]);
                        t.min = 0;
                        if constexpr (QT != QT_IQ2_XXS) t.min = group_sum_i32<2>(whole_min[p]);
                        const float v = c.combine(act_scale[p], t);
                        sums[r][w][p] = (g.seg & 1u) ? 0.0f : v;
                    }
                }
                if constexpr (Q8 && !UnitTraits<QT>::kIntegerCombine) {
                    // Q8_0: the term of a Q8_K block is one chain of eight fused multiply-adds over
                    // its eight 32-value blocks (kernel_primitives.h:342-359). The even lane of the
                    // pair runs the first four links, the odd lane goes on from there and holds the
                    // block's term.
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        float total = 0.0f;
#pragma unroll
                        for (int k = 0; k < kUnitsPerLane; ++k)
                            total = __builtin_fmaf(c.unit_scale(k) * act_scale[p], (float)unit_dots[p][k], total);
                        float carried = dpp_move_f32<0xa0, 0xf>(total);     // quad_perm [0,0,2,2]: the even neighbour's
#pragma unroll
                        for (int k = 0; k < kUnitsPerLane; ++k)
                            carried = __builtin_fmaf(c.unit_scale(k) * act_scale[p], (float)unit_dots[p][k], carried);
                        sums[r][w][p] = (g.seg & 1u) ? carried : 0.0f;
                    }
                }
            }
        }
        // ---- sum across the lanes of each row, then publish ----
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            if constexpr (Q8) {
                // One float term per superblock sits in a lane of its pair (the even one; Q8_0: the
                // odd one). The row's first lane adds them in double, in superblock order, and
                // rounds once: the row dot of the CPU path (src/gguf/quant_compute.c:152-172 adds a
                // row's blocks in double).
                const unsigned lane = threadIdx.x & 63u;
                constexpr unsigned kTermLane = UnitTraits<QT>::kIntegerCombine ? 0u : 1u;
                const unsigned blocks = a.width >> 8;
#pragma unroll
                for (int w = 0; w < kStreams; ++w)
#pragma unroll
                    for (int p = 0; p < N; ++p)
                        terms[(w * N + p) * 64 + lane] = row_live[r] ? sums[r][w][p] : 0.0f;
                wave_lds_fence();
                if (row_live[r] && g.seg == 0u) {
#pragma unroll
                    for (int w = 0; w < kStreams; ++w)
#pragma unroll
                        for (int p = 0; p < N; ++p) {
                            double sum = 0.0;
                            for (unsigned k = 0; k < blocks; ++k)
                                sum += (double)terms[(w * N + p) * 64 + lane + 2u * k + kTermLane];
                            sums[r][w][p] = (float)sum;
                        }
                }
                wave_lds_fence();
            } else {
                // F32 activations: the lanes' double sums added in double, rounded once
                // (the CPU row dot: src/gguf/quant_compute.c:152-172)
#pragma unroll
                for (int w = 0; w < kStreams; ++w)
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        double sum = row_live[r] ? wide[r][w][p] : 0.0;
                        for (unsigned offset = g.reduce_width >> 1; offset; offset >>= 1)
                            sum += __shfl_xor(sum, (int)offset, kWave);
                        sums[r][w][p] = (float)sum;
                    }
            }
            if constexpr (FUSED_UP) {
                // park (gate, up); the SwiGLU runs once per item with every lane busy
                const unsigned local = row[r] - row_begin;
                if (row_live[r] && g.seg == 0u && local < kItemRowsMax) {
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        park[(0u * kItemRowsMax + local) * kPass + p] = sums[r][0][p];
                        park[(1u * kItemRowsMax + local) * kPass + p] = sums[r][1][p];
                    }
                }
            } else if (row_live[r] && g.seg == 0u) {
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    const float value = bf16_round(sums[r][0][p]);
                    if (!finite_f32(value)) raise_status(a.status, 1);
                    else pr.out[out_index[p] * a.out_rows + row[r]] = value;
                }
            }
        }
    }
    if constexpr (FUSED_UP) {
        // LDS operations of one wave complete in order: no barrier between park and read
        const unsigned lane = threadIdx.x & 63u;
        const unsigned local = lane >> 2;
        const int p = (int)(lane & 3u);
        const unsigned out_row = row_begin + local;
        if (local < kItemRowsMax && out_row < row_end && p < N) {
            float rw = route_weight[0];
            unsigned long long oi = out_index[0];
#pragma unroll
            for (int q = 1; q < N; ++q) {
                if (p == q) {
                    rw = route_weight[q];
                    oi = out_index[q];
                }
            }
            const float value = swiglu_bf16(park[(0u * kItemRowsMax + local) * kPass + p],
                                            park[(1u * kItemRowsMax + local) * kPass + p], rw, a.limit);
            if (!finite_f32(value)) raise_status(a.status, 1);
            else pr.out[oi * a.out_rows + out_row] = value;
        }
    }
}

template <unsigned QT>
struct GroupedTables {
    using type = Iq2Tables;   // unused placeholder for qtypes without lookup tables
};
template <>
struct GroupedTables<QT_IQ2_XXS> {
    using type = Iq2TablesWide;
};

template <unsigned QT, bool Q8, bool FUSED_UP>
__global__ __launch_bounds__(kGroupedThreads) void grouped_kernel(GroupedArgs a)
{
    extern __shared__ __align__(16) unsigned char grouped_lds[];
    typename GroupedTables<QT>::type tables;
    unsigned char *after_tables = grouped_lds;
    if constexpr (QT == QT_IQ2_XXS) {
        // the lookups address LDS directly: the dynamic block must start at LDS address 0
        if (lds_address_of(grouped_lds) != 0u) {
            if (threadIdx.x == 0u) raise_status(a.status, 2);
            return;
        }
        tables = iq2_tables_wide_fill(grouped_lds);
        after_tables = grouped_lds + kIq2WideBytes;
        __syncthreads();
    }
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    float *park = reinterpret_cast<float *>(after_tables) + wave * (2u * kItemRowsMax * kPass);
    // per wave: the float terms of an iteration, one word per (stream, pair, lane)
    float *terms = reinterpret_cast<float *>(after_tables) + kGroupedWaves * (2u * kItemRowsMax * kPass) +
                   wave * (2u * kPass * 64u);

    const unsigned units = a.width >> 5;                          // multiple of 8
    const unsigned lanes_per_row = units / kUnitsPerLane;         // even, <= 64
    const bool pow2 = (lanes_per_row & (lanes_per_row - 1u)) == 0u;
    LaneGeometry g;
    g.rows_per_wave = pow2 ? 64u / lanes_per_row : 1u;
    g.reduce_width = pow2 ? lanes_per_row : 64u;
    g.sub = lane / lanes_per_row;
    g.seg = lane % lanes_per_row;
    g.lane_live = g.sub < g.rows_per_wave;
    g.unit0 = g.seg * kUnitsPerLane;                              // four units, one superblock
    g.super = g.unit0 >> 3;
    g.wave = wave;

    const unsigned tiles = (a.out_rows + a.item_rows - 1u) / a.item_rows;
    const unsigned long long wave_id = (unsigned long long)blockIdx.x * kGroupedWaves + wave;
    const unsigned long long wave_count = (unsigned long long)gridDim.x * kGroupedWaves;

    // The shared expert's items come first (their number is known at launch), then the routed
    // buckets the device-built worklist reports.
    for (int which = (int)a.problems - 1; which >= 0; --which) {
        const GroupedProblem &pr = a.problem[which];
        const bool fixed = pr.expert_ids == nullptr;
        // a work item is one sweep over one tile; sweeps are numbered across all buckets
        const unsigned long long buckets = fixed ? 1ull : pr.counts[0];
        const unsigned long long sweeps = fixed ? pr.sweeps : pr.counts[3];
        const unsigned long long items = sweeps * tiles;
        // stagger the second list so the waves that ran short on the first start it
        const unsigned long long shift = which == 0 && a.problems > 1
            ? ((unsigned long long)tiles * a.problem[1].sweeps) % wave_count : 0ull;
        unsigned long long item = (wave_id + wave_count - shift) % wave_count;
        for (; item < items; item += wave_count) {
            // Items of one bucket are contiguous and, inside a bucket, the sweeps over one tile
            // are neighbours: neighbouring waves stream the same bytes at the same time, so only
            // the first of them goes to HBM.
            unsigned long long expert = 0ull, first = 0ull, population = pr.pairs;
            unsigned long long local = item, bucket_sweeps = sweeps;
            if (!fixed) {
                // last bucket whose first item is <= item
                unsigned long long low = 0ull, high = buckets;
                while (low + 1ull < high) {
                    const unsigned long long middle = (low + high) >> 1;
                    if (pr.sweep_offsets[middle] * tiles <= item) low = middle;
                    else high = middle;
                }
                expert = pr.expert_ids[low];
                first = pr.bucket_offsets[low];
                population = pr.bucket_populations[low];
                local = item - pr.sweep_offsets[low] * tiles;
                bucket_sweeps = pr.sweep_offsets[low + 1ull] - pr.sweep_offsets[low];
            }
            if (bucket_sweeps == 0ull) {
                if (lane == 0u) raise_status(a.status, 2);
                continue;
            }
            const unsigned tile = (unsigned)(local / bucket_sweeps);
            const unsigned long long pass = (local % bucket_sweeps) * kPass;
            if (expert >= pr.experts || first + population > pr.pairs || pass >= population ||
                tile >= tiles) {
                if (lane == 0u) raise_status(a.status, 2);
                continue;
            }
            const unsigned char *gate_e = pr.gate + expert * pr.expert_bytes;
            const unsigned char *up_e = FUSED_UP ? pr.up + expert * pr.up_expert_bytes : nullptr;
            const unsigned row_begin = tile * a.item_rows;
            const unsigned row_end = row_begin + a.item_rows < a.out_rows ? row_begin + a.item_rows
                                                                          : a.out_rows;
            if (population - pass >= 2ull)
                grouped_sweep<QT, Q8, FUSED_UP, 2>(a, pr, tables, g, gate_e, up_e, first + pass,
                                                   row_begin, row_end, park, terms);
            else
                grouped_sweep<QT, Q8, FUSED_UP, 1>(a, pr, tables, g, gate_e, up_e, first + pass,
                                                   row_begin, row_end, park, terms);
        }
    }
}

// LANES columns per thread (4 when the width allows 16-byte accesses); each column's sum runs in
// rank order, so the result does not depend on LANES. The memory bounds it (a pair's outputs are read once and from there); a workgroup's
// place is its block numbers (a row's and a column's number by 64-bit division were what a thread did first, for as long
// as its loads took), and up to eight ranks' loads are in flight with the shared row's. Eight ranks of 7168 columns by 2048 rows
// 107 -> 88 us (6.7 TB/s), 1111 rows 55.6 -> 52, up to 100 rows level (a branch a rank around its load: 1 us more of five rows). STREAMING: kReduceStreaming.
template <int LANES, bool STREAMING>
__global__ __launch_bounds__(256) void reduce_combine_kernel(
    const float *__restrict__ pair_outputs, unsigned long long rows, unsigned topk,
    unsigned long long hidden, const float *__restrict__ shared, float *__restrict__ routed,
    float *__restrict__ combined, int *status)
{
    typedef float Pack __attribute__((ext_vector_type(LANES)));
    for (unsigned long long row = blockIdx.y; row < rows; row += gridDim.y) {
        for (unsigned long long column = (blockIdx.x * 256ull + threadIdx.x) * LANES; column < hidden; column += gridDim.x * 256ull * LANES) {
            const unsigned long long index = row * hidden + column;
            const float *source = pair_outputs + row * topk * hidden + column;
            Pack total, base;
#pragma unroll
            for (int i = 0; i < LANES; ++i) total[i] = base[i] = 0.0f;
            if (combined && shared) base = *reinterpret_cast<const Pack *>(shared + index);
            auto ranks = [&](auto batch, unsigned live) {       // (those behind the last repeat it, unused)
                constexpr unsigned kBatch = decltype(batch)::value;
                Pack part[kBatch];
#pragma unroll
                for (unsigned k = 0; k < kBatch; ++k) {
                    const Pack *const from = reinterpret_cast<const Pack *>(source + (k < live ? k : live - 1u) * hidden);
                    part[k] = STREAMING ? __builtin_nontemporal_load(from) : *from;
                }
#pragma unroll
                for (unsigned k = 0; k < kBatch; ++k) {
                    if (k >= live) break;
#pragma unroll
                    for (int i = 0; i < LANES; ++i) total[i] += part[k][i];
                }
                source += kBatch * hidden;
            };
            unsigned left = topk;
            for (; left >= 8u; left -= 8u) ranks(std::integral_constant<unsigned, 8u>{}, 8u);
            if (left >= 4u) ranks(std::integral_constant<unsigned, 4u>{}, 4u), left -= 4u;
            if (left) ranks(std::integral_constant<unsigned, 3u>{}, left);
            bool good = true;
#pragma unroll
            for (int i = 0; i < LANES; ++i) good = good && finite_f32(total[i]);
            if (!good) {
                raise_status(status, 1);
                continue;
            }
            if (routed) *reinterpret_cast<Pack *>(routed + index) = total;
            if (combined && shared) {
                Pack value;
#pragma unroll
                for (int i = 0; i < LANES; ++i) {
                    value[i] = bf16_round(total[i] + base[i]);
                    good = good && finite_f32(value[i]);
                }
                if (!good) raise_status(status, 1);
                else *reinterpret_cast<Pack *>(combined + index) = value;
            }
        }
    }
}

template <unsigned QT, bool Q8, bool FUSED>
static int launch_grouped_variant(const GroupedArgs &a, hipStream_t stream)
{
    const size_t lds = (QT == QT_IQ2_XXS ? kIq2WideBytes : 0u) +
                       (size_t)kGroupedWaves * 2u * kItemRowsMax * kPass * sizeof(float) +
                       (size_t)kGroupedWaves * 2u * kPass * 64u * sizeof(float);
    YVEX_ALLOW_DYNAMIC_LDS((grouped_kernel<QT, Q8, FUSED>), lds);
    grouped_kernel<QT, Q8, FUSED><<<compute_units(), kGroupedThreads, lds, stream>>>(a);
    return check_launch("moe_grouped");
}

template <unsigned QT>
static int launch_grouped(const GroupedArgs &a, bool q8, bool fused, hipStream_t stream)
{
    if (fused) return q8 ? launch_grouped_variant<QT, true, true>(a, stream)
                         : launch_grouped_variant<QT, false, true>(a, stream);
    return q8 ? launch_grouped_variant<QT, true, false>(a, stream)
              : launch_grouped_variant<QT, false, false>(a, stream);
}

static int dispatch_grouped(unsigned qtype, const GroupedArgs &a, bool q8, bool fused,
                            hipStream_t stream)
{
    bool aligned = true;   // the specialised sweeps load dwords: bases and strides must allow it
    for (unsigned i = 0; i < a.problems; ++i) {
        const GroupedProblem &pr = a.problem[i];
        aligned = aligned && ((uintptr_t)pr.gate % 4u == 0u) && pr.expert_bytes % 4u == 0u &&
                  (!pr.up || ((uintptr_t)pr.up % 4u == 0u && pr.up_expert_bytes % 4u == 0u));
    }
    unsigned long long all_pairs = 0ull;
    for (unsigned i = 0; i < a.problems; ++i) all_pairs += a.problem[i].pairs;
    // (Q2_K rows have the sweeps for a plain projection, the down experts, only)
    if (q8 && aligned && !(qtype == QT_Q2_K && fused) &&
        iq2_sweep_supported(qtype, a.width, a.out_rows, all_pairs, a.image != 0))
        return launch_iq2_sweep(a, qtype, fused, a.image != 0, stream);
    if (a.image) return ST_UNSUPPORTED;      // only the specialised sweeps read the image
    switch (qtype) {
    case QT_IQ2_XXS: return launch_grouped<QT_IQ2_XXS>(a, q8, fused, stream);
    case QT_Q4_K: return launch_grouped<QT_Q4_K>(a, q8, fused, stream);
    case QT_Q8_0: return launch_grouped<QT_Q8_0>(a, q8, fused, stream);
    case QT_Q2_K: return launch_grouped<QT_Q2_K>(a, q8, fused, stream);
    default: return ST_UNSUPPORTED;
    }
}

}  // namespace yvex

using namespace yvex;

extern "C" int yvex_hip_moe_route_rows(const float *logits, const float *bias, uint64_t rows,
                                       uint64_t experts, uint64_t topk, int scoring,
                                       int normalize, double scaling, uint64_t *selected,
                                       float *weights, int *status, yvex_hip_stream stream)
{
    if (!logits || !selected || !weights || !status || !rows || !experts || experts > 256u ||
        !topk || topk > 16u || topk > experts ||
        (scoring != YVEX_HIP_SCORING_SQRT_SOFTPLUS && scoring != YVEX_HIP_SCORING_SIGMOID))
        return ST_INVALID_ARG;
    const uint64_t grid = (rows + 3u) / 4u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    route_rows_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        logits, bias, rows, (unsigned)experts, (unsigned)topk, scoring, normalize, scaling,
        (unsigned long long *)selected, weights, status);
    return check_launch("moe_route_rows");
}

extern "C" int yvex_hip_moe_route_hash_rows(const float *logits, const uint8_t *table,
                                            const uint32_t *token_ids, uint64_t rows,
                                            uint64_t experts, uint64_t topk, uint64_t table_rows,
                                            uint64_t table_row_bytes, int single_row, int scoring,
                                            int normalize,
                                            double scaling, uint64_t *selected, float *weights,
                                            int *status, yvex_hip_stream stream)
{
    if (!logits || !table || !token_ids || !selected || !weights || !status || !rows || !experts ||
        experts > 256u || !topk || topk > 16u || topk > experts || !table_rows ||
        ((uintptr_t)table & 3u) ||
        (scoring != YVEX_HIP_SCORING_SQRT_SOFTPLUS && scoring != YVEX_HIP_SCORING_SIGMOID))
        return ST_INVALID_ARG;
    if (table_row_bytes < topk * 4u || (table_row_bytes & 3u)) return ST_BOUNDS;
    const uint64_t grid = (rows + 3u) / 4u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    route_hash_rows_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(
        logits, table, token_ids, rows, (unsigned)experts, (unsigned)topk, table_rows, table_row_bytes,
        single_row, scoring, normalize, scaling, (unsigned long long *)selected, weights, status);
    return check_launch("moe_route_hash_rows");
}

extern "C" int yvex_hip_moe_route_scores(const float *logits, uint64_t count, int scoring,
                                         float *scores, int *status, yvex_hip_stream stream)
{
    if (!logits || !scores || !status || !count || count > 0x7fffffffull ||
        (scoring != YVEX_HIP_SCORING_SQRT_SOFTPLUS && scoring != YVEX_HIP_SCORING_SIGMOID))
        return ST_INVALID_ARG;
    route_scores_kernel<<<(unsigned)((count + 255u) / 256u), 256, 0, as_stream(stream)>>>(
        logits, (unsigned)count, scoring, scores, status);
    return check_launch("moe_route_scores");
}

constexpr size_t kWorklistLdsLimit = 160u * 1024u - 64u;

// Dynamic LDS of the worklist workgroup; *with_below says whether the 16-bit table of rows below
// each bitmap word fits as well.
static size_t worklist_lds_bytes(uint64_t experts, uint64_t rows, int *with_below)
{
    const uint64_t words = (rows + 31u) / 32u;
    const size_t base = (size_t)(experts * worklist_pitch((unsigned)rows) + 3u * experts + 1u + 1537u) * sizeof(unsigned);
    const size_t table = (size_t)(experts * words) * sizeof(unsigned short);
    *with_below = base + table <= kWorklistLdsLimit;
    return *with_below ? base + table : base;
}

extern "C" int yvex_hip_worklist_build(const uint64_t *selected, uint64_t pairs, uint64_t topk,
                                       uint64_t experts, uint64_t *order, uint64_t *expert_ids,
                                       uint64_t *bucket_offsets, uint64_t *bucket_populations,
                                       uint64_t *sweep_offsets, uint64_t *counts, int *status,
                                       yvex_hip_stream stream)
{
    if (!selected || !order || !expert_ids || !bucket_offsets || !bucket_populations ||
        !sweep_offsets || !counts ||
        !status || !pairs || !topk || !experts || experts > 256u || pairs % topk)
        return ST_INVALID_ARG;
    const uint64_t rows = pairs / topk;
    if (rows > kWorklistMaxRows || pairs > kWorklistMaxPairs) return ST_BOUNDS;
    int with_below = 0;
    const size_t lds = worklist_lds_bytes(experts, rows, &with_below);
    YVEX_ALLOW_DYNAMIC_LDS(worklist_kernel, kWorklistLdsLimit);
    if (lds > kWorklistLdsLimit) return ST_BOUNDS;
    worklist_kernel<<<1, 1024, lds, as_stream(stream)>>>(
        (const unsigned long long *)selected, (unsigned)pairs, (unsigned)topk, (unsigned)experts,
        (unsigned long long *)order, (unsigned long long *)expert_ids,
        (unsigned long long *)bucket_offsets, (unsigned long long *)bucket_populations,
        (unsigned long long *)sweep_offsets, (unsigned long long *)counts, status, with_below);
    return check_launch("worklist_build");
}

extern "C" int yvex_hip_worklist_quantize(const uint64_t *selected, uint64_t pairs, uint64_t topk, uint64_t experts,
                                          uint64_t *order, uint64_t *expert_ids, uint64_t *bucket_offsets,
                                          uint64_t *bucket_populations, uint64_t *sweep_offsets, uint64_t *counts,
                                          const float *values, uint64_t width, uint8_t *encoded, int *status,
                                          yvex_hip_stream stream)
{
    if (!selected || !order || !expert_ids || !bucket_offsets || !bucket_populations || !sweep_offsets || !counts ||
        !status || !pairs || !topk || !experts || experts > 256u || pairs % topk || !values || !encoded || !width || width % 256u ||
        (((uintptr_t)values | (uintptr_t)encoded) & 3u))
        return ST_INVALID_ARG;
    const uint64_t rows = pairs / topk, blocks = width / 256u, tasks = rows * blocks;
    if (rows > kWorklistMaxRows || pairs > kWorklistMaxPairs || blocks > 0x7fffffffull || tasks > 0x7fffffffull) return ST_BOUNDS;
    int with_below = 0;
    size_t lds = worklist_lds_bytes(experts, rows, &with_below);
    if (lds > kWorklistLdsLimit) return ST_BOUNDS;
    const bool with_ordered = with_below && pairs <= 65536u && lds + pairs * sizeof(unsigned short) <= kWorklistLdsLimit;
    if (with_ordered) lds += pairs * sizeof(unsigned short);
    YVEX_ALLOW_DYNAMIC_LDS(worklist_quantize_kernel, kWorklistLdsLimit);
    const uint64_t groups = (tasks + 63u) / 64u, others = compute_units() > 1 ? (uint64_t)compute_units() - 1u : 1u;
    worklist_quantize_kernel<<<1u + (unsigned)(groups < others ? groups : others), 1024, lds, as_stream(stream)>>>(
        (const unsigned long long *)selected, (unsigned)pairs, (unsigned)topk, (unsigned)experts,
        (unsigned long long *)order, (unsigned long long *)expert_ids, (unsigned long long *)bucket_offsets,
        (unsigned long long *)bucket_populations, (unsigned long long *)sweep_offsets, (unsigned long long *)counts, status,
        with_below, with_ordered, values, (unsigned)tasks, encoded);
    return check_launch("worklist_quantize");
}

extern "C" int yvex_hip_moe_prepare_supported(uint64_t rows, uint64_t experts, uint64_t topk)
{
    return rows != 0u && rows <= kPrepareMaxRows && experts != 0u && experts <= 256u && topk != 0u &&
           topk <= experts && topk <= 16u;
}

// (a workgroup holds the rows' blocks in LDS, a wave quantizes one after another)
extern "C" int yvex_hip_moe_prepare_projecting_supported(const yvex_hip_projection_pair *pair, uint64_t rows, uint64_t width)
{
    return pair && pair->first && pair->second && !(((uintptr_t)pair->first | (uintptr_t)pair->second) & 1u) && rows &&
           rows <= 2u && width && width % 256u == 0u && width <= 14336u && rows * (width / 256u) <= 56u &&
           pair->row_bytes == width / 32u * 34u && pair->row_count && pair->row_count <= 0xffffffffull;
}

static int launch_moe_prepare(const float *logits, const float *scores, const float *bias, uint64_t rows,
                              uint64_t experts, uint64_t topk, int scoring, int normalize, double scaling,
                              uint64_t *selected, float *weights, uint64_t *order, uint64_t *expert_ids,
                              uint64_t *bucket_offsets, uint64_t *bucket_populations, uint64_t *sweep_offsets,
                              uint64_t *counts, const float *values, uint64_t width, uint64_t input_stride,
                              uint8_t *encoded, int *status, yvex_hip_stream stream,
                              const yvex_hip_projection_pair *pair = nullptr)
{
    const bool routed = !logits && !scores;
    if (!selected || (!weights && !routed) || !order || !expert_ids || !bucket_offsets ||
        !bucket_populations || !sweep_offsets || !counts || !status || (scoring != 0 && scoring != 1))
        return ST_INVALID_ARG;
    if (routed ? !rows || rows > kPrepareMaxRoutedRows || !experts || experts > 256u || !topk || topk > 16u || topk > experts
               : !yvex_hip_moe_prepare_supported(rows, experts, topk))
        return ST_UNSUPPORTED;
    uint64_t tasks = 0u;
    if (values) {
        if (!encoded || !width || width % 256u || input_stride < width || width / 256u > 0xffffu)
            return ST_INVALID_ARG;
        tasks = rows * (width / 256u);
    }
    int with_below = 0;
    const size_t lds = worklist_lds_bytes(experts, rows, &with_below);   // always fits at these sizes
    if (!with_below) return ST_BOUNDS;
    PairRows projected{};
    unsigned grid = (unsigned)(1u + (tasks + 15u) / 16u);
    size_t lds_here = lds;
    if (pair) {
        if (!tasks || !yvex_hip_moe_prepare_projecting_supported(pair, rows, width)) return ST_UNSUPPORTED;
        if (!pair->out_first || !pair->out_second || (((uintptr_t)pair->out_first | (uintptr_t)pair->out_second) & 3u))
            return ST_INVALID_ARG;
        projected = PairRows{pair->first, pair->second, pair->row_count, pair->row_bytes, pair->out_first, pair->out_second};
        // (one round of workgroups, one a compute unit, with those of the routing and the quantization)
        const uint64_t groups = (2u * pair->row_count + kHeldWaves - 1u) / kHeldWaves, cus = (uint64_t)compute_units();
        const uint64_t most = cus > grid ? cus - grid : 1u;
        grid += (unsigned)(groups < most ? groups : most);
        const size_t held = (size_t)held_bytes(rows, width / 256u);
        if (held > lds_here) lds_here = held;
    }
    const auto kernel = routed ? decode_prepare_kernel<0, false> : !pair ? decode_prepare_kernel<0, true>
                      : rows == 1u ? decode_prepare_kernel<1, true> : decode_prepare_kernel<2, true>;
    kernel<<<grid, 1024, lds_here, as_stream(stream)>>>(
        logits, bias, (unsigned)rows, (unsigned)experts, (unsigned)topk, scoring, normalize, scaling,
        (unsigned long long *)selected, weights, (unsigned long long *)order,
        (unsigned long long *)expert_ids, (unsigned long long *)bucket_offsets,
        (unsigned long long *)bucket_populations, (unsigned long long *)sweep_offsets,
        (unsigned long long *)counts, values, (unsigned)(width / 256u), input_stride, encoded, status, scores, projected);
    return check_launch("moe_prepare");
}

extern "C" int yvex_hip_moe_prepare(const float *logits, const float *bias, uint64_t rows, uint64_t experts,
                                    uint64_t topk, int scoring, int normalize, double scaling,
                                    uint64_t *selected, float *weights, uint64_t *order,
                                    uint64_t *expert_ids, uint64_t *bucket_offsets,
                                    uint64_t *bucket_populations, uint64_t *sweep_offsets, uint64_t *counts,
                                    const float *values, uint64_t width, uint64_t input_stride,
                                    uint8_t *encoded, int *status, yvex_hip_stream stream)
{
    if (!logits) return ST_INVALID_ARG;
    return launch_moe_prepare(logits, nullptr, bias, rows, experts, topk, scoring, normalize, scaling, selected,
                              weights, order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets,
                              counts, values, width, input_stride, encoded, status, stream);
}

extern "C" int yvex_hip_moe_prepare_projecting(
    const float *logits, const float *bias, uint64_t rows, uint64_t experts, uint64_t topk, int scoring, int normalize,
    double scaling, uint64_t *selected, float *weights, uint64_t *order, uint64_t *expert_ids, uint64_t *bucket_offsets,
    uint64_t *bucket_populations, uint64_t *sweep_offsets, uint64_t *counts, const float *values, uint64_t width,
    uint64_t input_stride, uint8_t *encoded, const yvex_hip_projection_pair *pair, int *status, yvex_hip_stream stream)
{
    if (!logits || !values || !pair) return ST_INVALID_ARG;
    return launch_moe_prepare(logits, nullptr, bias, rows, experts, topk, scoring, normalize, scaling, selected,
                              weights, order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets,
                              counts, values, width, input_stride, encoded, status, stream, pair);
}

extern "C" int yvex_hip_moe_prepare_scored(const float *scores, const float *bias, uint64_t rows,
                                           uint64_t experts, uint64_t topk, int normalize, double scaling,
                                           uint64_t *selected, float *weights, uint64_t *order,
                                           uint64_t *expert_ids, uint64_t *bucket_offsets,
                                           uint64_t *bucket_populations, uint64_t *sweep_offsets,
                                           uint64_t *counts, const float *values, uint64_t width,
                                           uint64_t input_stride, uint8_t *encoded, int *status,
                                           yvex_hip_stream stream)
{
    if (!scores) return ST_INVALID_ARG;
    return launch_moe_prepare(nullptr, scores, bias, rows, experts, topk, 0, normalize, scaling, selected, weights,
                              order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets, counts,
                              values, width, input_stride, encoded, status, stream);
}

extern "C" int yvex_hip_moe_prepare_routed(const uint64_t *selected, uint64_t rows, uint64_t experts, uint64_t topk,
                                           uint64_t *order, uint64_t *expert_ids, uint64_t *bucket_offsets,
                                           uint64_t *bucket_populations, uint64_t *sweep_offsets,
                                           uint64_t *counts, const float *values, uint64_t width,
                                           uint64_t input_stride, uint8_t *encoded, int *status,
                                           yvex_hip_stream stream)
{
    return launch_moe_prepare(nullptr, nullptr, nullptr, rows, experts, topk, 0, 0, 1.0, (uint64_t *)selected, nullptr,
                              order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets, counts,
                              values, width, input_stride, encoded, status, stream);
}

extern "C" int yvex_hip_moe_up(const yvex_hip_expert_weights *w, const void *activations,
                               int act_q8, const float *route_weights, const uint64_t *order,
                               const uint64_t *expert_ids, const uint64_t *bucket_offsets,
                               const uint64_t *bucket_populations, const uint64_t *sweep_offsets,
                               const uint64_t *counts, uint64_t pairs, uint64_t topk,
                               uint64_t experts, double limit,
                               float *intermediate, const yvex_hip_expert_weights *shared,
                               uint64_t shared_rows, float *shared_intermediate, int *status,
                               yvex_hip_stream stream)
{
    if (!w || !w->gate || !w->up || !activations || !intermediate || !status || !pairs || !topk ||
        !experts || !(limit > 0.0) || (act_q8 != 0 && act_q8 != 1) ||
        (expert_ids && (!bucket_offsets || !bucket_populations || !sweep_offsets || !counts)) ||
        (shared && (!shared->gate || !shared->up || !shared_rows || !shared_intermediate)))
        return ST_INVALID_ARG;
    if (w->gate_qtype != w->up_qtype) return ST_UNSUPPORTED;
    int rc = w->gate_up_image
        ? check_image_matrix(w->gate_qtype, w->hidden, w->gate_row_bytes, w->gate, w->gate_expert_bytes)
        : check_matrix(w->gate_qtype, w->hidden, w->gate_row_bytes);
    if (rc) return rc;
    if (w->gate_up_image && (!act_q8 || ((uintptr_t)w->up & 3u) || (w->up_expert_bytes & 3u)))
        return ST_UNSUPPORTED;
    if (w->up_row_bytes != w->gate_row_bytes) return ST_BOUNDS;
    if (pairs > 0xffffffffull || w->intermediate > 0xffffffffull || shared_rows > 0xffffffffull)
        return ST_BOUNDS;
    if (shared && (!same_shape(w, shared) || shared->gate_row_bytes != w->gate_row_bytes ||
                   shared->up_row_bytes != w->up_row_bytes ||
                   (shared->gate_up_image != 0) != (w->gate_up_image != 0)))
        return ST_UNSUPPORTED;   // launch the shared expert on its own instead
    GroupedArgs a{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets, counts};
    fill_up_problem(a.problem[0], w, activations, act_q8, route_weights, wl, pairs, topk, experts,
                    intermediate);
    a.problems = 1u;
    if (shared) {
        const WorklistView none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
        fill_up_problem(a.problem[1], shared, activations, act_q8, nullptr, none, shared_rows, 1u,
                        1u, shared_intermediate);
        a.problems = 2u;
    }
    a.width = (unsigned)w->hidden;
    a.out_rows = (unsigned)w->intermediate;
    a.item_rows = kItemRowsMax;
    a.limit = limit;
    a.status = status;
    a.image = w->gate_up_image != 0;
    return dispatch_grouped(w->gate_qtype, a, act_q8 != 0, true, as_stream(stream));
}

extern "C" int yvex_hip_moe_down(const yvex_hip_expert_weights *w, const void *intermediate,
                                 int act_q8, const uint64_t *order, const uint64_t *expert_ids,
                                 const uint64_t *bucket_offsets,
                                 const uint64_t *bucket_populations, const uint64_t *sweep_offsets,
                                 const uint64_t *counts, uint64_t pairs, uint64_t experts,
                                 float *pair_outputs,
                                 const yvex_hip_expert_weights *shared, uint64_t shared_rows,
                                 const void *shared_intermediate, float *shared_outputs,
                                 int *status, yvex_hip_stream stream)
{
    if (!w || !w->down || !intermediate || !pair_outputs || !status || !pairs || !experts ||
        (act_q8 != 0 && act_q8 != 1) ||
        (expert_ids && (!bucket_offsets || !bucket_populations || !sweep_offsets || !counts)) ||
        (shared && (!shared->down || !shared_rows || !shared_intermediate || !shared_outputs)))
        return ST_INVALID_ARG;
    int rc = w->down_image
        ? check_image_matrix(w->down_qtype, w->intermediate, w->down_row_bytes, w->down, w->down_expert_bytes)
        : check_matrix(w->down_qtype, w->intermediate, w->down_row_bytes);
    if (rc) return rc;
    if (w->down_image && !act_q8) return ST_UNSUPPORTED;
    if (pairs > 0xffffffffull || w->hidden > 0xffffffffull || shared_rows > 0xffffffffull)
        return ST_BOUNDS;
    if (shared && (!same_shape(w, shared) || shared->down_row_bytes != w->down_row_bytes ||
                   (shared->down_image != 0) != (w->down_image != 0)))
        return ST_UNSUPPORTED;
    GroupedArgs a{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, sweep_offsets, counts};
    fill_down_problem(a.problem[0], w, intermediate, act_q8, wl, pairs, experts, pair_outputs);
    a.problems = 1u;
    if (shared) {
        const WorklistView none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
        fill_down_problem(a.problem[1], shared, shared_intermediate, act_q8, none, shared_rows, 1u,
                          shared_outputs);
        a.problems = 2u;
    }
    a.width = (unsigned)w->intermediate;
    a.out_rows = (unsigned)w->hidden;
    a.item_rows = 64u;
    a.limit = 1.0;
    a.status = status;
    a.image = w->down_image != 0;
    return dispatch_grouped(w->down_qtype, a, act_q8 != 0, false, as_stream(stream));
}

// The clamped SiLU-gated products of given gate and up sums (src/graph/moe.c:605-611), rounded
// to bfloat16 as the fused kernels round them; out may be either input.
__global__ __launch_bounds__(256) void swiglu_rows_kernel(const float *gate, const float *up,
                                                          unsigned long long count, double limit, float *out,
                                                          int *status)
{
    const unsigned long long at = (unsigned long long)blockIdx.x * 256ull + threadIdx.x;
    if (at >= count) return;
    const float value = swiglu_bf16_fast(gate[at], up[at], 1.0f, limit, (float)limit);
    if (!finite_f32(value)) raise_status(status, 1);
    else out[at] = value;
}

extern "C" int yvex_hip_moe_swiglu_rows(const float *gate, const float *up, uint64_t count, double limit,
                                        float *out, int *status, yvex_hip_stream stream)
{
    if (!gate || !up || !out || !status || !count || !(limit > 0.0)) return ST_INVALID_ARG;
    const uint64_t grid = (count + 255u) / 256u;
    if (grid > 0x7fffffffull) return ST_BOUNDS;
    swiglu_rows_kernel<<<(unsigned)grid, 256, 0, as_stream(stream)>>>(gate, up, count, limit, out, status);
    return check_launch("moe_swiglu_rows");
}

// From here on pair outputs are loaded past the caches: eight ranks of 7168 columns by 100 / 333 / 700 / 1111 / 2048 rows (23 to 470 MB) 7.3 /
// 17.3 / 33.5 / 49.6 / 93 us so, 7.0 / 17.8 / 34.3 / 54.3 / 105 through them.
constexpr uint64_t kReduceStreaming = 64ull << 20;

extern "C" int yvex_hip_moe_reduce_combine(const float *pair_outputs, uint64_t rows,
                                           uint64_t topk, uint64_t hidden, const float *shared,
                                           float *routed, float *combined, int *status,
                                           yvex_hip_stream stream)
{
    if (!pair_outputs || !status || !rows || !topk || !hidden || (!routed && !combined) ||
        (combined && !shared) || topk > 0xffffffffull)
        return ST_INVALID_ARG;
    if (rows > UINT64_MAX / hidden) return ST_BOUNDS;
    const uintptr_t addresses = (uintptr_t)pair_outputs | (uintptr_t)shared | (uintptr_t)routed |
                                (uintptr_t)combined;
    const bool quads = hidden % 4u == 0u && addresses % 16u == 0u;
    if ((rows * hidden / (quads ? 4u : 1u) + 255u) / 256u > 0x7fffffffull) return ST_BOUNDS;
    const uint64_t blocks = (hidden / (quads ? 4u : 1u) + 255u) / 256u;
    const dim3 grid((unsigned)blocks, (unsigned)(rows < 65535u ? rows : 65535u));
    const auto kernel = !quads ? reduce_combine_kernel<1, false>
                      : rows * topk * hidden * sizeof(float) > kReduceStreaming ? reduce_combine_kernel<4, true> : reduce_combine_kernel<4, false>;
    kernel<<<grid, 256, 0, as_stream(stream)>>>(pair_outputs, rows, (unsigned)topk, hidden, shared, routed, combined, status);
    return check_launch("moe_reduce_combine");
}
