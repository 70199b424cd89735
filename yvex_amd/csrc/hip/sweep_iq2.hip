// Decode-width expert sweeps specialised for IQ2_XXS (and, with the same pieces, streams and
// finishing pass, Q4_K rows and the Q2_K rows of a down projection) weights and Q8_K activations
// on gfx950. The notes below are about IQ2_XXS; what differs for Q4_K rows stands above
// `Q4kHalf`, for Q2_K rows above `Q2kHalf`.
//
// Same contract as the generic grouped kernel in moe.hip (src/backend/cuda/moe_kernels.cu:431-582
// is the reference's counterpart), built around the instruction budget of this one format: at
// 2.0625 bits per weight the vector ALU, not HBM, is the first limit, so every 32-weight unit is
// decoded with as few vector instructions as the format allows.
//
//   * magnitudes: one 16-byte LDS read returns the eight level bytes of a codebook entry and their
//     negations; signs: one 8-byte LDS read returns two byte-permute selectors for the 7 stored
//     sign bits plus parity; V_PERM_B32 then picks +level or -level per byte. Four signed weights
//     cost one vector instruction after the two reads.
//   * a sweep serves up to four (row, rank) pairs of a bucket, whose Q8_K columns stay in
//     registers (128 columns per lane), so an expert's bytes are decoded once for most buckets.
//   * the exact int32 superblock sum (kernel_primitives.h:287-313) is formed in the lane pair
//     that shares a superblock and scaled to fp32 as ((0.125 d_w) d_a) T (gate on even lanes, up
//     on odd lanes, or two row groups of the down projection): one float term per superblock,
//     the same float the CPU path forms. Every lane parks its term in an LDS window; when the
//     window is full a lane per weight row adds that row's terms in double, in superblock
//     order, and rounds the sum to float once: the row dot is bit for bit the sum the CPU path
//     computes (double accumulation over the blocks of a row, src/gguf/quant_compute.c:152-172),
//     so every value that is rounded to bfloat16 afterwards rounds as it does there.
//
// One workgroup per compute unit stays resident. The rows of all sweeps, weighed by what a sweep
// costs, are dealt out to the workgroups in one piece each (a piece may end in the middle of a
// sweep and the next begin there). A workgroup's waves draw short chunks of its piece from a
// counter in LDS: the older wave of a SIMD is served first and gets through 1.2 to 1.6 times the
// rows of the younger one. A wave whose next chunk belongs to the same sweep goes on with the
// activation columns it holds, and asks for that chunk's first rows before it is done with this
// one's, so that a chunk costs no round trip to memory.
//
// IMAGE: the weights come from the backend's own re-packing of the canonical bytes (built once at
// residency time, the canonical tensor stays the authority), made for this kernel's instruction
// budget. A superblock is two records of 36 bytes, one per lane of the pair that shares it:
//     dword 0      f16 d of the superblock | the four 4-bit group scales of this half << 16
//     dword 1 + 2j the four codebook bytes of group j of this half
//     dword 2 + 2j its four 7-bit sign fields, one to a byte
// so every load is dword-aligned with nothing to shift into place, a sign lookup address is one
// byte permute like a codebook lookup address (the canonical 7-bit fields need a shift and a
// mask each), and the scale arrives with the lane's own record. 72 bytes against 66.
#include "common.hpp"
#include "launch.hpp"
#include "grouped.hpp"

namespace yvex {

constexpr unsigned kSweepWaves = 8u;           // two per SIMD: the sweep of four pairs needs their registers
constexpr unsigned kSweepThreads = kSweepWaves * 64u;
constexpr int kSweepPairs = 4;                 // pairs of one bucket served by one sweep
constexpr int kSweepAheadSmall = 1;            // rows requested ahead of the one decoded, sweeps of one or two pairs
constexpr unsigned kSweepChunkShift = 4u;      // iterations a wave draws at a time (at most), as a power of two

// What a weight row costs a sweep that serves n pairs, relative to the other sweeps of the launch:
// what the workgroups' pieces of a launch are measured in. Fitted to the times of the workgroups of
// decode launches (23 to 96 rows) against what they had swept: IQ2_XXS 1 : 1.25 : 1.52 : 1.73 (the LDS
// pipe's share is the same whatever n is, the dot products come on top), Q2_K 1 : 1.17 : 1.34 : 1.48,
// Q4_K 1 : 0.95 : 1 : 1.03 (it waits for memory).
template <unsigned QT>
__device__ __forceinline__ constexpr unsigned sweep_cost(unsigned n)
{
    if (QT == QT_IQ2_XXS) return n >= 4u ? 14u : n == 3u ? 12u : n == 2u ? 10u : 8u;
    if (QT == QT_Q2_K) return n >= 4u ? 12u : n == 3u ? 11u : n == 2u ? 9u : 8u;
    return n >= 4u ? 13u : 12u;
}
// ... and the rows of one matrix with n pairs: sweeps of four and one of what is left.
template <unsigned QT>
__device__ __forceinline__ unsigned bucket_cost(unsigned n)
{
    return n / 4u * sweep_cost<QT>(4u) + (n % 4u ? sweep_cost<QT>(n % 4u) : 0u);
}

// LDS map (byte addresses; the dynamic block starts at LDS address 0)
constexpr unsigned kMagBase = 0u;              // 256 entries x 16 replicas x {+lo, +hi, -lo, -hi}
constexpr unsigned kSelBase = 65536u;          // 128 entries x 32 replicas x {selector lo, hi}
constexpr unsigned kTicketAddress = kSelBase + 128u * 32u * 8u;   // work-item counter of the workgroup
constexpr unsigned kPlaceAddress = kTicketAddress + 32u;          // what wave kPlacingWave found out for the workgroup
constexpr unsigned kPlacingWave = 4u;
constexpr unsigned kParkBase = kPlaceAddress + 32u;
// Per wave: a window of kWindowLines lines of 64 float terms (one line per iteration and packed
// value: even lanes' terms in the first 32 words, odd lanes' in the last 32, a weight row's
// terms next to each other in superblock order), then the (gate, up) row sums of a fused item
// ([stream][pair][row of the item]) for the SwiGLU pass at its end.
constexpr unsigned kWindowLines = 16u;
constexpr unsigned kWindowBytes = kWindowLines * 256u;
constexpr unsigned kFusedItemRows = 32u;       // weight row pairs of a chunk, at most
constexpr unsigned kResultBytes = 2u * 4u * kFusedItemRows * 4u;
// Behind them, for each of the sweep's pairs, {the row its results go to, its route weight}. A chunk's end finds them there by
// the pair: kept in registers through the loop they were what the compiler spilled, and scratch loads wait for the weight
// rows asked for ahead as well. With swiglu_bf16's exponential out of the loop's registers too, experts of one
// pair over the image, gate and up of 7168 x 2048: 40 of them 80 -> 73 us, 168 of them 285 -> 281 (265 to 310 and 257 to 318 by
// where the experts lie); 94 of one pair, 47 of two, 16 of three and 3 of four, down: 137 -> 134.
constexpr unsigned kInfoOffset = kWindowBytes + kResultBytes, kInfoBytes = 4u * 8u;
constexpr unsigned kParkBytes = kInfoOffset + kInfoBytes;
constexpr unsigned kMaxSweeps = 4096u;
// What opens an item without a round trip to memory: expert, first ordered pair and population of
// every routed bucket, and {source pair, route weight} of every ordered pair when the routed
// problem has at most kPairCacheMax of them (decode widths; wider batches read them from memory).
constexpr unsigned kBucketBase = kParkBase + kSweepWaves * kParkBytes;     // 256 x {expert, first, population, -}
constexpr unsigned kPairCacheBase = kBucketBase + 256u * 16u;
constexpr unsigned kPairCacheMax = 1024u;
constexpr unsigned kSweepLdsBytes = kPairCacheBase + kPairCacheMax * 8u;
static_assert(kSweepLdsBytes <= 160u * 1024u, "the sweep's tables, lists and caches must fit the LDS of a compute unit");

__device__ __forceinline__ void lds_store_u32(unsigned address, unsigned v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    *reinterpret_cast<__attribute__((address_space(3))) unsigned *>(address) = v;
#else
    (void)address;
    (void)v;
#endif
}
__device__ __forceinline__ void lds_store_uint2(unsigned address, uint2 v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    *reinterpret_cast<__attribute__((address_space(3))) uint2 *>(address) = v;
#else
    (void)address;
    (void)v;
#endif
}
__device__ __forceinline__ void lds_store_uint4(unsigned address, uint4 v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    *reinterpret_cast<__attribute__((address_space(3))) uint4 *>(address) = v;
#else
    (void)address;
    (void)v;
#endif
}
__device__ __forceinline__ uint2 lds_load_uint2(unsigned address)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *reinterpret_cast<__attribute__((address_space(3))) const uint2 *>(address);
#else
    (void)address;
    return make_uint2(0u, 0u);
#endif
}
__device__ __forceinline__ unsigned lds_load_u32(unsigned address)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *reinterpret_cast<__attribute__((address_space(3))) const unsigned *>(address);
#else
    (void)address;
    return 0u;
#endif
}

// The lookup tables: the first 256 threads form one codebook entry each and store its sixteen
// replicas, the others one sign entry in twos, sixteen replicas each. Step t stores the replica
// after the lane's own by t, so that a store's lanes spread over all banks. (One replica a thread and
// turn, all turns unrolled, was several kilobytes of code that every launch fetched to run it
// once, and eight codebook loads a thread: 1.5 us, with it 3 of the 7 us a launch opened with.)
static_assert(kSweepThreads == 512u, "a thread a codebook entry, two a sign entry");

__device__ __forceinline__ unsigned sweep_table_digits() { return k_iq2_digits[threadIdx.x & 255u]; }

__device__ __forceinline__ void sweep_levels_fill(unsigned digits)       // threads 0 .. 255
{
    const uint2 m = iq2_magnitude_of_digits(digits);
    // byte-wise negation: every level is >= 8, so (x ^ 0xff) + 1 never carries
    const uint4 entry = make_uint4(m.x, m.y, (m.x ^ 0xffffffffu) + 0x01010101u, (m.y ^ 0xffffffffu) + 0x01010101u);
#pragma unroll 4
    for (unsigned t = 0; t < 16u; ++t)
        lds_store_uint4(kMagBase + threadIdx.x * 256u + ((threadIdx.x + t) & 15u) * 16u, entry);
}

__device__ __forceinline__ void sweep_signs_fill()                       // threads 256 .. 511
{
    const unsigned s7 = (threadIdx.x - 256u) >> 1, upper = threadIdx.x & 1u;
    const unsigned s = s7 | ((__popc(s7) & 1u) << 7);
    // selector byte k = k (take +level, source 1) or k + 4 (take -level, source 0)
    unsigned lo = 0x03020100u, hi = 0x03020100u;
#pragma unroll
    for (unsigned l = 0; l < 4u; ++l) {
        lo += ((s >> l) & 1u) << (8u * l + 2u);
        hi += ((s >> (l + 4u)) & 1u) << (8u * l + 2u);
    }
#pragma unroll 4
    for (unsigned t = 0; t < 16u; ++t)
        lds_store_uint2(kSelBase + s7 * 256u + upper * 128u + ((s7 + t) & 15u) * 8u, make_uint2(lo, hi));
}

// A lane's share of one IQ2_XXS weight row: half a superblock, 32 packed bytes plus the scale.
// Superblocks are 66 bytes, so the codes start on a 2-byte boundary, and vector loads that are
// not dword-aligned run at less than half rate on this part. Every load here is dword-aligned:
// eight dwords from the aligned address at or below the codes and a ninth whose place depends on
// the lane; the consumer shifts the codes into place with byte-align instructions. Each load
// instruction costs the memory pipeline about two cycles per cache line its lanes touch, so the
// fp16 scale gets no instruction of its own. Rows start on dword boundaries and superblocks are
// 66 bytes, so in even superblocks the codes start two bytes into their aligned window: the
// ninth dword is the end of the codes, and the scale is the low half of the first dword of the
// superblock's first half. In odd superblocks the codes fill eight aligned dwords exactly and
// the ninth load fetches the dword whose high half is the scale.
struct Iq2Half {
    uint4 lo, hi;
    unsigned tail;
    // rows: wave-uniform address of the iteration's first weight row; the rest are this lane's
    // byte offsets from it (scalar base + 32-bit lane offset addressing)
    __device__ __forceinline__ void load(const unsigned char *rows, unsigned codes_at, unsigned tail_at)
    {
        lo = *reinterpret_cast<const uint4 *>(rows + codes_at);          // 4-byte aligned
        hi = *reinterpret_cast<const uint4 *>(rows + codes_at + 16u);
        tail = *reinterpret_cast<const unsigned *>(rows + tail_at);
    }
};

struct SweepLane {
    unsigned lanes_per_row, rows_per_iter;
    unsigned sub, super, half;
    bool live;
    unsigned mag_lane;     // (lane % 16) * 16
    unsigned sel_lane;     // kSelBase + (lane % 32) * 8
    unsigned code_shift;   // bytes the codes sit above their aligned load address: 0 or 2
    unsigned scale_shift;  // bits the fp16 scale sits above its aligned load address: 0 or 16
    unsigned park;         // this wave's term window
    unsigned term_slot;    // the lane's word inside a line of the window (byte offset)
    unsigned results;      // the wave's row sums of a fused item
    unsigned terms;        // superblocks of a weight row: the float terms of one row sum
    unsigned row_shift;    // log2(rows_per_iter)
};

__device__ __forceinline__ int dot4_from_zero(unsigned a, unsigned b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    int d;
    asm("v_dot4_i32_i8 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
    return d;
#else
    (void)a;
    (void)b;
    return 0;
#endif
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v)
{
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// Exact integer sums of this lane's four units of each of STREAMS weight rows against N
// activation rows. The work is cut into eight stages of half a unit per stream (two codebook
// lookups, two selector lookups, sixteen weights); the LDS reads of stage s + DEPTH are issued
// before stage s is consumed, so their latency runs under the permutes and dot products of the
// stages between. A stage holds independent dependency chains (one per stream, or the even and
// odd products of a single stream), because a dependent vector instruction issues only about
// nine cycles after its producer.
template <int STREAMS, int N, bool IMAGE>
__device__ __forceinline__ void iq2_half_dots(const Iq2Half (&c)[STREAMS], const SweepLane &g,
                                              const unsigned (&act)[N][32], int (&total)[STREAMS][N])
{
    constexpr int kStages = 8;
    constexpr int DEPTH = STREAMS == 2 ? 1 : 2;
    constexpr int CHAINS = STREAMS == 2 ? 1 : 2;   // accumulators per (stream, pair)
    unsigned q[STREAMS][8];
#pragma unroll
    for (int w = 0; w < STREAMS; ++w) {
        const unsigned raw[9] = {c[w].lo.x, c[w].lo.y, c[w].lo.z, c[w].lo.w,
                                 c[w].hi.x, c[w].hi.y, c[w].hi.z, c[w].hi.w, c[w].tail};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            q[w][i] = IMAGE ? raw[i] : __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], g.code_shift);
#pragma unroll
        for (int p = 0; p < N; ++p) total[w][p] = 0;
    }
    uint4 mag[DEPTH + 1][STREAMS][2];
    uint2 sel[DEPTH + 1][STREAMS][2];
    auto issue = [&](int stage) {
        const int k = stage >> 1, h = stage & 1, slot = stage % (DEPTH + 1);
#pragma unroll
        for (int w = 0; w < STREAMS; ++w) {
            const unsigned grids = q[w][2 * k], aux = q[w][2 * k + 1];
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
                const unsigned j = 2u * (unsigned)h + (unsigned)jj;
                // magnitude address = index byte j << 8 | replica offset
                const unsigned ma = __builtin_amdgcn_perm(grids, g.mag_lane, 0x0c0c0400u + (j << 8));
                // selector address = sign field j moved to bit 8 | replica offset: the image holds
                // the field in byte j (the table base's third byte comes from the replica word),
                // the canonical word holds it at bit 7j
                unsigned sa;
                if constexpr (IMAGE) {
                    sa = __builtin_amdgcn_perm(aux, g.sel_lane, 0x0c020400u + (j << 8));
                } else {
                    const unsigned moved = 7u * j >= 8u ? aux >> (7u * j - 8u) : aux << (8u - 7u * j);
                    sa = (moved & 0x7f00u) | g.sel_lane;
                }
                mag[slot][w][jj] = lds_read_uint4(ma);
                sel[slot][w][jj] = lds_read_uint2(sa);
            }
        }
    };
#pragma unroll
    for (int stage = 0; stage < DEPTH; ++stage) issue(stage);
    int d[STREAMS][N][CHAINS];
#pragma unroll
    for (int stage = 0; stage < kStages; ++stage) {
        if (stage + DEPTH < kStages) issue(stage + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        const int k = stage >> 1, h = stage & 1, slot = stage % (DEPTH + 1);
        unsigned weights[STREAMS][4];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int w = 0; w < STREAMS; ++w) {
                weights[w][2 * jj] = __builtin_amdgcn_perm(mag[slot][w][jj].z, mag[slot][w][jj].x, sel[slot][w][jj].x);
                weights[w][2 * jj + 1] = __builtin_amdgcn_perm(mag[slot][w][jj].w, mag[slot][w][jj].y, sel[slot][w][jj].y);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int p = 0; p < N; ++p)
#pragma unroll
                for (int w = 0; w < STREAMS; ++w) {
                    const int chain = i % CHAINS;
                    const unsigned x = act[p][8 * k + 4 * h + i];
                    // the first product of a chain starts from the constant zero
                    if (h == 0 && i < CHAINS) d[w][p][chain] = dot4_from_zero(weights[w][i], x);
                    else d[w][p][chain] = dot4(weights[w][i], x, d[w][p][chain]);
                }
        if (h == 1) {
#pragma unroll
            for (int w = 0; w < STREAMS; ++w) {
                // 2 s + 1: bit 27 of the canonical word is a sign bit, forced to 1; the image
                // keeps the scale of group k in bits 16 + 4k of the record's first dword
                const int factor = IMAGE ? (int)(((c[w].tail >> (15 + 4 * k)) & 0x1eu) | 1u)
                                         : (int)((q[w][2 * k + 1] >> 27) | 1u);
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    int sum = d[w][p][0];
                    if (CHAINS == 2) sum += d[w][p][1];
                    total[w][p] += __mul24(sum, factor);   // |sum| < 2^23
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ---- Q4_K rows in the same sweeps ---------------------------------------------------------------
//
// A lane's share of one Q4_K weight row: the superblock's 16-byte head (d, dmin, the twelve bytes
// of 6-bit scales and minimums) and the 64 code bytes of its half (sub-blocks 4 h .. 4 h + 3:
// two chunks of 32 bytes, low nibbles one sub-block and high nibbles the next). Superblocks are
// 144 bytes, so every load is 16-byte aligned relative to the row.
struct Q4kHalf {
    uint4 head;
    uint4 q[4];
    __device__ __forceinline__ void load(const unsigned char *rows, unsigned codes_at, unsigned head_at)
    {
        head = *reinterpret_cast<const uint4 *>(rows + head_at);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const uint4 *>(rows + codes_at + 16u * i);
    }
};

// ---- Q2_K rows in the same sweeps (the down experts of the reference's model file) --------------
//
// A lane's share of one Q2_K weight row (public ggml block_q2_K, 84 bytes: sixteen bytes
// scale | minimum << 4 of the 16-value sub-blocks, 64 bytes of 2-bit codes, fp16 d and dmin): the
// 32 code bytes of its half (byte l holds the values 32 s + l of the half at bit 2 s), the half's
// eight scale bytes and the dword of d and dmin. Superblocks are dword-aligned, not more.
struct Q2kHalf {
    uint4 q[2];
    uint2 scales;
    unsigned dd;
    __device__ __forceinline__ void load(const unsigned char *rows, unsigned codes_at, unsigned scales_at,
                                         unsigned dd_at)
    {
        q[0] = *reinterpret_cast<const uint4 *>(rows + codes_at);
        q[1] = *reinterpret_cast<const uint4 *>(rows + codes_at + 16u);
        scales = *reinterpret_cast<const uint2 *>(rows + scales_at);
        dd = *reinterpret_cast<const unsigned *>(rows + dd_at);
    }
};

template <unsigned QT>
struct SweepHalf {
    using type = Iq2Half;
};
template <>
struct SweepHalf<QT_Q4_K> {
    using type = Q4kHalf;
};
template <>
struct SweepHalf<QT_Q2_K> {
    using type = Q2kHalf;
};

// Exact integer sums of this lane's eight Q2_K sub-blocks of each of STREAMS weight rows against N
// activation rows: dot = sum over sub-blocks of scale * (codes . activations), minimum = sum of
// minimum * (sum of the sub-block's sixteen activations), the two terms of the reference's
// primitive (src/backend/cuda/kernel_primitives.h:314-341). A code is a shift and a mask away.
template <int STREAMS, int N>
__device__ __forceinline__ void q2k_half_dots(const Q2kHalf (&c)[STREAMS], const unsigned (&act)[N][32],
                                              const int (&act_sums)[N][8], int (&dot)[STREAMS][N],
                                              int (&minimum)[STREAMS][N])
{
#pragma unroll
    for (int w = 0; w < STREAMS; ++w) {
        const unsigned packed[2] = {c[w].scales.x, c[w].scales.y};
        const unsigned words[8] = {c[w].q[0].x, c[w].q[0].y, c[w].q[0].z, c[w].q[0].w,
                                   c[w].q[1].x, c[w].q[1].y, c[w].q[1].z, c[w].q[1].w};
#pragma unroll
        for (int p = 0; p < N; ++p) {
            int m = 0;
#pragma unroll
            for (int sub = 0; sub < 8; ++sub)       // 15 * 16 * 128 * 8 < 2^23
                m += __mul24((int)((packed[sub >> 2] >> (8 * (sub & 3) + 4)) & 15u), act_sums[p][sub]);
            minimum[w][p] = m;
            dot[w][p] = 0;
        }
#pragma unroll
        for (int shift = 0; shift < 4; ++shift) {
            int first[N], second[N];     // sub-blocks 2 shift (bytes 0-15) and 2 shift + 1 (bytes 16-31)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned codes = (words[i] >> (2 * shift)) & 0x03030303u;
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    if (i < 4) first[p] = i == 0 ? dot4_from_zero(codes, act[p][8 * shift + i])
                                                  : dot4(codes, act[p][8 * shift + i], first[p]);
                    else second[p] = i == 4 ? dot4_from_zero(codes, act[p][8 * shift + i])
                                            : dot4(codes, act[p][8 * shift + i], second[p]);
                }
            }
            const int sc_first = (int)((packed[shift >> 1] >> (16 * (shift & 1))) & 15u);
            const int sc_second = (int)((packed[shift >> 1] >> (16 * (shift & 1) + 8)) & 15u);
#pragma unroll
            for (int p = 0; p < N; ++p)   // |sum| <= 3 * 128 * 16 < 2^13
                dot[w][p] += __mul24(first[p], sc_first) + __mul24(second[p], sc_second);
        }
    }
}

// Exact integer sums of this lane's four sub-blocks of each of STREAMS weight rows against N
// activation rows: dot = sum over sub-blocks of scale * (nibbles . activations), minimum = sum of
// minimum * (sum of the sub-block's activations), the two terms of the reference's primitive
// (src/backend/cuda/kernel_primitives.h:315-340). No tables: a nibble is a mask away.
template <int STREAMS, int N>
__device__ __forceinline__ void q4k_half_dots(const Q4kHalf (&c)[STREAMS], const SweepLane &g,
                                              const unsigned (&act)[N][32], const int (&act_sums)[N][4],
                                              int (&dot)[STREAMS][N], int (&minimum)[STREAMS][N])
{
#pragma unroll
    for (int w = 0; w < STREAMS; ++w) {
        const unsigned s0 = c[w].head.y, s1 = c[w].head.z, s2 = c[w].head.w;
        // the four scales and the four minimums of this half, one to a byte
        const unsigned scales = g.half ? ((s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)) : (s0 & 0x3f3f3f3fu);
        const unsigned minimums = g.half ? (((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u))
                                         : (s1 & 0x3f3f3f3fu);
#pragma unroll
        for (int p = 0; p < N; ++p) {
            int m = 0;
#pragma unroll
            for (int sub = 0; sub < 4; ++sub)
                m += __mul24((int)((minimums >> (8 * sub)) & 255u), act_sums[p][sub]);   // 63 * 32 * 127 * 4 < 2^23
            minimum[w][p] = m;
            dot[w][p] = 0;
        }
#pragma unroll
        for (int chunk = 0; chunk < 2; ++chunk) {
            const unsigned words[8] = {c[w].q[2 * chunk].x, c[w].q[2 * chunk].y, c[w].q[2 * chunk].z,
                                       c[w].q[2 * chunk].w, c[w].q[2 * chunk + 1].x, c[w].q[2 * chunk + 1].y,
                                       c[w].q[2 * chunk + 1].z, c[w].q[2 * chunk + 1].w};
            int low[N], high[N];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned lo = words[i] & 0x0f0f0f0fu, hi = (words[i] >> 4) & 0x0f0f0f0fu;
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    low[p] = i == 0 ? dot4_from_zero(lo, act[p][16 * chunk + i]) : dot4(lo, act[p][16 * chunk + i], low[p]);
                    high[p] = i == 0 ? dot4_from_zero(hi, act[p][16 * chunk + 8 + i])
                                     : dot4(hi, act[p][16 * chunk + 8 + i], high[p]);
                }
            }
#pragma unroll
            for (int p = 0; p < N; ++p)   // |sum| <= 15 * 127 * 32 < 2^16
                dot[w][p] += __mul24(low[p], (int)((scales >> (16 * chunk)) & 255u)) +
                             __mul24(high[p], (int)((scales >> (16 * chunk + 8)) & 255u));
        }
    }
}

// The workgroup's next chunk, for every lane of the wave.
__device__ __forceinline__ unsigned draw_chunk()
{
    unsigned got = 0u;
    if ((threadIdx.x & 63u) == 0u)
        got = __hip_atomic_fetch_add(reinterpret_cast<__attribute__((address_space(3))) unsigned *>(kTicketAddress), 1u,
                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return (unsigned)__builtin_amdgcn_readfirstlane((int)got);
}

// One sweep over weight rows [row_begin, row_end) for N live pairs: chunk `chunk` of them
// (1 << chunk_shift iterations each) and whatever chunks of the same rows this wave draws next; returns
// the first one drawn that lies behind them (as drawn: the rows' first chunk is number `base`).
// MODE 0: one weight row group (the rows of one iteration) at a time; MODE 1: a gate row group
// and the matching up row group, SwiGLU in the finishing pass; MODE 2: two consecutive row groups
// of one matrix, which share the activation columns as gate and up rows do: the fixed cost of an
// iteration (requests, waits, reduction, loop control) is spent once per two groups.
template <int MODE, int N, bool IMAGE, unsigned QT>
__device__ __forceinline__ unsigned iq2_sweep(const GroupedArgs &a, const GroupedProblem &pr,
                                              const SweepLane &g, const unsigned char *gate_e,
                                              const unsigned char *up_e, unsigned long long first_ordered,
                                              unsigned row_begin, unsigned row_end, bool pairs_in_lds,
                                              unsigned chunk, unsigned base, unsigned chunk_shift)
{
    constexpr bool FUSED = MODE == 1;
    constexpr bool TWIN = MODE != 0;     // two streams of weight rows against the same activation columns
    constexpr bool Q4 = QT == QT_Q4_K, Q2 = QT == QT_Q2_K;
    constexpr bool KQ = Q4 || Q2;        // formats with a minimum term
    static_assert(!(KQ && IMAGE), "the image is a layout of IQ2_XXS rows");
    const unsigned lane = threadIdx.x & 63u;
    const bool odd = (lane & 1u) != 0u;
    // packed values per iteration: (first, second stream) of pair v with two streams, else pairs (2v, 2v + 1)
    constexpr int PV = TWIN ? N : (N + 1) / 2;

    // ---- the sweep's activation rows: this lane's 128 columns stay in registers ----
    unsigned act[N][32];
    // the sums of the activations under each of the lane's sub-blocks: four of 32 (Q4_K), eight of 16 (Q2_K)
    int act_sums[N][Q4 ? 4 : Q2 ? 8 : 1];
    float act_scale[N];
#pragma unroll
    for (int p = 0; p < N; ++p) {
        const unsigned long long ordered = first_ordered + p;
        unsigned source;             // (the launch wrapper bounds the pairs)
        float route_weight;
        if (pairs_in_lds) {      // wave-uniform
            const uint2 cached = lds_load_uint2(kPairCacheBase + 8u * (unsigned)ordered);
            source = cached.x;
            route_weight = __uint_as_float(cached.y);
        } else {
            source = (unsigned)(pr.order ? pr.order[ordered] : ordered);
            route_weight = pr.route_weights ? pr.route_weights[source] : 1.0f;
        }
        const unsigned long long arow = pr.act_by_ordered_pair ? ordered : source / pr.topk;
        if (lane == 0u)
            lds_store_uint2(g.park + kInfoOffset + 8u * (unsigned)p,
                            make_uint2(pr.out_by_source_pair ? source : (unsigned)ordered, __float_as_uint(route_weight)));
        const unsigned char *blk = (const unsigned char *)pr.activations + arow * pr.act_stride +
                                   (unsigned long long)(g.live ? g.super : 0u) * kQ8KBytes;
        // lanes past the last row group multiply zeros
        act_scale[p] = g.live ? *reinterpret_cast<const float *>(blk) : 0.0f;
        const unsigned char *qv = blk + 4u + 128u * g.half;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            uint4 v;
            __builtin_memcpy(&v, qv + 16 * k, 16);
            act[p][4 * k] = g.live ? v.x : 0u;
            act[p][4 * k + 1] = g.live ? v.y : 0u;
            act[p][4 * k + 2] = g.live ? v.z : 0u;
            act[p][4 * k + 3] = g.live ? v.w : 0u;
        }
        if constexpr (Q4) {
            // the block's sixteen sums of 16 activations follow its 256 values: eight belong to this half
            uint4 sums;
            __builtin_memcpy(&sums, blk + 260u + 16u * g.half, 16);
            const unsigned pairs_of_sums[4] = {sums.x, sums.y, sums.z, sums.w};
#pragma unroll
            for (int sub = 0; sub < 4; ++sub)
                act_sums[p][sub] = g.live ? (int)(short)(pairs_of_sums[sub] & 0xffffu) + (int)(short)(pairs_of_sums[sub] >> 16)
                                          : 0;
        } else if constexpr (Q2) {
            uint4 sums;
            __builtin_memcpy(&sums, blk + 260u + 16u * g.half, 16);
            const unsigned pairs_of_sums[4] = {sums.x, sums.y, sums.z, sums.w};
#pragma unroll
            for (int sub = 0; sub < 8; ++sub)
                act_sums[p][sub] = !g.live ? 0 : sub % 2 ? (int)pairs_of_sums[sub / 2] >> 16
                                                         : (int)(short)(pairs_of_sums[sub / 2] & 0xffffu);
        } else {
            act_sums[p][0] = 0;
        }
    }
    // the activation scale each lane applies to packed value v
    float packed_scale[PV];
#pragma unroll
    for (int v = 0; v < PV; ++v) {
        if constexpr (TWIN) packed_scale[v] = act_scale[v];
        else packed_scale[v] = odd ? (2 * v + 1 < N ? act_scale[2 * v + 1 < N ? 2 * v + 1 : 0] : 0.0f)
                                   : act_scale[2 * v];
    }

    const unsigned rows_per_turn = MODE == 2 ? 2u * g.rows_per_iter : g.rows_per_iter;
    const unsigned rows = row_end - row_begin;               // a multiple of rows_per_turn
    const unsigned iterations = rows >> (g.row_shift + (MODE == 2 ? 1u : 0u)), chunk_turns = 1u << chunk_shift;
    // wave-uniform row bases advance by a scalar stride; the lane's place inside an iteration's
    // rows is a constant 32-bit offset
    const unsigned char *gate_rows = gate_e + (unsigned long long)row_begin * pr.row_bytes;
    const unsigned long long second_row_bytes = FUSED ? pr.up_row_bytes : pr.row_bytes;
    const unsigned char *up_rows = FUSED ? up_e + (unsigned long long)row_begin * pr.up_row_bytes
        : MODE == 2 ? gate_rows + (unsigned long long)g.rows_per_iter * pr.row_bytes : nullptr;
    const unsigned long long gate_step = (unsigned long long)rows_per_turn * pr.row_bytes;
    const unsigned long long up_step = (unsigned long long)rows_per_turn * second_row_bytes;
    const unsigned lane_row = g.live ? g.sub : 0u, lane_super = g.live ? g.super : 0u;
    // (row bases and row strides are multiples of four bytes: checked on the host)
    constexpr unsigned kSuperBytes = Q4 ? 144u : Q2 ? 84u : IMAGE ? 72u : 66u;
    const unsigned gate_block = lane_row * (unsigned)pr.row_bytes + lane_super * kSuperBytes;
    const unsigned up_block = lane_row * (unsigned)second_row_bytes + lane_super * kSuperBytes;
    // image: the lane's record is its first dword (scale and group scales) and eight more
    // (Q4_K: the half's 64 code bytes behind the 16-byte head, which is the "tail" load)
    // (Q2_K: the half's 32 code bytes behind the sixteen scale bytes; "tail" is the half's eight scale bytes)
    const unsigned gate_codes_at = Q4 ? gate_block + 16u + 64u * g.half
        : Q2 ? gate_block + 16u + 32u * g.half
        : IMAGE ? gate_block + 36u * g.half + 4u
                : (gate_block + 2u + 32u * g.half) & ~3u;   // + code_shift = codes
    const unsigned up_codes_at = Q4 ? up_block + 16u + 64u * g.half
        : Q2 ? up_block + 16u + 32u * g.half
        : IMAGE ? up_block + 36u * g.half + 4u : (up_block + 2u + 32u * g.half) & ~3u;
    // ninth dword: the end of the codes where they start two bytes in, else the scale's dword
    const unsigned gate_tail_at = Q4 ? gate_block : Q2 ? gate_block + 8u * g.half : IMAGE ? gate_codes_at - 4u
                                        : g.code_shift ? gate_codes_at + 32u : gate_block & ~3u;
    const unsigned up_tail_at = Q4 ? up_block : Q2 ? up_block + 8u * g.half
        : IMAGE ? up_codes_at - 4u : g.code_shift ? up_codes_at + 32u : up_block & ~3u;
    // Ring of packed rows: the bytes of iteration it + AHEAD are requested before iteration it is
    // decoded, so about AHEAD iterations of arithmetic cover the HBM latency.
    // The loop body is one basic block: every turn requests a row (the last ones clamped to the
    // final row) and every lane stores (lanes that hold no result write to a spare word), so no
    // branch sits between a request and the wait that consumes it and the waits stay counted.
    constexpr int AHEAD = N <= 2 ? kSweepAheadSmall : 1;   // rows requested ahead of the one decoded
    constexpr int STREAMS = TWIN ? 2 : 1;
    using Half = typename SweepHalf<QT>::type;
    Half ring[AHEAD + 1][STREAMS];
    auto request = [&](Half (&slot)[STREAMS], unsigned it) {
        if constexpr (Q2) {
            slot[0].load(gate_rows + it * gate_step, gate_codes_at, gate_tail_at, gate_block + 80u);
            if constexpr (TWIN)
                slot[1].load(up_rows + it * up_step, up_codes_at, up_tail_at, up_block + 80u);
        } else {
            slot[0].load(gate_rows + it * gate_step, gate_codes_at, gate_tail_at);
            if constexpr (TWIN)
                slot[1].load(up_rows + it * up_step, up_codes_at, up_tail_at);
        }
    };
    static_assert(AHEAD == 1, "a chunk's last turn asks for the first rows of the next");
    const unsigned chunks = (iterations + chunk_turns - 1u) >> chunk_shift;
    unsigned begin = chunk << chunk_shift;
    __builtin_amdgcn_sched_barrier(0);
    request(ring[0], begin);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the window's row sums: a lane per (line, parity, row of the iteration) adds that
    // row's float terms in double, in superblock order, and rounds once ----
    // A fused item keeps the sums for the SwiGLU pass at its end; a plain projection rounds to
    // bfloat16 and stores here.
    const unsigned R = g.rows_per_iter;
    auto flush = [&](unsigned first_iteration, unsigned count, unsigned chunk_begin) {
        // LDS operations of one wave complete in order, so the terms parked above are visible here
        wave_lds_fence();
        const unsigned sums = (count * (unsigned)PV * 2u) << g.row_shift;
        const unsigned segment_bytes = 128u >> g.row_shift;       // a row's terms of one parity
        for (unsigned s = lane; s < sums; s += 64u) {
            const unsigned line = s >> (g.row_shift + 1u), rest = s & (2u * R - 1u);
            const unsigned parity = rest >> g.row_shift, group = rest & (R - 1u);
            const unsigned at = g.park + line * 256u + parity * 128u + group * segment_bytes;
            double sum = 0.0;
            unsigned k = 0u;
            // (long rows of formats that have the registers: two reads on their way before the first addition)
            const unsigned doubled = !Q4 && g.terms > 16u ? g.terms & ~7u : 0u;
            if constexpr (!Q4) for (; k < doubled; k += 8u) {
                const uint4 t = lds_read_uint4(at + 4u * k), u = lds_read_uint4(at + 4u * k + 16u);
                sum += (double)__uint_as_float(t.x);
                sum += (double)__uint_as_float(t.y);
                sum += (double)__uint_as_float(t.z);
                sum += (double)__uint_as_float(t.w);
                sum += (double)__uint_as_float(u.x);
                sum += (double)__uint_as_float(u.y);
                sum += (double)__uint_as_float(u.z);
                sum += (double)__uint_as_float(u.w);
            }
            for (; k + 4u <= g.terms; k += 4u) {
                const uint4 t = lds_read_uint4(at + 4u * k);
                sum += (double)__uint_as_float(t.x);
                sum += (double)__uint_as_float(t.y);
                sum += (double)__uint_as_float(t.z);
                sum += (double)__uint_as_float(t.w);
            }
            for (; k < g.terms; ++k) sum += (double)__uint_as_float(lds_load_u32(at + 4u * k));
            const float row_sum = (float)sum;
            const unsigned iteration = first_iteration + line / (unsigned)PV, v = line % (unsigned)PV;
            if constexpr (FUSED) {
                const unsigned local = ((iteration - chunk_begin) << g.row_shift) + group;   // < kFusedItemRows
                lds_store_u32(g.results + ((parity * (unsigned)N + v) * kFusedItemRows + local) * 4u,
                              __float_as_uint(row_sum));
            } else {
                // two row groups an iteration: pair v, group `parity`; one: pairs 2v and 2v + 1
                const unsigned p = TWIN ? v : 2u * v + parity;
                const unsigned row = row_begin + (TWIN ? ((2u * iteration + parity) << g.row_shift)
                                                       : (iteration << g.row_shift)) + group;
                const float value = bf16_round(row_sum);
                if (p < (unsigned)N) {
                    const unsigned long long oi = lds_load_u32(g.park + kInfoOffset + 8u * p);
                    if (!finite_f32(value)) raise_status(a.status, 1);
                    else pr.out[oi * a.out_rows + row] = value;
                }
            }
        }
        wave_lds_fence();
    };
    // iterations a window holds (a multiple of the turns of one trip through the loop below)
    constexpr unsigned kWindowIters = (kWindowLines / (unsigned)PV) / (AHEAD + 1) * (AHEAD + 1);
    static_assert(kWindowIters >= AHEAD + 1, "a window holds at least one trip's lines");

    for (;;) {
    // the chunk behind this one, whose rows the last turn below asks for (past the last of these
    // rows: this chunk's last rows once more, which nobody uses)
    const unsigned drawn = draw_chunk(), next = drawn - base;
    const unsigned finish = begin + chunk_turns < iterations ? begin + chunk_turns : iterations;
    const unsigned padded = begin + ((finish - begin + 1u) & ~1u);
    const unsigned follow = next < chunks ? next << chunk_shift : finish - 1u;
    unsigned window_begin = begin;
    while (window_begin < finish) {
      const unsigned window_end = window_begin + kWindowIters < finish ? window_begin + kWindowIters : finish;
      unsigned park_at = g.park + g.term_slot;
      for (unsigned it0 = window_begin; it0 < window_end; it0 += AHEAD + 1) {
#pragma unroll
      for (int turn = 0; turn <= AHEAD; ++turn) {
        const unsigned it = it0 + (unsigned)turn;   // may run past the chunk's last rows by a turn
        const unsigned ahead = it + 1u;
        request(ring[(turn + AHEAD) % (AHEAD + 1)], ahead >= padded ? follow : ahead < finish ? ahead : finish - 1u);
        const Half (&now)[STREAMS] = ring[turn];
        int total_gate[N], total_up[N];
        int min_gate[N], min_up[N];          // Q4_K: the sums of the minimum term
        {
            int totals[STREAMS][N], minimums[STREAMS][N];
            if constexpr (Q4) {
                q4k_half_dots<STREAMS, N>(now, g, act, act_sums, totals, minimums);
            } else if constexpr (Q2) {
                q2k_half_dots<STREAMS, N>(now, act, act_sums, totals, minimums);
            } else {
                iq2_half_dots<STREAMS, N, IMAGE>(now, g, act, totals);
#pragma unroll
                for (int w = 0; w < STREAMS; ++w)
#pragma unroll
                    for (int p = 0; p < N; ++p) minimums[w][p] = 0;
            }
#pragma unroll
            for (int p = 0; p < N; ++p) {
                total_gate[p] = totals[0][p];
                total_up[p] = totals[STREAMS - 1][p];
                min_gate[p] = minimums[0][p];
                min_up[p] = minimums[STREAMS - 1][p];
            }
        }
        // the two lanes of a superblock add their halves: exact int32 superblock sums
#pragma unroll
        for (int p = 0; p < N; ++p) {
            total_gate[p] += dpp_move<0xb1, 0xf>(total_gate[p]);
            if constexpr (TWIN) total_up[p] += dpp_move<0xb1, 0xf>(total_up[p]);
            if constexpr (KQ) {
                min_gate[p] += dpp_move<0xb1, 0xf>(min_gate[p]);
                if constexpr (TWIN) min_up[p] += dpp_move<0xb1, 0xf>(min_up[p]);
            }
        }
        // The even lane of a pair scales the first stream and the odd lane the last one. An odd
        // lane holds the second half of its superblock, so where the scale rides in the first
        // half's codes it comes from the neighbour.
        const Half &mine = odd ? now[STREAMS - 1] : now[0];
        float weight_scale, weight_minimum = 0.0f;
        if constexpr (Q4) {
            weight_scale = f16_bits_to_float(mine.head.x & 0xffffu);       // d
            weight_minimum = f16_bits_to_float(mine.head.x >> 16);         // dmin
        } else if constexpr (Q2) {
            weight_scale = f16_bits_to_float(mine.dd & 0xffffu);
            weight_minimum = f16_bits_to_float(mine.dd >> 16);
        } else if constexpr (IMAGE) {
            weight_scale = 0.125f * f16_bits_to_float(mine.tail & 0xffffu);
        } else {
            // (the exchange runs in every lane: it reads its neighbour, which must be executing it)
            const unsigned neighbour_word = (unsigned)dpp_move<0xb1, 0xf>((int)now[STREAMS - 1].lo.x);
            const unsigned first_word = odd ? neighbour_word : now[0].lo.x;
            weight_scale = 0.125f * f16_bits_to_float(
                ((g.code_shift ? first_word : mine.tail) >> g.scale_shift) & 0xffffu);
        }
#pragma unroll
        for (int v = 0; v < PV; ++v) {
            int t, m = 0;
            if constexpr (TWIN) t = odd ? total_up[v] : total_gate[v];
            else t = odd ? total_gate[2 * v + 1 < N ? 2 * v + 1 : 2 * v] : total_gate[2 * v];
            float value;
            if constexpr (KQ) {
                if constexpr (TWIN) m = odd ? min_up[v] : min_gate[v];
                else m = odd ? min_gate[2 * v + 1 < N ? 2 * v + 1 : 2 * v] : min_gate[2 * v];
                // (d_a d) dot - (d_a dmin) minimum, each product rounded: the order of the reference's primitive
                const float left = packed_scale[v] * weight_scale * (float)t;
                const float right = packed_scale[v] * weight_minimum * (float)m;
                value = left - right;
            } else {
                value = weight_scale * packed_scale[v] * (float)t;
            }
            // every lane parks its term (lanes past the last row group park zeros nobody adds)
            lds_store_u32(park_at, __float_as_uint(value));
            park_at += 256u;
        }
      }
      }
      flush(window_begin, window_end - window_begin, begin);
      window_begin = window_end;
    }

    // ---- the end of a fused chunk: SwiGLU of the (gate, up) row sums, coalesced stores ----
    if constexpr (FUSED) {
        const unsigned chunk_rows = (finish - begin) << g.row_shift, chunk_row = row_begin + (begin << g.row_shift);
        // (consecutive lanes: consecutive rows. A chunk's rows are numbered as if it were whole, which takes no division: 298
        // -> 296 us of a launch of 32 rows, another 3 by the flush above; the Q4_K sweeps have no registers for either)
        const unsigned row_bits = chunk_shift + g.row_shift;
        const unsigned outputs = Q4 ? chunk_rows * (unsigned)N : (unsigned)N << row_bits;
        for (unsigned o = lane; o < outputs; o += 64u) {
            const unsigned p = Q4 ? o / chunk_rows : o >> row_bits;
            const unsigned local = Q4 ? o % chunk_rows : o & ((1u << row_bits) - 1u);
            if (!Q4 && local >= chunk_rows) continue;
            const float first = __uint_as_float(lds_load_u32(g.results + (p * kFusedItemRows + local) * 4u));
            const float second = __uint_as_float(
                lds_load_u32(g.results + (((unsigned)N + p) * kFusedItemRows + local) * 4u));
            const uint2 info = lds_load_uint2(g.park + kInfoOffset + 8u * p);
            const float value = swiglu_bf16_fast(first, second, __uint_as_float(info.y), a.limit, (float)a.limit);
            if (!finite_f32(value)) raise_status(a.status, 1);
            else pr.out[(unsigned long long)info.x * a.out_rows + chunk_row + local] = value;
        }
        wave_lds_fence();
    }
    if (next >= chunks) return drawn;
    begin = next << chunk_shift;
    }
}

__device__ __forceinline__ unsigned uniform(unsigned v)
{
    return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ unsigned long long uniform64(unsigned long long v)
{
    return ((unsigned long long)uniform((unsigned)(v >> 32)) << 32) | uniform((unsigned)v);
}

template <int MODE, bool IMAGE, unsigned QT>
__global__ __launch_bounds__(kSweepThreads) void iq2_sweep_kernel(GroupedArgs a)
{
    constexpr bool FUSED = MODE == 1;
    extern __shared__ __align__(16) unsigned char sweep_lds[];
    if (lds_address_of(sweep_lds) != 0u) {   // the lookups address LDS by absolute byte offsets
        if (threadIdx.x == 0u) raise_status(a.status, 2);
        return;
    }
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = uniform(tid >> 6);
    const GroupedProblem &routed = a.problem[0];
    const bool routed_fixed = routed.expert_ids == nullptr;
    const bool pairs_in_lds = !routed_fixed && routed.order != nullptr && routed.pairs <= kPairCacheMax;
    static_assert(kPairCacheMax <= 2u * kSweepThreads, "two cached pairs a thread");
    // ---- what opens the launch. Everything is requested before any of it is used: the tables' digits by the waves that
    // form the codebook entries, the routed buckets (four a lane) by the wave that finds the workgroup's piece, the
    // pairs' sources by all; the sign entries need nothing and are stored meanwhile. Every wave used to find the piece, with
    // divisions, and to fill its part of the tables behind that: 5.7 us to the first sweep of a gate/up launch and 4.9 of a
    // down launch of one row, 4.6 and 4.0 now, of which 2.3 pass before the buckets are there; launches of one row over IQ2_XXS
    // and Q2_K 18.6 and 11.7 -> 18.1 and 11.3 us, of 96 rows 257 -> 254. (A second wave for the piece's end is another 0.5 us,
    // but costs the loops their registers: Q4_K 434 -> 454.) ----
    unsigned digits = 0u;
    if constexpr (QT == QT_IQ2_XXS) {                                 // (the other formats need no tables)
        if (wave < 4u) digits = sweep_table_digits();
    }
    const bool placing = wave == kPlacingWave;
    unsigned long long bucket_count = 0ull, population64[4], expert64[4], first64[4];
    if (placing) {
        bucket_count = routed_fixed ? 1ull : routed.counts[0];
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) {
            const unsigned slot = 4u * lane + j;
            population64[j] = routed_fixed ? (slot == 0u ? routed.pairs : 0ull) : 0ull;
            expert64[j] = first64[j] = 0ull;
            if (!routed_fixed && slot < routed.experts) {
                population64[j] = routed.bucket_populations[slot];
                expert64[j] = routed.expert_ids[slot];
                first64[j] = routed.bucket_offsets[slot];
            }
        }
    }
    unsigned long long source_here[2] = {~0ull, ~0ull};
    if (pairs_in_lds) {
#pragma unroll
        for (unsigned k = 0; k < 2u; ++k)
            if (tid + k * kSweepThreads < routed.pairs) source_here[k] = routed.order[tid + k * kSweepThreads];
    }
    if constexpr (QT == QT_IQ2_XXS) {
        if (wave >= 4u) sweep_signs_fill();
    }
    if (tid == 0u) lds_store_u32(kTicketAddress, 0u);

    // (shifts and comparisons: a division by a number that only the launch knows is forty dependent instructions)
    SweepLane g;
    g.lanes_per_row = a.width >> 7;                                // 16 .. 64, checked on the host
    g.row_shift = g.lanes_per_row == 16u ? 2u : g.lanes_per_row == 32u ? 1u : 0u;
    g.rows_per_iter = 1u << g.row_shift;
    g.sub = (lane >= g.lanes_per_row ? 1u : 0u) + (lane >= 2u * g.lanes_per_row ? 1u : 0u) +
            (lane >= 3u * g.lanes_per_row ? 1u : 0u);
    const unsigned seg = lane - g.sub * g.lanes_per_row;
    g.live = g.sub < g.rows_per_iter;
    g.super = seg >> 1;
    g.half = seg & 1u;
    // superblock `super` starts 66 * super bytes into a row whose start is dword-aligned
    const unsigned block_start = 66u * (g.live ? g.super : 0u);
    g.code_shift = (block_start + 2u + 32u * g.half) & 3u;
    g.scale_shift = 8u * (block_start & 3u);
    g.mag_lane = (lane & 15u) * 16u;
    g.sel_lane = kSelBase + (lane & 31u) * 8u;
    g.park = kParkBase + (tid >> 6) * kParkBytes;      // (in a vector register: the window's stores lose their immediate offsets otherwise)
    g.results = g.park + kWindowBytes;
    g.terms = g.lanes_per_row / 2u;
    {
        // a line of the window: parity, then the rows of an iteration, then the row's superblocks
        const unsigned span_shift = 6u - g.row_shift, span = 64u >> g.row_shift;      // lanes of a weight row's slot
        g.term_slot = ((lane & 1u) * 32u + (lane >> span_shift) * (span / 2u) + (lane & (span - 1u)) / 2u) * 4u;
    }
    const unsigned turn_shift = g.row_shift + (MODE == 2 ? 1u : 0u), turn_rows = 1u << turn_shift;
    const GroupedProblem &extra = a.problem[a.problems > 1u ? 1u : 0u];
    const unsigned extra_pairs = a.problems > 1u ? extra.pairs : 0u;
    struct Place {
        unsigned slot, sweep, row;
    };

    // ---- the launch's work and this workgroup's piece of it, by one wave ----
    // Slot 0 is the shared expert (no rows of its own when there is none), slot 1 + b bucket b. A
    // slot of n pairs has n / 4 sweeps of four pairs and one of what is left. The prefix sums of cost and sweeps over the
    // slots are a scan across the wave's 64 lanes, four slots each, no barrier and no LDS. (It was a list of all sweeps
    // sorted by their pairs, built by the workgroup in LDS behind two barriers: 2.5 us of every launch's first 8.5.)
    unsigned warm[2] = {0u, 0u};
    if (placing) {
        const unsigned extra_cost = bucket_cost<QT>(extra_pairs), extra_sweeps = (extra_pairs + 3u) / 4u;
        const unsigned buckets = (unsigned)bucket_count;
        unsigned population[4], cost_here = 0u, sweeps_here = 0u;
        bool bad = bucket_count > 256ull;
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) {
            const bool live = 4u * lane + j < bucket_count;
            bad |= live && (population64[j] > routed.pairs || expert64[j] >= routed.experts || first64[j] > routed.pairs);
            population[j] = live ? (unsigned)population64[j] : 0u;
            cost_here += bucket_cost<QT>(population[j]);
            sweeps_here += (population[j] + 3u) / 4u;
        }
        const unsigned all_pairs = (unsigned)group_sum_i32<64>((int)(population[0] + population[1] + population[2] + population[3]));
        // (the launch wrapper bounds the pairs, and with them what the packed sums below can hold)
        const bool refused = __ballot(bad) != 0ull || all_pairs > routed.pairs || routed.pairs + extra_pairs > kMaxSweeps;
        if (refused) {
            if (lane == 0u) raise_status(a.status, 2);
            lds_store_uint4(kPlaceAddress, make_uint4(0u, 0u, 0u, 1u));
        } else {
            static_assert(kMaxSweeps * sweep_cost<QT>(4u) < 65536u, "a prefix is two 16-bit sums");
            const unsigned packed = (sweeps_here << 16) | cost_here;
            const unsigned inclusive = wave_inclusive_sum_u32(packed);
            const unsigned before = inclusive - packed;
            const unsigned totals = (unsigned)__builtin_amdgcn_readlane((int)inclusive, 63);
            const unsigned row_cost = extra_cost + (totals & 0xffffu), all_sweeps = extra_sweeps + (totals >> 16);
#pragma unroll
            for (unsigned j = 0; j < 4u; ++j)
                lds_store_uint4(kBucketBase + 16u * (4u * lane + j),
                                make_uint4((unsigned)expert64[j], (unsigned)first64[j], population[j], 0u));

            const unsigned granule = 2u * turn_rows;                   // the ring turns twice a trip through its loop
            // iterations of a piece: a batch of a few rows leaves a wave a handful of them, and is cut finely
            const unsigned piece_turns = uniform((unsigned)((float)all_sweeps * (float)(a.out_rows >> turn_shift) *
                                                            __builtin_amdgcn_rcpf((float)gridDim.x)));
            // (integer arithmetic on the scalar unit; any share does whose pieces do not reach past the end)
            const unsigned long long all_cost = (unsigned long long)row_cost * a.out_rows;
            const unsigned long long share = (gridDim.x & (gridDim.x - 1u)) == 0u
                ? all_cost >> (31 - __builtin_clz(gridDim.x)) : uniform64((unsigned long long)((double)all_cost / (double)gridDim.x));
            const unsigned long long left_over = all_cost - share * gridDim.x;
            auto place_of = [&](unsigned who) -> Place {        // where the piece of workgroup `who` begins
                if (who >= gridDim.x) return Place{buckets + 1u, 0u, 0u};
                unsigned long long at = share * who + (who < left_over ? who : left_over);
                unsigned slot = 0u, n = extra_pairs;
                if (at >= (unsigned long long)extra_cost * a.out_rows) {
                    at -= (unsigned long long)extra_cost * a.out_rows;
                    const unsigned long long below = __ballot((unsigned long long)(before & 0xffffu) * a.out_rows <= at);
                    const int holder = 63 - __builtin_clzll(below);
                    at -= (unsigned long long)((unsigned)__builtin_amdgcn_readlane((int)before, holder) & 0xffffu) * a.out_rows;
                    slot = 4u * (unsigned)holder + 1u;
                    n = (unsigned)__builtin_amdgcn_readlane((int)population[0], holder);
#pragma unroll
                    for (unsigned j = 1; j < 4u; ++j) {
                        const unsigned long long rows = (unsigned long long)bucket_cost<QT>(n) * a.out_rows;
                        const unsigned behind = (unsigned)__builtin_amdgcn_readlane((int)population[j], holder);
                        if (slot == 4u * (unsigned)holder + j && at >= rows) {
                            at -= rows;
                            ++slot;
                            n = behind;
                        }
                    }
                }
                const unsigned full = n / 4u;
                const unsigned sweep_rows = sweep_cost<QT>(4u) * a.out_rows;
                unsigned sweep = 0u;
                if (full) {
                    // (a quotient of at most kMaxSweeps / 4: out by one at most)
                    sweep = uniform((unsigned)((float)at * __builtin_amdgcn_rcpf((float)sweep_rows)));
                    if ((unsigned long long)sweep * sweep_rows > at) --sweep;
                    if ((unsigned long long)(sweep + 1u) * sweep_rows <= at) ++sweep;
                    if (sweep > full) sweep = full;
                    at -= (unsigned long long)sweep * sweep_rows;
                }
                const unsigned rest = (unsigned)at;
                unsigned row = sweep < full ? rest / sweep_cost<QT>(4u)
                    : n % 4u == 1u ? rest / sweep_cost<QT>(1u) : n % 4u == 2u ? rest / sweep_cost<QT>(2u)
                                                                             : rest / sweep_cost<QT>(3u);
                if (row > a.out_rows) row = a.out_rows;
                return Place{uniform(slot), uniform(sweep), uniform(row & ~(granule - 1u))};
            };
            Place now{}, end{};
#pragma unroll 1
            for (unsigned ends = 0; ends < 2u; ++ends) {      // (the code of one, run twice)
                now = end;
                end = place_of(blockIdx.x + ends);
            }
            lds_store_uint4(kPlaceAddress, make_uint4(now.slot, now.sweep, now.row, 0u));
            lds_store_uint4(kPlaceAddress + 16u, make_uint4(end.slot, end.sweep, end.row, piece_turns));

            // The first weight rows of the piece start on their way to the caches (64 bytes apart, so the lanes cover
            // 4 KB of each stream).
            if (now.slot <= buckets) {
                const unsigned bucket = now.slot ? now.slot - 1u : 0u;
                unsigned expert = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)expert64[0], (int)(bucket >> 2));
#pragma unroll
                for (unsigned j = 1; j < 4u; ++j) {
                    const unsigned other = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)expert64[j], (int)(bucket >> 2));
                    if ((bucket & 3u) == j) expert = other;
                }
                const GroupedProblem &pr = a.problem[now.slot == 0u ? a.problems - 1u : 0u];
                if (now.slot == 0u) expert = 0u;
                const unsigned rows_left = a.out_rows - now.row;
                unsigned long long offset = 64ull * lane;
                const unsigned long long bytes_left = rows_left * pr.row_bytes;
                if (bytes_left >= 8ull) {
                    if (offset + 4ull > bytes_left) offset = bytes_left - 4ull;
                    const unsigned char *rows = pr.gate + expert * pr.expert_bytes + now.row * pr.row_bytes;
                    warm[0] = *reinterpret_cast<const unsigned *>(rows + (offset & ~3ull));
                    if (FUSED) {
                        warm[1] = *reinterpret_cast<const unsigned *>(pr.up + expert * pr.up_expert_bytes +
                                                                      now.row * pr.up_row_bytes + (offset & ~3ull));
                    } else if (offset + 4096ull + 4ull <= bytes_left) {
                        warm[1] = *reinterpret_cast<const unsigned *>(rows + 4096u + (offset & ~3ull));
                    }
                }
            }
        }
    }
    if constexpr (QT == QT_IQ2_XXS) {
        if (wave < 4u) sweep_levels_fill(digits);
    }
    if (pairs_in_lds) {
        float weight_here[2];
#pragma unroll
        for (unsigned k = 0; k < 2u; ++k)   // a source outside the problem reads no weight here; the sweep's own checks refuse it
            weight_here[k] = routed.route_weights && source_here[k] < routed.pairs
                ? routed.route_weights[source_here[k]] : 1.0f;
#pragma unroll
        for (unsigned k = 0; k < 2u; ++k)
            if (tid + k * kSweepThreads < routed.pairs)
                lds_store_uint2(kPairCacheBase + 8u * (tid + k * kSweepThreads),
                                make_uint2(source_here[k] < 0xffffffffull ? (unsigned)source_here[k] : 0xffffffffu,
                                           __float_as_uint(weight_here[k])));
    }
    // (LDS traffic only: the warming loads may still be on their way)
    lds_barrier();
    const uint4 first_place = lds_read_uint4(kPlaceAddress), last_place = lds_read_uint4(kPlaceAddress + 16u);
    if (uniform(first_place.w)) return;                               // refused
    Place now{uniform(first_place.x), uniform(first_place.y), uniform(first_place.z)};
    const Place end{uniform(last_place.x), uniform(last_place.y), uniform(last_place.z)};
    const unsigned piece_turns = uniform(last_place.w);
    // A wave holds one chunk and has drawn the next, and waves of a launch end 10 to 15 % apart, so short chunks are the
    // better ones until their ends cost more. A chunk of a plain projection ends in a flush: four turns (of 32 rows, IQ2_XXS
    // 151.5 us with eight turns, 148.9 with four, 153.4 with two; of 23 rows Q4_K 234.3, 229.5, 236.1; of 96 rows Q2_K 154.5,
    // 152.5, 163.4). One of gate and up rows ends in the SwiGLU as well: sixteen turns of one pair and eight of
    // more (32 rows: 293 us; eight of any 305; four 316; sixteen of any 299), of Q4_K eight (429; 433 with sixteen of one pair).
    auto chunk_shift_of = [&](unsigned n) -> unsigned {
        unsigned shift = !FUSED ? kSweepChunkShift - 2u : QT == QT_Q4_K || n >= 2u ? kSweepChunkShift - 1u : kSweepChunkShift;
        while (shift > 1u && ((4u * kSweepWaves << shift) > piece_turns || (FUSED && (turn_rows << shift) > kFusedItemRows)))
            --shift;
        return shift;
    };
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" ::"v"(warm[0]), "v"(warm[1]));
#endif

    // ---- the piece: its sweeps one after another, each with the chunks of its rows ----
    unsigned drawn = draw_chunk(), base = 0u;
    while (now.slot < end.slot || (now.slot == end.slot &&
                                   (now.sweep < end.sweep || (now.sweep == end.sweep && now.row < end.row)))) {
        const unsigned slot = now.slot, sweep = now.sweep, row_begin = now.row;
        const bool last = slot == end.slot && sweep == end.sweep;
        const unsigned row_end = last ? end.row : a.out_rows;
        const bool is_routed = slot != 0u;
        const GroupedProblem &pr = a.problem[!is_routed && a.problems > 1u ? 1u : 0u];
        unsigned long long expert = 0ull, first = 0ull;
        unsigned n = extra_pairs;
        if (is_routed) {
            const uint4 bucket = lds_read_uint4(kBucketBase + 16u * (slot - 1u));
            expert = uniform(bucket.x);
            first = uniform(bucket.y);
            n = uniform(bucket.z);
        }
        now.row = 0u;
        if ((sweep + 1u) * 4u < n) {
            ++now.sweep;
        } else {
            now.sweep = 0u;
            ++now.slot;
        }
        if (last) now = end;
        const unsigned pass = sweep * (unsigned)kSweepPairs;
        if (pass >= n || row_begin >= row_end) continue;
        if (first + n > pr.pairs) {
            if (lane == 0u) raise_status(a.status, 2);
            continue;
        }
        const unsigned live = n - pass < 4u ? n - pass : 4u;
        const unsigned chunk_shift = chunk_shift_of(live), rows_shift = chunk_shift + turn_shift;
        const unsigned chunks = (row_end - row_begin + (1u << rows_shift) - 1u) >> rows_shift;
        if (drawn - base < chunks) {
            const unsigned char *gate_e = pr.gate + expert * pr.expert_bytes;
            const unsigned char *up_e = FUSED ? pr.up + expert * pr.up_expert_bytes : nullptr;
            const bool cached = pairs_in_lds && is_routed;
            const unsigned chunk = drawn - base;
            static_assert(kSweepPairs == 4, "a sweep serves one to four pairs");
            if (live == 4u)
                drawn = iq2_sweep<MODE, 4, IMAGE, QT>(a, pr, g, gate_e, up_e, first + pass, row_begin, row_end, cached, chunk, base, chunk_shift);
            else if (live == 3u)
                drawn = iq2_sweep<MODE, 3, IMAGE, QT>(a, pr, g, gate_e, up_e, first + pass, row_begin, row_end, cached, chunk, base, chunk_shift);
            else if (live == 2u)
                drawn = iq2_sweep<MODE, 2, IMAGE, QT>(a, pr, g, gate_e, up_e, first + pass, row_begin, row_end, cached, chunk, base, chunk_shift);
            else
                drawn = iq2_sweep<MODE, 1, IMAGE, QT>(a, pr, g, gate_e, up_e, first + pass, row_begin, row_end, cached, chunk, base, chunk_shift);
        }
        base += chunks;
    }
}

bool iq2_sweep_supported(unsigned qtype, unsigned width, unsigned out_rows, unsigned long long pairs, bool image)
{
    if (qtype != QT_IQ2_XXS && qtype != QT_Q4_K && qtype != QT_Q2_K) return false;
    if (image && qtype != QT_IQ2_XXS) return false;
    if (pairs > kMaxSweeps) return false;            // every sweep serves at least one pair
    const unsigned lanes_per_row = width / 128u;
    if (width % 256u != 0u || lanes_per_row < 16u || lanes_per_row > 64u) return false;
    // IQ2_XXS rows must start on dword boundaries (Q4_K rows are multiples of 144 bytes, Q2_K rows of 84)
    if (qtype == QT_IQ2_XXS && !image && (width / 256u * 66u) % 4u != 0u) return false;
    const unsigned rows_per_iter = lanes_per_row % 16u == 0u && 64u % lanes_per_row == 0u
        ? 64u / lanes_per_row : 1u;
    return out_rows % rows_per_iter == 0u;   // an iteration never reads past the last row
}

template <int MODE, bool IMAGE, unsigned QT>
static int launch_iq2_sweep_variant(const GroupedArgs &a, hipStream_t stream)
{
    YVEX_ALLOW_DYNAMIC_LDS((iq2_sweep_kernel<MODE, IMAGE, QT>), kSweepLdsBytes);
    iq2_sweep_kernel<MODE, IMAGE, QT><<<compute_units(), kSweepThreads, kSweepLdsBytes, stream>>>(a);
    return check_launch("moe_sweep");
}

template <bool IMAGE, unsigned QT>
static int launch_iq2_sweep_mode(const GroupedArgs &a, int mode, hipStream_t stream)
{
    return mode == 1 ? launch_iq2_sweep_variant<1, IMAGE, QT>(a, stream)
         : mode == 2 ? launch_iq2_sweep_variant<2, IMAGE, QT>(a, stream)
                     : launch_iq2_sweep_variant<0, IMAGE, QT>(a, stream);
}

int launch_iq2_sweep(const GroupedArgs &a, unsigned qtype, bool fused, bool image, hipStream_t stream)
{
    // a projection that is not fused takes two row groups an iteration where the rows allow it
    // (every item then holds whole pairs of groups: the short items are half a long one)
    const unsigned lanes_per_row = a.width / 128u;
    const unsigned rows_per_iter = lanes_per_row % 16u == 0u && 64u % lanes_per_row == 0u ? 64u / lanes_per_row : 1u;
    const int mode = fused ? 1 : a.out_rows % (2u * rows_per_iter) == 0u ? 2 : 0;
    if (qtype == QT_Q4_K) return image ? ST_UNSUPPORTED : launch_iq2_sweep_mode<false, QT_Q4_K>(a, mode, stream);
    if (qtype == QT_Q2_K) {      // the down experts: a plain projection
        if (image || fused) return ST_UNSUPPORTED;
        return mode == 2 ? launch_iq2_sweep_variant<2, false, QT_Q2_K>(a, stream)
                         : launch_iq2_sweep_variant<0, false, QT_Q2_K>(a, stream);
    }
    if (qtype != QT_IQ2_XXS) return ST_UNSUPPORTED;
    return image ? launch_iq2_sweep_mode<true, QT_IQ2_XXS>(a, mode, stream)
                 : launch_iq2_sweep_mode<false, QT_IQ2_XXS>(a, mode, stream);
}

// ---- the image: canonical IQ2_XXS superblocks re-packed for the sweeps -------------------------

// One thread per half superblock: nine dwords out of the 66 canonical bytes.
__global__ __launch_bounds__(256) void iq2_sweep_image_kernel(const unsigned char *canonical,
                                                              unsigned long long blocks, unsigned *image)
{
    const unsigned long long at = (unsigned long long)blockIdx.x * 256ull + threadIdx.x;
    if (at >= 2ull * blocks) return;
    const unsigned long long block = at >> 1;
    const unsigned half = (unsigned)(at & 1ull);
    const unsigned char *b = canonical + block * 66ull;
    unsigned *record = image + at * 9ull;
    unsigned scales = 0u;
#pragma unroll
    for (unsigned j = 0; j < 4u; ++j) {
        const unsigned char *group = b + 2u + 8u * (4u * half + j);
        const unsigned grids = load_u32(group), aux = load_u32(group + 4u);
        record[1u + 2u * j] = grids;
        record[2u + 2u * j] = (aux & 127u) | (((aux >> 7) & 127u) << 8) | (((aux >> 14) & 127u) << 16) |
                              (((aux >> 21) & 127u) << 24);
        scales |= (aux >> 28) << (4u * j);
    }
    record[0] = load_u16(b) | (scales << 16);
}

}  // namespace yvex

extern "C" uint64_t yvex_hip_iq2_sweep_image_bytes(uint64_t blocks) { return blocks * 72u; }

extern "C" int yvex_hip_iq2_sweep_image_build(const uint8_t *canonical, uint64_t blocks, void *image,
                                              yvex_hip_stream stream)
{
    if (!canonical || !image || !blocks || ((uintptr_t)image & 3u)) return yvex::ST_INVALID_ARG;
    const uint64_t groups = (2u * blocks + 255u) / 256u;
    if (groups > 0x7fffffffull) return yvex::ST_BOUNDS;
    yvex::iq2_sweep_image_kernel<<<(unsigned)groups, 256, 0, yvex::as_stream(stream)>>>(canonical, blocks,
                                                                                         (unsigned *)image);
    return yvex::check_launch("iq2_sweep_image");
}
