// Q4_K weight rows against a batch of Q8_K input rows on the int8 matrix cores: the dense
// projection at prefill width (16 input rows and more; the reference turns its tensor-core
// kernels on there, src/backend/cuda/private.h:461-464).
//
// Arithmetic, per 256-value superblock (public ggml block_q4_K against the Q8_K block of
// src/backend/cuda/kernel_primitives.h:274-312, in the shape of the reference's Q2_K primitive,
// kernel_primitives.h:314-341):
//     dot     = sum_j sc_j * sum_{i in sub-block j} nibble_i * a_i        (int32, exact)
//     minimum = sum_j m_j  * (bsums[2j] + bsums[2j+1])                    (int32, exact)
//     value   = (d_a * d) * float(dot) - (d_a * dmin) * float(minimum)    (two products, one subtraction)
// and the superblock values of a row are added in double and rounded to float once, as the
// CPU path adds a row's blocks (src/gguf/quant_compute.c:152-172).
//
// A 32-value sub-block is exactly the reduction depth of V_MFMA_I32_32X32X32_I8. The weight
// operand carries sc_j * nibble (at most 63 * 15 = 945) as two int8 limbs, value = 8 hi + lo
// with lo = (sc_j mod 8) * nibble and hi = (sc_j div 8) * nibble, both at most 105, so each
// sub-block costs two matrix instructions per 32 tokens and the int32 accumulators run over the
// whole superblock without rescaling. The minimum term is one K step of an f16 instruction whose float
// sums are exact (kquant_limbs.hpp); on the 16 x 16 tiles it is one more reduction of depth 8, the m_j against the pair sums
// of bsums in two limbs of base 128, through the int8 instruction. Products of the scales are outer products on
// the matrix cores (rows_q4k.hip), on the 16 x 16 tiles multiplications.
//
// A workgroup owns 32 weight rows x 32 or 64 tokens; its four waves take every fourth
// superblock and their double-precision partial tiles are added in wave order, so results do not depend on
// timing. Lane (r, h) of a wave holds bytes 16h..16h+15 of weight row r's sub-block as the A
// operand and the same bytes of token r's activations as the B operand; accumulator i of that
// lane is weight row 8 (i / 4) + 4 h + i % 4 against token r.
#include "common.hpp"
#include "launch.hpp"
#include "grouped.hpp"
#include "publish.hpp"
#include "kquant_limbs.hpp"

namespace yvex {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct DenseQ4kArgs {
    const unsigned char *encoded;
    unsigned long long row_count, row_bytes;
    unsigned blocks;                         // superblocks per row
    const unsigned char *act;                // Q8_K rows, blocks * 292 bytes each
    unsigned long long input_rows;
    const float *additive;
    float *out;
    unsigned long long out_stride;
    int output_bf16;
    int *status;
    Publication publication;
};

// What one wave needs of one superblock: the weight row's block and NT token blocks.
template <unsigned NT>
struct SuperInputs {
    unsigned head;          // f16 d | f16 dmin << 16
    uint3 scales;           // the 12 scale bytes
    uint4 qs[4];            // this lane's 16 bytes of each 32-byte nibble group
    float act_scale[NT];
    uint4 a[NT][8];         // this lane's 16 bytes of each sub-block's activations
    uint4 bsums[NT][2];     // the 16 int16 sums of 16 activations each
};

template <unsigned NT>
__device__ __forceinline__ void load_super(const DenseQ4kArgs &g, const unsigned char *wrow,
                                           const unsigned char *const (&arow)[NT], unsigned sb,
                                           unsigned h, SuperInputs<NT> &in)
{
    const unsigned char *w = wrow + (unsigned long long)sb * 144ull;
    in.head = *reinterpret_cast<const unsigned *>(w);
    in.scales = *reinterpret_cast<const uint3 *>(w + 4u);
#pragma unroll
    for (unsigned j = 0; j < 4u; ++j) in.qs[j] = *reinterpret_cast<const uint4 *>(w + 16u + 32u * j + 16u * h);
#pragma unroll
    for (unsigned nt = 0; nt < NT; ++nt) {
        const unsigned char *a = arow[nt] + (unsigned long long)sb * kQ8KBytes;
        in.act_scale[nt] = *reinterpret_cast<const float *>(a);
#pragma unroll
        for (unsigned c = 0; c < 8u; ++c) {
            // the activation bytes start 4 bytes into the block: dword-aligned, read as dwords
            const unsigned *p = reinterpret_cast<const unsigned *>(a + 4u + 32u * c + 16u * h);
            in.a[nt][c] = make_uint4(p[0], p[1], p[2], p[3]);
        }
        const unsigned *b = reinterpret_cast<const unsigned *>(a + 260u);
        in.bsums[nt][0] = make_uint4(b[0], b[1], b[2], b[3]);
        in.bsums[nt][1] = make_uint4(b[4], b[5], b[6], b[7]);
    }
    (void)g;
}

// q4k_limbs of a whole scale. (Its two parts as arguments leave the registers of two workgroups a compute unit worse off:
// 4096 x 4096 by 150 rows 35.3 -> 37.4 us, 2048 x 7168 by 300 54.1 -> 59.1.)
__device__ __forceinline__ void limbs(unsigned x, unsigned sc, unsigned &lo, unsigned &hi)
{
    const unsigned nibbles = x & 0x0f0f0f0fu;
    const unsigned low = (sc & 7u) * 0x00010001u, high = ((sc >> 3) & 7u) * 0x00010001u;
    lo = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * __builtin_bit_cast(u16x2, low));
    hi = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, nibbles) * __builtin_bit_cast(u16x2, high));
}

__device__ __forceinline__ v4i as_v4i(uint4 v)
{
    v4i r = {(int)v.x, (int)v.y, (int)v.z, (int)v.w};
    return r;
}

// A workgroup that has its compute unit to itself requests a superblock ahead, on as many registers as that takes; where 64-token
// tiles outnumber the compute units (PAIRED) two of them share one on half the registers and cover each other's loads. us a
// call one way and the other (tiles_share_units has the line): 7168 x 2048 by 120 rows 36.3 and 29.0, 4096 x 4096 by 150 42.4 and 36.1, 2048 x 7168 by 300 57.9 and
// 55.3; with a tile a compute unit or fewer 2048 x 7168 by 200 37.0 and 45.2, 4096 x 4096 by 96 30.0 and 32.4, 1024 x 4096 by 300 30.4 and 33.4.
template <unsigned NT, bool PAIRED = false>
__global__ __launch_bounds__(256, NT == 1u || PAIRED ? 2 : 1) void dense_q4k_kernel(DenseQ4kArgs g)
{
    __shared__ double partial[3][NT][16][64];
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned r = lane & 31u, h = lane >> 5;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 32ull;
    const unsigned long long tok0 = (unsigned long long)blockIdx.y * (32ull * NT);
    unsigned long long wr = row0 + r;
    if (wr >= g.row_count) wr = g.row_count - 1ull;              // a ragged edge repeats the last row
    const unsigned char *wrow = g.encoded + wr * g.row_bytes;
    const unsigned char *arow[NT];
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;
#pragma unroll
    for (unsigned nt = 0; nt < NT; ++nt) {
        unsigned long long t = tok0 + 32ull * nt + r;
        if (t >= g.input_rows) t = g.input_rows - 1ull;
        arow[nt] = g.act + t * act_row_bytes;
    }
    double acc[NT][16];
#pragma unroll
    for (unsigned nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[nt][i] = 0.0;

    SuperInputs<NT> cur;
    if (wave < g.blocks) load_super<NT>(g, wrow, arow, wave, h, cur);
    for (unsigned sb = wave; sb < g.blocks; sb += 4u) {
        // the next superblock's bytes travel while this one is worked on
        SuperInputs<NT> nxt;
        const unsigned ahead = sb + 4u < g.blocks ? sb + 4u : sb;
        load_super<NT>(g, wrow, arow, ahead, h, nxt);
        if (!PAIRED) __builtin_amdgcn_sched_barrier(0);      // (they would be requested where they are used)

        // scales and minima of the eight sub-blocks, four to a dword (ggml get_scale_min_k4)
        const unsigned s0 = cur.scales.x, s1 = cur.scales.y, s2 = cur.scales.z;
        const unsigned sc_pack[2] = {s0 & 0x3f3f3f3fu, (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)};
        const unsigned mn_pack[2] = {s1 & 0x3f3f3f3fu, ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)};
        v16i lo_sum[NT], hi_sum[NT];
#pragma unroll
        for (unsigned nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) lo_sum[nt][i] = hi_sum[nt][i] = 0;
#pragma unroll
        for (unsigned c = 0; c < 8u; ++c) {
            const unsigned sc = (sc_pack[c >> 2] >> (8u * (c & 3u))) & 255u;
            const uint4 q = cur.qs[c >> 1];
            const unsigned shift = (c & 1u) * 4u;
            v4i a_lo, a_hi;
            unsigned lo, hi;
            limbs(q.x >> shift, sc, lo, hi); a_lo[0] = (int)lo; a_hi[0] = (int)hi;
            limbs(q.y >> shift, sc, lo, hi); a_lo[1] = (int)lo; a_hi[1] = (int)hi;
            limbs(q.z >> shift, sc, lo, hi); a_lo[2] = (int)lo; a_hi[2] = (int)hi;
            limbs(q.w >> shift, sc, lo, hi); a_lo[3] = (int)lo; a_hi[3] = (int)hi;
#pragma unroll
            for (unsigned nt = 0; nt < NT; ++nt) {
                const v4i b = as_v4i(cur.a[nt][c]);
                lo_sum[nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_lo, b, lo_sum[nt], 0, 0, 0);
                hi_sum[nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_hi, b, hi_sum[nt], 0, 0, 0);
            }
        }
        // minimum term and products of the scales as in rows_q4k.hip: a K step on f16 operands whose float sums are exact, and two
        // outer products (d on the lanes of half 0, dmin on the others)
        const f16x8 m_op = bytes_to_f16(mn_pack[0], mn_pack[1]);
        const float row_scale = f16_bits_to_float(cur.head >> (16u * h) & 0xffffu);
#pragma unroll
        for (unsigned nt = 0; nt < NT; ++nt) {
            v16f zero16;
            v32f zero32;
#pragma unroll
            for (int i = 0; i < 16; ++i) zero16[i] = zero32[i] = zero32[i + 16] = 0.0f;
            const v16f minimum = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                m_op, q4k_bsum_operand(cur.bsums[nt][0], cur.bsums[nt][1], h), zero16, 0, 0, 0);
            const v32f scale = __builtin_amdgcn_mfma_f32_32x32x1f32(row_scale, cur.act_scale[nt], zero32, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int dot = (hi_sum[nt][i] << 3) + lo_sum[nt][i];
                const float left = scale[i] * (float)dot;
                const float right = scale[i + 16] * minimum[i];
                acc[nt][i] += (double)(left - right);
            }
        }
        cur = nxt;
    }

    if (wave) {
#pragma unroll
        for (unsigned nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) partial[wave - 1u][nt][i][lane] = acc[nt][i];
    }
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (unsigned nt = 0; nt < NT; ++nt) {
        const unsigned long long token = tok0 + 32ull * nt + r;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const unsigned long long row = row0 + 8u * (i >> 2) + 4u * h + (i & 3);
            const float sum = (float)(((acc[nt][i] + partial[0][nt][i][lane]) + partial[1][nt][i][lane]) +
                                      partial[2][nt][i][lane]);
            if (row >= g.row_count || token >= g.input_rows) continue;
            const unsigned long long at = token * g.out_stride + row;
            const float value = g.additive ? sum + g.additive[at] : sum;
            if (!finite_f32(value)) raise_status(g.status, 1);
            else g.out[at] = g.output_bf16 ? bf16_round(value) : value;
        }
    }
}

// LDS of a wave of the kernel below: 16 weight rows' superblock (144 bytes a row), 16 input rows' codes, sums and scale
// (256, 32 and 4 bytes of 304 a row, which spreads the rows over the banks).
constexpr unsigned kSmallWeights = 16u * 144u, kSmallActPitch = 304u, kSmallWindow = kSmallWeights + 16u * kSmallActPitch;

// The same product for few input rows on V_MFMA_I32_16X16X64_I8: a workgroup owns 16
// weight rows x 16 tokens, so a batch of 16 wastes no token slot and twice as many
// workgroups share the matrix; its waves take every eighth superblock, or every fourth. One K
// step is a 64-value nibble group, i.e. two sub-blocks, which is fine because the limbs already
// carry their sub-block's scale. Lane (r, q) holds bytes 16q..16q+15 of weight row r's group as
// the A operand (q = 0, 1: low nibbles of nibble bytes 16q.., the first sub-block; q = 2, 3:
// high nibbles of nibble bytes 16(q-2).., the second) and the same positions of token r's
// activations as the B operand; accumulator i of that lane is weight row 4 q + i against token r.
// Lanes that loaded their own pieces took twenty instructions of 16 to 32 cache lines a superblock, at two cycles
// a line 12 of the 14 us of 2048 x 7168 by 19. Loads take consecutive pieces of consecutive rows now, a superblock ahead,
// and the bytes pass through a window of LDS of the wave's own. 2048 x 7168 by 19 rows 13.6 -> 8.2 us, by 4
// 8.8 -> 7.7, 4096 x 4096 by 32 12.4 -> 9.2.
template <unsigned WAVES>
__global__ __launch_bounds__(64 * WAVES) void dense_q4k16_kernel(DenseQ4kArgs g)
{
    typedef int v4s __attribute__((ext_vector_type(4)));
    typedef int v4i_dword __attribute__((ext_vector_type(4), aligned(4)));
    constexpr unsigned kActPieces = 18u, kActLoads = (16u * kActPieces + 63u) / 64u;        // of 16 rows: 4.5 instructions
    __shared__ __align__(16) float row_scale[WAVES][2][16];
    __shared__ __align__(16) unsigned char windows[WAVES * kSmallWindow + 1024u];    // (and where lanes without a piece write)
    double (*const partial)[4][64] = reinterpret_cast<double (*)[4][64]>(windows);     // when the superblocks are done
    static_assert((WAVES - 1u) * 4u * 64u * sizeof(double) <= WAVES * kSmallWindow, "the partial tiles fit the windows");
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned r = lane & 15u, q = lane >> 4;
    const unsigned long long row0 = (unsigned long long)blockIdx.x * 16ull;
    const unsigned long long tok0 = (unsigned long long)blockIdx.y * 16ull;
    const unsigned rows_here = (unsigned)(g.row_count - row0 < 16ull ? g.row_count - row0 : 16ull);
    const unsigned toks_here = (unsigned)(g.input_rows - tok0 < 16ull ? g.input_rows - tok0 : 16ull);
    const unsigned long long act_row_bytes = (unsigned long long)g.blocks * kQ8KBytes;
    const unsigned char *const weights = g.encoded + row0 * g.row_bytes, *const acts = g.act + tok0 * act_row_bytes;
    unsigned char *const window = windows + wave * kSmallWindow, *const spare = windows + WAVES * kSmallWindow + 16u * lane;

    // the lane's pieces (a ragged edge repeats the last row) and their places in the window
    const unsigned char *weight_at[3], *act_at[kActLoads];
    unsigned char *act_to[kActLoads];
#pragma unroll
    for (unsigned k = 0; k < 3u; ++k) {
        const unsigned piece = k < 2u ? 64u * k + lane : 128u + r, row = piece / 9u;
        weight_at[k] = weights + (row < rows_here ? row : rows_here - 1u) * g.row_bytes + 16u * (piece - 9u * row);
    }
#pragma unroll
    for (unsigned k = 0; k < kActLoads; ++k) {
        const unsigned piece = 64u * k + lane, held = piece < 16u * kActPieces ? piece : 16u * kActPieces - 1u;
        const unsigned token = held / kActPieces, part = held - kActPieces * token;
        act_at[k] = acts + (token < toks_here ? token : toks_here - 1u) * act_row_bytes + 4u + 16u * part;
        act_to[k] = piece == held ? window + kSmallWeights + token * kSmallActPitch + 16u * part : spare;
    }
    const unsigned char *const scale_at = acts + (r < toks_here ? r : toks_here - 1u) * act_row_bytes;
    unsigned char *const scale_to = lane < 16u ? window + kSmallWeights + lane * kSmallActPitch + 288u : spare;
    struct {
        v4i weights[3], acts[kActLoads];
        unsigned scale;
    } ahead;
    auto request = [&](unsigned sb) {
        const unsigned long long w = sb * 144ull, a = (unsigned long long)sb * kQ8KBytes;
#pragma unroll
        for (unsigned k = 0; k < 3u; ++k) ahead.weights[k] = *reinterpret_cast<const v4i_dword *>(weight_at[k] + w);
#pragma unroll
            for (unsigned k = 0; k < kActLoads; ++k) ahead.acts[k] = *reinterpret_cast<const v4i_dword *>(act_at[k] + a);
        ahead.scale = *reinterpret_cast<const unsigned *>(scale_at + a);
    };

    double acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = 0.0;

    if (wave < g.blocks) request(wave);
    for (unsigned sb = wave; sb < g.blocks; sb += WAVES) {
        // (LDS operations of one wave complete in order)
#pragma unroll
        for (unsigned k = 0; k < 2u; ++k) *reinterpret_cast<v4i *>(window + 1024u * k + 16u * lane) = ahead.weights[k];
        *reinterpret_cast<v4i *>(window + 2048u + 16u * r) = ahead.weights[2];
#pragma unroll
        for (unsigned k = 0; k < kActLoads; ++k) *reinterpret_cast<v4i *>(act_to[k]) = ahead.acts[k];
        *reinterpret_cast<unsigned *>(scale_to) = ahead.scale;
        request(sb + WAVES < g.blocks ? sb + WAVES : sb);
        wave_lds_fence();
        const unsigned char *const w = window + 144u * r;
        const uint4 opening = *reinterpret_cast<const uint4 *>(w);
        const unsigned head = opening.x;
        uint4 qs[4];
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j)
            qs[j] = *reinterpret_cast<const uint4 *>(w + 16u + 32u * j + 16u * (q & 1u));
        uint4 a[4], bsums[2];
        float da;
        const unsigned char *ab = window + kSmallWeights + r * kSmallActPitch;
        da = *reinterpret_cast<const float *>(ab + 288u);
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) a[j] = *reinterpret_cast<const uint4 *>(ab + 64u * j + 16u * q);
        bsums[0] = *reinterpret_cast<const uint4 *>(ab + 256u);
        bsums[1] = *reinterpret_cast<const uint4 *>(ab + 272u);
        const unsigned s0 = opening.y, s1 = opening.z, s2 = opening.w;
        const unsigned sc_pack[2] = {s0 & 0x3f3f3f3fu, (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)};
        const unsigned mn_pack[2] = {s1 & 0x3f3f3f3fu, ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)};
        if (q == 0u) {
            row_scale[wave][0][r] = f16_bits_to_float(head & 0xffffu);
            row_scale[wave][1][r] = f16_bits_to_float(head >> 16);
        }
        v4s lo_sum, hi_sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) lo_sum[i] = hi_sum[i] = 0;
        const unsigned high = q >> 1;                          // this lane decodes the high nibbles
#pragma unroll
        for (unsigned j = 0; j < 4u; ++j) {
            // sub-block 2 j + high: its scale is byte (2 j + high) of the packed scales
            const unsigned sc = (sc_pack[j >> 1] >> (16u * (j & 1u) + 8u * high)) & 255u;
            const unsigned shift = 4u * high;
            v4i a_lo, a_hi;
            unsigned lo, hi;
            limbs(qs[j].x >> shift, sc, lo, hi); a_lo[0] = (int)lo; a_hi[0] = (int)hi;
            limbs(qs[j].y >> shift, sc, lo, hi); a_lo[1] = (int)lo; a_hi[1] = (int)hi;
            limbs(qs[j].z >> shift, sc, lo, hi); a_lo[2] = (int)lo; a_hi[2] = (int)hi;
            limbs(qs[j].w >> shift, sc, lo, hi); a_lo[3] = (int)lo; a_hi[3] = (int)hi;
            const v4i b = as_v4i(a[j]);
            lo_sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, b, lo_sum, 0, 0, 0);
            hi_sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, b, hi_sum, 0, 0, 0);
        }
        v4i m_op = {0, 0, 0, 0};
        if (q == 0u) {
            m_op[0] = (int)mn_pack[0];
            m_op[1] = (int)mn_pack[1];
        }
        v4s min_lo, min_hi;
        uint2 bl, bh;
        q4k_bsum_limbs(bsums, bl, bh);
        v4i b_lo = {0, 0, 0, 0}, b_hi = {0, 0, 0, 0};
        if (q == 0u) {
            b_lo[0] = (int)bl.x; b_lo[1] = (int)bl.y;
            b_hi[0] = (int)bh.x; b_hi[1] = (int)bh.y;
        }
        const v4s zero = {0, 0, 0, 0};
        min_lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(m_op, b_lo, zero, 0, 0, 0);
        min_hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(m_op, b_hi, zero, 0, 0, 0);
        wave_lds_fence();
        const float4 d4 = *reinterpret_cast<const float4 *>(&row_scale[wave][0][4u * q]);
        const float4 m4 = *reinterpret_cast<const float4 *>(&row_scale[wave][1][4u * q]);
        const float d_of[4] = {d4.x, d4.y, d4.z, d4.w}, dmin_of[4] = {m4.x, m4.y, m4.z, m4.w};
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int dot = (hi_sum[i] << 3) + lo_sum[i];
            const int minimum = (min_hi[i] << 7) + min_lo[i];
            const float left = (da * d_of[i]) * (float)dot;
            const float right = (da * dmin_of[i]) * (float)minimum;
            acc[i] += (double)(left - right);
        }
    }

    __syncthreads();
    if (wave) {
#pragma unroll
        for (int i = 0; i < 4; ++i) partial[wave - 1u][i][lane] = acc[i];
    }
    __syncthreads();
    const unsigned long long token = tok0 + r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (wave) break;
        const unsigned long long row = row0 + 4u * q + (unsigned)i;
        double wide = acc[i];
#pragma unroll
        for (unsigned wv = 0; wv + 1u < WAVES; ++wv) wide += partial[wv][i][lane];
        const float sum = (float)wide;
        if (row >= g.row_count || token >= g.input_rows) continue;
        const unsigned long long at = token * g.out_stride + row;
        const float value = g.additive ? sum + g.additive[at] : sum;
        if (!finite_f32(value)) raise_status(g.status, 1);
        else store_published(g.publication, g.out + at, g.output_bf16 ? bf16_round(value) : value);
    }
    publish_when_last(g.publication, g.status, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
}

}  // namespace

// Whether two workgroups of 32 x 64 tiles share a compute unit, where the tiles outnumber them. The longer the row, the nearer a
// pair's time comes to that of two tiles one behind the other, so a third round of tiles, which is half a pair's, is
// dearer in pairs from some 6000 columns on, and any from 11 500 (multiples of 8192 apart, which gain in pairs as short rows do). us a call,
// in pairs and not, 384 / 640 / 896 tiles: 4096 columns 38.6 / 57.8 / 65.9 and 45.3 / 61.5 / 77.6; 5888 48.4 / 76.8 / 88.1 and 54.3 / 77.1 / 97.5; 7424 57.1 / 92.5 / 107.1
// and 61.3 / 87.4 / 111.0; 11 264 76.1 / 125.2 / 142.3 and 76.4 / 110.1 / 141.8; 12 288 81.4 / 132.9 / 152.5 and 80.9 / 114.1 / 146.7; 8192 (576, 832 tiles) 104.5 / 128.4 and
// 108.8 / 143.4.
static bool tiles_share_units(uint64_t tiles, uint64_t units, uint64_t row_width)
{
    if (tiles <= units) return false;
    if (row_width < 6144u || row_width % 8192u == 0u) return true;
    return row_width < 11520u && (tiles <= 2u * units || tiles > 3u * units);
}

int launch_q4k_rows_dense(const uint8_t *encoded, uint64_t row_count, uint64_t row_width,
                          uint64_t row_bytes, const void *act_q8k, uint64_t input_rows,
                          const float *additive, float *out, uint64_t out_stride, bool output_bf16,
                          int *status, hipStream_t stream, Publisher *publisher)
{
    if (!row_count || !input_rows || row_width % 256u || row_width / 256u * 144u != row_bytes)
        return ST_BOUNDS;
    if (((uintptr_t)encoded & 15u) || ((uintptr_t)act_q8k & 3u)) return ST_INVALID_ARG;
    const uint64_t row_tiles = (row_count + 31u) / 32u;
    if (row_tiles > 0x7fffffffull || row_width / 256u > 0xffffffffull) return ST_BOUNDS;
    DenseQ4kArgs g{encoded, row_count, row_bytes, (unsigned)(row_width / 256u),
                   (const unsigned char *)act_q8k, input_rows, additive, out, out_stride,
                   output_bf16 ? 1 : 0, status, {}};
    // 16 x 16 tiles, on four waves where several workgroups share a compute unit (7168 x 7168 by 32 rows 23.2 us, on
    // eight 26.8; 7168 x 2048 by 32 9.8 and 13.1), up to 32 input rows and beyond them while tiles of twice the tokens would fit
    // the device in one round (2048 x 7168 by 64 rows 12.7 us, on the 32 x 32 tiles 16.7).
    const uint64_t units = (uint64_t)compute_units(), small_tiles = (row_count + 15u) / 16u;
    const uint64_t token_tiles16 = (input_rows + 15u) / 16u, token_tiles32 = (input_rows + 31u) / 32u;
    if (input_rows <= 32u || small_tiles * token_tiles32 <= units) {
        if (small_tiles > 0x7fffffffull || token_tiles16 > 65535ull) return ST_BOUNDS;
        const dim3 grid((unsigned)small_tiles, (unsigned)token_tiles16);
        // A launch ends the operation while a compute unit has up to five of its tiles: the next ones wait for the stores of
        // those before them. us a call, published by the launch and behind it: 4096 x 512 by 32 rows (two tiles a compute
        // unit) 14.6 and 14.9, 16384 x 4096 by 16 (four) 25.6 and 26.5, 8192 x 512 by 32 (four) 17.9 and 17.6; 12288 x 512 / 4096 by 32 (six)
        // 18.9 / 31.4 and 18.5 / 31.5, 16384 x 512 / 2048 by 32 (eight) 21.1 / 27.3 and 20.1 / 27.1.
        g.publication = take_publication(publisher, small_tiles * token_tiles16, 5u * units);
        if (small_tiles * token_tiles16 <= units) dense_q4k16_kernel<8><<<grid, 512, 0, stream>>>(g);
        else dense_q4k16_kernel<4><<<grid, 256, 0, stream>>>(g);
    } else {
        const uint64_t token_tiles = (input_rows + 63u) / 64u;
        // enough (128 rows x 64 tokens) tiles for every compute unit: operands staged through LDS
        if ((row_count + 127u) / 128u * token_tiles >= units)
            return launch_q4k_rows_staged(encoded, row_count, row_width, row_bytes, act_q8k, input_rows,
                                          additive, out, out_stride, output_bf16, status, stream);
        // A workgroup's pass over the row width takes about as long on a full device as on an
        // empty one, so while the smaller tiles still fit the device in one round they are the
        // faster ones (2048 x 7168 at 96 rows: 17 us on 32 x 32 tiles, 21 on 16 x 32; at 256 rows 27 us on 32 x 64).
        if (row_tiles * token_tiles32 <= units)
            dense_q4k_kernel<1><<<dim3((unsigned)row_tiles, (unsigned)token_tiles32), 256, 0, stream>>>(g);
        else if (tiles_share_units(row_tiles * token_tiles, units, row_width))
            dense_q4k_kernel<2, true><<<dim3((unsigned)row_tiles, (unsigned)token_tiles), 256, 0, stream>>>(g);
        else
            dense_q4k_kernel<2><<<dim3((unsigned)row_tiles, (unsigned)token_tiles), 256, 0, stream>>>(g);
    }
    return check_launch("dense_q4k");
}

}  // namespace yvex
