// Row-batch (prefill-width) grouped expert projections on the int8 matrix cores of gfx950.
//
// A workgroup walks runs: one token tile (up to 64 ordered pairs of a bucket) against row tiles of 256 weight rows (128 gate rows
// and the 128 matching up rows when the SwiGLU is fused), one after another. It has eight waves, two per
// SIMD; each owns 32 weight rows of a row tile and multiplies them by all of the token tile's Q8_K activation rows
// with V_MFMA_I32_32X32X32_I8. 256 registers a wave are what decides the tile: 32 rows x 64 tokens of int32
// limb sums and double-precision row sums.
//
// What bounds it is not the matrix pipe: with two waves a SIMD vector instructions run under matrix instructions (a 32 x 32 x 32
// instruction and k byte permutes take a SIMD max(33, 9 + 4.5 k) cycles), and without its
// matrix instructions a launch takes as many cycles. A wave alone on its SIMD hides up to seven permutes under its own matrix
// instruction (46 cycles) and from eight on none (41 + 4.5 k: 77 of eight, 95 of twelve); this loop has 9.6 vector instructions for
// each, and would have 7.4 with 128 tokens a wave. It is the issue of everything else, about five cycles a vector or LDS
// instruction and forty a window copy, and the matrix instructions' power: 1.9 to 2.0 GHz under this kernel, 2.2 without
// them. The wave's number is kept scalar, and with it every LDS address of a copy and every distance it adds to its
// lanes' pointers (330 -> 318 vector instructions a superblock: 7168 x 2 x 4096 by 2048 rows 317 -> 301 us, 2048 x 8192 by 2048 122.2 -> 119.4).
// Two things that look the same and are slower: stages with sixteen bytes between groups of tokens, which make the fragments' places
// immediate offsets (a copy into LDS that does not start on 64 bytes is split: 582K cycles against 570K), and windows without their
// spare pieces (64 scattered dwords cost a copy more than 64 pieces of sixteen bytes: 600K against 590K).
//
//   A operand (weights): built in registers, one K chunk (32 columns) ahead of its use. Lane
//       (r, h) = (lane % 32, lane / 32) owns weight row r and the groups 4h .. 4h + 3 of the
//       current superblock (128 columns); K chunk m of the superblock is, for that lane, the 16
//       weights 16 (m % 2) .. + 15 of group 4h + m / 2. The order of K inside a matrix
//       instruction is free as long as both operands agree.
//       The IQ2_XXS value of one weight is level * sign * (2s+1), up to 43 * 31 = 1333, so it is
//       split into two int8 limbs, value = 128 * hi + lo with hi in [1, 11] and lo in
//       [-120, 63], and every K chunk costs two matrix instructions per token block. For one
//       scale there are only three levels, so the six signed limb values of a group fit two
//       registers and one V_PERM_B32 per four weights picks them: the selector byte of a weight
//       is its level code (0..2) plus 4 when it is negative. Three LDS tables feed this, sixteen
//       replicas each so that the lanes of a quarter-wave never share a bank: level codes of a
//       codebook entry (8 bytes), sign selectors of a 7-bit sign field (8 bytes) and the limb
//       words of a scale (16 bytes).
//   Weight bytes: each wave copies, per superblock, the aligned 68 bytes around the superblock of
//       each of its 32 rows into an LDS window (GLOBAL_LOAD_LDS_DWORDX4, every cache line
//       fetched once), two superblocks ahead; the lanes take their records out with three
//       16-byte LDS reads from a piece-major window (no two lanes of sixteen on one bank; dword
//       reads of rows 80 bytes apart put four lanes on a bank).
//   B operand (activations): the tile's int8 blocks of one superblock, copied from global memory
//       straight into LDS, in a ring of stages. 16-byte piece c of token t sits at piece position
//       c ^ (t % 16), so the 16 lanes that read one fragment column together hit 16 different
//       bank groups.
//   C: per (superblock, 32-token block) two int32 accumulators of 32 x 32; T = 128 * C_hi + C_lo
//       is the exact integer superblock sum of the reference's primitive
//       (src/backend/cuda/kernel_primitives.h:287-313), scaled into the float term
//       ((0.125 * d_w) * d_a) * T; a row's terms are added in double, in superblock order, and
//       the sum is rounded to float once, which is what the CPU path computes for a row (double
//       accumulation over a row's blocks, src/gguf/quant_compute.c:152-172): every value
//       rounded to bfloat16 afterwards rounds as it does there.
//       The products of a row's and a token's scale are one V_MFMA_F32_32X32X1_2B_F32 a superblock, the outer products
//       of both token blocks at once: a product of two floats rounded once, the bits of V_MUL_F32. 363 -> 330 vector and
//       61 -> 56 LDS instructions a superblock and wave of 64 tokens, and a row's scale stays in its lane's register
//       (it went through LDS to the lanes that hold the row's sums). 2048 rows of 7168 by eight of 256 experts with uneven routing, us
//       a layer: 2995 -> 2967 on one box, 3010 -> 3005 on another. The instruction holds the wave for as long as sixteen
//       multiplications, which takes most of the gain; at one token block it is level.
//   Output: accumulator i of lane (r, h) is token r's sum for row 8 (i / 4) + 4 h + i % 4 of the
//       wave's 32 (gate sums in the first eight, the matching up sums in the last eight when
//       fused), so a lane stores four consecutive rows of its token, 16 bytes, straight from its
//       registers; the stores of a wave complete whole cache lines, which the L2 merges.
//
// Same inputs, outputs and rounding points as the decode-width sweeps in moe.hip
// (src/backend/cuda/tensorcore.cu:378-702 is the reference's counterpart, unused there).
#include "common.hpp"
#include "launch.hpp"
#include "grouped.hpp"
#include "lds_copy.hpp"
#include "iq2_limbs.hpp"

namespace yvex {

constexpr unsigned kRowWaves = 8u;                          // two per SIMD
constexpr unsigned kRowThreads = 64u * kRowWaves;
constexpr unsigned kTileTokens = 64u;
constexpr unsigned kActPitch = 256u;                       // one Q8_K block's int8 payload
// LDS map (absolute byte offsets; the dynamic allocation starts at 0, checked at kernel start).
// Codebook entry e owns the 256 bytes at 256 e: sixteen replicas of its 8 level codes in the
// first half; the second half of entries 0-127 holds sixteen replicas of the sign selectors of
// sign field e.
constexpr unsigned kCodeBase = 0u;
constexpr unsigned kSelBase = 128u;
constexpr unsigned kLutBase = 65536u;                       // 16 scales x 16 replicas x 16 bytes
constexpr unsigned kPairInfoBase = kLutBase + 16u * 16u * 16u;   // {out row, route weight} x 64
// Item numbering: first full 64-pair tile of every bucket (257 words), then per class of last,
// partial, tile (33-63, 1-32 pairs) a count and the list of its buckets (u16).
constexpr unsigned kTileStartBase = kPairInfoBase + kTileTokens * 8u;
constexpr unsigned kClassCountBase = kTileStartBase + 260u * 4u;
constexpr unsigned kClassListBase = kClassCountBase + 16u;
constexpr unsigned kTrashBase = kClassListBase + 2u * 256u * 2u;   // 256 bytes nobody reads
// Weight windows: per wave two buffers of six 16-byte pieces for each of the wave's 32 rows,
// piece-major (piece p of row r at slot 32 p + r; three full copies fill a buffer): the pieces a
// lane's record lies in are three conflict-free 16-byte reads. Canonical bytes: the aligned 68
// bytes around a superblock (pieces at 0, 16, 32, 48 and 52, the sixth repeats the fifth); the
// image: the two 36-byte lane records (pieces at 0, 16, 32 and at 36, 52, 56).
constexpr unsigned kWindowBase = (kTrashBase + 256u + 255u) & ~255u;
constexpr unsigned kWindowBytes = 32u * 96u;
constexpr unsigned kStageBase = kWindowBase + kRowWaves * 2u * kWindowBytes;
// activation stages: a ring of 4 / NTB stages of NTB x 32 slots (256 bytes each) + 64 scales
constexpr unsigned kStageRingBytes = 128u * kActPitch + 4u * 256u;
constexpr unsigned kMfmaLdsBytes = kStageBase + kStageRingBytes;
static_assert(kMfmaLdsBytes <= 160u * 1024u, "one workgroup per compute unit");

struct MfmaArgs {
    GroupedProblem pr;
    unsigned width;          // reduction width
    unsigned out_rows;       // weight rows per expert
    double limit;
    int *status;
    int plain_output;        // plain projection: outputs stay fp32 instead of being rounded to bf16
    int image;               // weights are the sweep image (72-byte records) instead of canonical bytes
    unsigned few;            // pairs of a tile of the few-pair kernel (rows16.hip), which has a part of the buckets' last tiles
};

__device__ __forceinline__ void mfma_tables_fill()
{
    for (unsigned index = threadIdx.x; index < 256u * 16u; index += blockDim.x)
        lds_write_uint2(kCodeBase + (index >> 4) * 256u + (index & 15u) * 8u, iq2_level_codes(index >> 4));
    for (unsigned index = threadIdx.x; index < 128u * 16u; index += blockDim.x)
        lds_write_uint2(kSelBase + (index >> 4) * 256u + (index & 15u) * 8u, iq2_sign_selectors(index >> 4));
    for (unsigned index = threadIdx.x; index < 16u * 16u; index += blockDim.x)
        lds_write_uint4(kLutBase + index * 16u, iq2_limb_words(index >> 4));
}

__device__ __forceinline__ unsigned uniform32(unsigned v)
{
    return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}

// Row tiles [row_tile, row_end) of one token tile.
struct MfmaRun {
    unsigned long long expert, pair0;
    unsigned tokens, row_tile, row_end;
};

// A run of row tiles against one token tile of NTB live 32-token blocks (NTB is 1 or 2).
//
// Time slot (sb, m) = superblock sb, K chunk m: 2 NTB matrix instructions (low and high limb for
// every token block) on the chunk's operands, which were built during the slot before: the
// weights of a superblock are decoded chunk by chunk just ahead of their use, two chunks' worth
// of operand registers in all. Between the matrix instructions the slot carries the LDS reads of
// the activation fragments two slots ahead, the table lookups of the chunk two slots ahead,
// the selector words and permutes of the next chunk, and its share of the copies. After the
// last chunk the integer sums of the superblock are scaled and added to the row sums. Two waves
// share a SIMD: while one waits for its own matrix instructions or scales its sums the other's
// instructions run.
//
// Everything that comes from memory inside the loop arrives by GLOBAL_LOAD_LDS copies, whose
// completion the kernel counts by hand (they retire in order):
//   * activations: a ring of R = 4 / NTB stages of NTB x 32 slots (256 int8 + one scale each);
//     the copies of superblock sb + R are issued right after the barrier of superblock sb, which
//     every wave passes once all its reads of that stage have returned;
//   * weights: per wave two windows holding, for each of its 32 rows, the aligned 68 bytes
//     around one superblock (five 16-byte pieces a row, the fifth ending with the dword that
//     holds the superblock's last byte, so nothing behind it is touched; the image: the three
//     pieces that hold each of the two lane records), stored piece-major. Each cache line of a
//     row is fetched once; taking the records out of the window is LDS work. Loading the
//     records lane by lane from global memory touched every row's line four times per
//     superblock, and the memory pipeline spends about two cycles per line an instruction
//     touches: with eight waves that was the longest pole of the step.
// The loop body is one superblock in one basic block (requests past the end are clamped, and
// superblocks past the end run with a zero row scale), so nothing leaves registers.
//
// From row tile to row tile nothing stops: superblocks are counted through (`step`), the windows fetched ahead are the
// next tile's, the stages begin again with the token tile's first, and a tile's sums are published between two
// steps. Only a run opens: where its tokens' rows lie, the first copies' round trip, the first operands, 9 000 to
// 10 000 cycles that every item paid (36 000 in the loop of eight superblocks, 121 000 in one of 28) while items were dealt out one by
// one. A tile that is not whole has lanes that repeat a row, and runs alone.
template <bool FUSED_UP, unsigned NTB, bool IMAGE>
__device__ __forceinline__ void rows_run(const MfmaArgs &a, const MfmaRun &it)
{
    const GroupedProblem &pr = a.pr;
    constexpr unsigned R = 4u / NTB;                 // activation stages
    constexpr unsigned T = NTB * 32u;                // token slots of one stage
    constexpr unsigned kStageBytes = T * kActPitch + 256u;
    constexpr unsigned kBarrierSlot = 5u;
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = uniform32(tid >> 6);
    const unsigned r = lane & 31u, h = lane >> 5;
    constexpr unsigned kItemRows = FUSED_UP ? 128u : 256u;
    const unsigned superblocks = a.width >> 8;
    const unsigned last = superblocks - 1u;

    // ---- weight rows: rows 0-15 of a wave are gate rows and rows 16-31 the matching up rows
    // when the SwiGLU is fused ----
    auto row_pointer = [&](unsigned wave_row) {
        unsigned row;
        bool is_up = false;
        if constexpr (FUSED_UP) {
            row = it.row_tile * kItemRows + wave * 16u + (wave_row & 15u);
            is_up = wave_row >= 16u;
        } else {
            row = it.row_tile * kItemRows + wave * 32u + wave_row;
        }
        if (row >= a.out_rows) row = a.out_rows - 1u;
        return is_up
            ? pr.up + it.expert * pr.up_expert_bytes + (unsigned long long)row * pr.up_row_bytes
            : pr.gate + it.expert * pr.expert_bytes + (unsigned long long)row * pr.row_bytes;
    };
    // Superblocks are 66 bytes, so they start on 2-byte boundaries, and vector accesses that are
    // not dword-aligned run at less than half rate: a window starts at the aligned dword that
    // holds the superblock's first byte. Copy k of a window moves pieces 64 k + lane of the
    // wave's 160 (row = piece / 5).
    const unsigned row_misalign = (unsigned)(unsigned long long)row_pointer(r) & 3u;    // of the lane's own row
    const unsigned char *window_from[3];    // row start + piece offset, of the row this lane copies
#pragma unroll
    for (unsigned k = 0; k < 3u; ++k) {
        if constexpr (IMAGE) {
            // The 72-byte record of a row's superblock is two lane records of 36 bytes (dword
            // aligned): bytes 0-35 lie in the pieces at 0, 16 and 32, bytes 36-71 in the pieces at
            // 36, 52 and 56 (the last one ends with the record, so nothing behind it is touched).
            const unsigned piece = 2u * k + (lane >> 5);        // slot 64 k + lane = 32 piece + row
            const unsigned at = piece < 3u ? 16u * piece : piece == 3u ? 36u : piece == 4u ? 52u : 56u;
            window_from[k] = row_pointer(lane & 31u) + at;
        } else {
            // The aligned 68 bytes around a superblock lie in the pieces at 0, 16, 32, 48 and 52
            // (the last ends with the dword that holds the superblock's last byte); the sixth slot
            // repeats the fifth.
            const unsigned piece = 2u * k + (lane >> 5);
            window_from[k] = row_pointer(lane & 31u) + (piece < 4u ? 16u * piece : 52u);
        }
    }
    const unsigned window_base = kWindowBase + wave * 2u * kWindowBytes;
    // The window of the step that is asked for next: its superblock, the distance to its row tile, its step.
    const unsigned steps = (it.row_end - it.row_tile) * superblocks;
    const unsigned long long tile_bytes = (unsigned long long)kItemRows * pr.row_bytes;
    unsigned window_sb = 0u, window_step = 0u;
    unsigned long long window_tile = 0ull;
    auto window_passed = [&] {                       // (behind the run's last step its bytes are fetched again)
        const bool more = window_step + 1u < steps, wraps = window_sb == last;
        ++window_step;
        if (more) {
            window_sb = wraps ? 0u : window_sb + 1u;
            window_tile += wraps ? tile_bytes : 0ull;
        }
    };
    auto weight_piece = [&](unsigned k) {            // the pieces of a window in order
        const unsigned to = window_base + (window_step & 1u) * kWindowBytes + k * 1024u;
        unsigned long long offset = window_tile + window_sb * (IMAGE ? 72u : 66u);
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+s"(offset));       // (one sum on the scalar unit, one addition a lane)
#endif
        const unsigned char *from = IMAGE
            ? window_from[k] + offset
            : (const unsigned char *)((unsigned long long)(window_from[k] + offset) & ~3ull);
        copy_to_lds_16(from, to);
        if (k == 2u) window_passed();
    };

    // ---- activation rows this lane copies: wave w owns the 4-slot groups w (and w + 8) ----
    // Lane l of a group moves piece position l % 16 of slot 4 g + l / 16; LDS receives the wave's
    // 64 pieces back to back, so the swizzle is applied on the global side.
    auto token_row = [&](unsigned token) {
        const unsigned live = token < it.tokens ? token : it.tokens - 1u;   // padding repeats a row
        const unsigned long long ordered = it.pair0 + live;
        const unsigned long long source = pr.order ? pr.order[ordered] : ordered;
        const unsigned long long arow = pr.act_by_ordered_pair ? ordered : (unsigned)source / pr.topk;      // (pairs fit 32 bits)
        return (const unsigned char *)pr.activations + arow * pr.act_stride;
    };
    const unsigned char *copy_from[NTB];
#pragma unroll
    for (unsigned j = 0; j < NTB; ++j) {
        const unsigned token = 4u * (wave + kRowWaves * j) + (lane >> 4);
        copy_from[j] = token_row(token) + 4u + 16u * ((lane & 15u) ^ (token & 15u));
    }
    // Wave 0 also copies the stage's slot scales, laid out [token % 32][token block] so that a lane
    // reads the scales of its NTB tokens with one LDS read. The other waves run the same
    // instruction on one address for all lanes (one cache line: next to free) into bytes nobody
    // reads, which is cheaper than a branch around the copy.
    const unsigned char *scale_from;
    {
        const unsigned index = wave == 0u ? lane % T : 0u;
        scale_from = token_row((index % NTB) * 32u + index / NTB);
    }
    // Where each pair's results go and its route weight, for the publishing passes: requested now,
    // put into LDS once the previous run's last one is over.
    const bool info_lane = tid < kTileTokens && tid < it.tokens;
    unsigned info_out = 0u;
    float info_weight = 1.0f;
    if (info_lane) {
        const unsigned long long ordered = it.pair0 + tid;
        const unsigned long long source = pr.order ? pr.order[ordered] : ordered;
        info_out = (unsigned)(pr.out_by_source_pair ? source : ordered);
        if (pr.route_weights) info_weight = pr.route_weights[source];
    }
    constexpr unsigned kActPieces = NTB + 1u;
    // the stage that is asked for next: its superblock and its place
    unsigned stage_sb = 0u, stage_to = kStageBase;
    auto act_piece = [&](unsigned j) {               // the pieces of a stage in order
        const unsigned base = stage_to;
        unsigned offset = stage_sb * kQ8KBytes;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+s"(offset));
#endif
        if (j < NTB) {
            copy_to_lds_16(copy_from[j] + offset, base + (wave + kRowWaves * j) * 1024u);
        } else {
            copy_to_lds_4(scale_from + offset, wave == 0u ? base + T * kActPitch : kTrashBase);
            stage_sb = stage_sb == last ? 0u : stage_sb + 1u;
            stage_to = stage_to == kStageBase + (R - 1u) * kStageBytes ? kStageBase : stage_to + kStageBytes;
        }
    };
    // the copies issued after the barrier of a step: the stage and the window just released, R and three steps ahead
    constexpr unsigned kRoundPieces = kActPieces + 3u;
    auto round_piece = [&](unsigned j) {
        if (j < kActPieces) act_piece(j);
        else weight_piece(j - kActPieces);
    };

    // ---- decode state ----
    const unsigned code_lane = kCodeBase + (lane & 15u) * 8u;
    const unsigned sel_lane = kSelBase + (lane & 15u) * 8u;
    const unsigned lut_lane = kLutBase + (lane & 15u) * 16u;
    unsigned grids[4], aux[4];           // group records of the superblock being decoded
    unsigned head = 0u;                  // image: fp16 scale | the four group scales of this half << 16
    float row_scale = 0.0f;              // of the superblock being decoded, of the lane's own row
    uint2 codes[2][2], signs[2][2];      // [chunk & 1]: table words of the chunk's two subgroups
    uint4 limbs[2];                      // [group & 1]: limb words of a group
    v4i a_lo[2], a_hi[2];                // [chunk & 1]: A operands of a K chunk

    // Records of superblock sb out of its window, and the row's scale (zero past the end: such superblocks add nothing). With o = (row start
    // + 66 sb) mod 4 (0 or 2) the fp16 scale sits o bytes into the window and the lane's 32 code
    // bytes at o + 2 + 32 h: in aligned dwords 8 h + o / 2 onwards, shifted by 2 bytes when o is
    // 0. Aligned dword 16 is the last dword of the fifth piece.
    auto settle = [&](unsigned step, unsigned sb) {  // (superblock `sb`, which only its parity and the last step need)
        if constexpr (IMAGE) {
            // The lane's record is nine dwords: pieces 3 h and 3 h + 1 whole, and of piece 3 h + 2
            // the first dword (bytes 32-35 of the row's 72) or the last (bytes 68-71).
            const unsigned at = window_base + (step & 1u) * kWindowBytes + (3u * h * 32u + r) * 16u;
            const v4i first = lds_read_v4i(at), second = lds_read_v4i(at + 512u), third = lds_read_v4i(at + 1024u);
            head = (unsigned)first[0];
            grids[0] = (unsigned)first[1];
            aux[0] = (unsigned)first[2];
            grids[1] = (unsigned)first[3];
            aux[1] = (unsigned)second[0];
            grids[2] = (unsigned)second[1];
            aux[2] = (unsigned)second[2];
            grids[3] = (unsigned)second[3];
            aux[3] = (unsigned)(h ? third[3] : third[0]);
            row_scale = step < steps ? 0.125f * f16_bits_to_float(head & 0xffffu) : 0.0f;
            return;
        }
        const unsigned o = (row_misalign + 2u * sb) & 3u;
        // Aligned dwords 8 h .. 8 h + 8 of the window: pieces 2 h and 2 h + 1 whole, and the dword
        // behind them (the first of piece 2, or the last of the fifth piece, which is aligned
        // dword 16). The lane's nine dwords start at dword 8 h + o / 2 of the window.
        const unsigned at = window_base + (step & 1u) * kWindowBytes + (2u * h * 32u + r) * 16u;
        const v4i first = lds_read_v4i(at), second = lds_read_v4i(at + 512u), third = lds_read_v4i(at + 1024u);
        const unsigned d[9] = {(unsigned)first[0], (unsigned)first[1], (unsigned)first[2], (unsigned)first[3],
                               (unsigned)second[0], (unsigned)second[1], (unsigned)second[2], (unsigned)second[3],
                               (unsigned)(h ? third[3] : third[0])};
        unsigned w[9];
#pragma unroll
        for (unsigned i = 0; i < 8u; ++i) w[i] = o ? d[i + 1u] : d[i];
        w[8] = d[8];           // (the ninth is only part of a record when o is 0)
        // the fp16 scale sits o bytes into the window: in the first dword of the first half's lanes,
        // from where those of the second half have it too
        const unsigned scale16 = ((unsigned)first[0] >> (8u * o)) & 0xffffu;
        const unsigned shift = (o + 2u) & 3u;
#pragma unroll
        for (unsigned g = 0; g < 4u; ++g) {
            grids[g] = __builtin_amdgcn_alignbyte(w[2u * g + 1u], w[2u * g], shift);
            aux[g] = __builtin_amdgcn_alignbyte(w[2u * g + 2u], w[2u * g + 1u], shift);
        }
        const float mine = step < steps ? 0.125f * f16_bits_to_float(scale16) : 0.0f;
        row_scale = __uint_as_float((unsigned)__builtin_amdgcn_ds_bpermute((int)(4u * r), (int)__float_as_uint(mine)));
    };
    // table lookups of K chunk c: subgroups 2 (c & 1) and 2 (c & 1) + 1 of group c / 2
    auto lookup = [&](unsigned c) {
        const unsigned g = c >> 1;
#pragma unroll
        for (unsigned i = 0; i < 2u; ++i) {
            const unsigned j = 2u * (c & 1u) + i;
            codes[c & 1u][i] = lds_read_uint2(__builtin_amdgcn_perm(grids[g], code_lane, 0x0c0c0400u + (j << 8)));
            if constexpr (IMAGE) {      // the field has a byte of its own
                signs[c & 1u][i] = lds_read_uint2(__builtin_amdgcn_perm(aux[g], sel_lane, 0x0c0c0400u + (j << 8)));
            } else {
                const unsigned field = j == 0u ? aux[g] << 8 : j == 1u ? aux[g] << 1 : aux[g] >> (7u * j - 8u);
                signs[c & 1u][i] = lds_read_uint2((field & 0x7f00u) | sel_lane);
            }
        }
        if ((c & 1u) == 0u)
            limbs[g & 1u] = lds_read_uint4((IMAGE ? (head >> (8u + 4u * g)) & 0xf00u : (aux[g] >> 20) & 0xf00u) | lut_lane);
    };
    // selector words and permutes of K chunk c
    auto build = [&](unsigned c) {
        const uint4 lw = limbs[(c >> 1) & 1u];
        const unsigned s0 = codes[c & 1u][0].x | signs[c & 1u][0].x, s1 = codes[c & 1u][0].y | signs[c & 1u][0].y;
        const unsigned s2 = codes[c & 1u][1].x | signs[c & 1u][1].x, s3 = codes[c & 1u][1].y | signs[c & 1u][1].y;
        a_lo[c & 1u] = v4i{(int)__builtin_amdgcn_perm(lw.y, lw.x, s0), (int)__builtin_amdgcn_perm(lw.y, lw.x, s1),
                           (int)__builtin_amdgcn_perm(lw.y, lw.x, s2), (int)__builtin_amdgcn_perm(lw.y, lw.x, s3)};
        a_hi[c & 1u] = v4i{(int)__builtin_amdgcn_perm(lw.w, lw.z, s0), (int)__builtin_amdgcn_perm(lw.w, lw.z, s1),
                           (int)__builtin_amdgcn_perm(lw.w, lw.z, s2), (int)__builtin_amdgcn_perm(lw.w, lw.z, s3)};
    };

    // ---- activation fragments: piece 8 h + m of slot r (+ 32 tb) of the current stage; stage
    // bases are multiples of 256, so the piece position is bits 4-7 of the address ----
    unsigned frag_at = kStageBase + r * kActPitch + (((8u * h) ^ (r & 15u)) << 4);

    // ---- prologue ----
    // Copies in flight when the loop starts are those of its own schedule: a round (stage step + R,
    // window step + 3) is issued after the barrier of a step, four pieces in slots 6 and 7 and
    // the rest at the start of the next one, so rounds -(R - 1) .. -1 are issued here (windows 0 and 1 are needed before
    // them; a round before -1 has three copies to where nobody reads in the place of a window, which keeps the counts below the same for
    // every step).
    lds_barrier();     // every wave is done with the previous run's stages and pair records (whose copies and stores have all completed: see its end)
#pragma unroll
    for (unsigned k = 0; k < 3u; ++k) weight_piece(k);
#pragma unroll
    for (unsigned j = 0; j < kActPieces; ++j) act_piece(j);
#pragma unroll
    for (unsigned k = 0; k < 3u; ++k) weight_piece(k);
    __builtin_amdgcn_s_waitcnt(0x0f73u);   // vmcnt(3): window 0 and stage 0 have landed
    if (info_lane) lds_write_uint2(kPairInfoBase + tid * 8u, make_uint2(info_out, __float_as_uint(info_weight)));
    settle(0u, 0u);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the window's reads have returned before it is refilled
#pragma unroll
    for (unsigned x = 1; x + 1u < R; ++x) {
#pragma unroll
        for (unsigned j = 0; j < kActPieces; ++j) act_piece(j);
#pragma unroll
        for (unsigned k = 0; k < 3u; ++k) copy_to_lds_4(scale_from, kTrashBase);
    }
#pragma unroll
    for (unsigned j = 0; j < 4u; ++j) round_piece(j);
    lookup(0u);
    lookup(1u);
    build(0u);
    __syncthreads();   // every wave's share of stage 0 has landed

    v16i sum_lo[NTB], sum_hi[NTB];   // integer sums of the running superblock
    v4i frag[2][NTB];                // [slot & 1]: re-requested for two slots on as soon as it is used
#pragma unroll
    for (unsigned tb = 0; tb < NTB; ++tb) {
        frag[0][tb] = lds_read_v4i(frag_at + tb * 32u * kActPitch);
        frag[1][tb] = lds_read_v4i((frag_at ^ 16u) + tb * 32u * kActPitch);
    }
    // Waits, counted in copies issued later than the one needed (a tile's stores among them make a wait longer, never
    // shorter), step by step:
    //   * before settle(step + 1) at slot 5: window step + 1 belongs to round step - 2, so one full
    //     round (step - 1) may be in flight;
    //   * at the barrier of a step: stage step + 1 belongs to round step + 1 - R, so the
    //     window of that round and R - 2 full rounds may be in flight.
    constexpr unsigned kSettleInFlight = kRoundPieces;
    constexpr unsigned kBarrierInFlight = 3u + (R - 2u) * kRoundPieces;

    unsigned step = 0u, stage = kStageBase;              // the running step and its stage
    const float limit_f32 = (float)a.limit;
    const bool whole_quads = (a.out_rows & 3u) == 0u;
    for (unsigned row_tile = it.row_tile; row_tile < it.row_end; ++row_tile) {
    double acc[NTB][16];            // row sums: float terms added in double, in superblock order
#pragma unroll
    for (unsigned tb = 0; tb < NTB; ++tb)
#pragma unroll
        for (unsigned i = 0; i < 16u; ++i) acc[tb][i] = 0.0;
    for (unsigned sb = 0; sb < superblocks; ++sb, ++step) {
        float rs = 0.0f, ts = 0.0f;  // scales of the lane's weight row and of its token (of block h) in this superblock
        v32f scale;                  // their products, where the sums of that row and token are
#pragma unroll
        for (unsigned m = 0; m < 8u; ++m) {
            // ---- 2 NTB matrix instructions with the rest of the slot's work between them, a
            // few instructions at a time ----
            auto matrix = [&](unsigned tb, bool high) {
                const v4i b = frag[m & 1u][tb];
                v16i zero;
#pragma unroll
                for (unsigned i = 0; i < 16u; ++i) zero[i] = 0;
                if (!high) sum_lo[tb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_lo[m & 1u], b, m ? sum_lo[tb] : zero, 0, 0, 0);
                else sum_hi[tb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_hi[m & 1u], b, m ? sum_hi[tb] : zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            const unsigned next_chunk = (m + 1u) & 7u;
            const uint4 lw = limbs[(next_chunk >> 1) & 1u];
            unsigned selector[4];
            matrix(0u, false);
            // the table lookups of the chunk two slots on
            lookup((m + 2u) & 7u);
            __builtin_amdgcn_sched_barrier(0);
            matrix(0u, true);
            // selector words and low limbs of the next chunk
            selector[0] = codes[next_chunk & 1u][0].x | signs[next_chunk & 1u][0].x;
            selector[1] = codes[next_chunk & 1u][0].y | signs[next_chunk & 1u][0].y;
            selector[2] = codes[next_chunk & 1u][1].x | signs[next_chunk & 1u][1].x;
            selector[3] = codes[next_chunk & 1u][1].y | signs[next_chunk & 1u][1].y;
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) a_lo[next_chunk & 1u][i] = (int)__builtin_amdgcn_perm(lw.y, lw.x, selector[i]);
            if constexpr (NTB == 2u) {
                __builtin_amdgcn_sched_barrier(0);
                matrix(1u, false);
            }
            // high limbs of the next chunk
#pragma unroll
            for (unsigned i = 0; i < 4u; ++i) a_hi[next_chunk & 1u][i] = (int)__builtin_amdgcn_perm(lw.w, lw.z, selector[i]);
            if constexpr (NTB == 2u) {
                __builtin_amdgcn_sched_barrier(0);
                matrix(1u, true);
            }
            // ---- the fragments two slots on (past the barrier slot the addresses already
            // point into the next superblock's stage) ----
            {
                unsigned piece = frag_at ^ (((m + 2u) & 7u) << 4);
                asm volatile("" : "+v"(piece));   // kept opaque so that the token block offset stays the instruction's immediate
#pragma unroll
                for (unsigned tb = 0; tb < NTB; ++tb) frag[m & 1u][tb] = lds_read_v4i(piece + tb * 32u * kActPitch);
            }
            if (m == 5u) {
                // chunk 7's lookups are on their way: the next superblock's records replace this
                // one's (its window has landed: see the counts above)
                __builtin_amdgcn_s_waitcnt(0x0f70u | (kSettleInFlight & 15u) | ((kSettleInFlight >> 4) << 14));
                rs = row_scale;
                settle(step + 1u, sb == last ? 0u : sb + 1u);
            }
            if (m == 4u) {
                // this superblock's token scales, while its stage is still held
                ts = __uint_as_float(lds_read_u32(stage + T * kActPitch + (r * NTB + (NTB == 2u ? h : 0u)) * 4u));
            }
            if (m == 6u) {
                // the scaling's factors: block h of the instruction is the rows against token block h
                v32f zero;
#pragma unroll
                for (unsigned i = 0; i < 32u; ++i) zero[i] = 0.0f;
                scale = __builtin_amdgcn_mfma_f32_32x32x1f32(rs, ts, zero, 0, 0, 0);
            }
            if (m == kBarrierSlot) {
                // Every read of this superblock's stage and of the next one's window has returned
                // and this wave's share of the next stage has landed: after the barrier nobody
                // reads this stage again and the next one is complete.
                __builtin_amdgcn_s_waitcnt(0x0070u | (kBarrierInFlight & 15u) | ((kBarrierInFlight >> 4) << 14));
                __syncthreads();
                const unsigned flip = stage == kStageBase + (R - 1u) * kStageBytes ? 0u - (R - 1u) * kStageBytes : kStageBytes;
                frag_at += flip;
                stage += flip;
            }
            // ---- the round of copies into the stage and the window just released: two pieces a
            // slot behind the barrier, the rest at the start of the next superblock ----
            if (m > kBarrierSlot) {
                round_piece(2u * (m - kBarrierSlot - 1u));
                round_piece(2u * (m - kBarrierSlot - 1u) + 1u);
            }
            if (m < kRoundPieces - 4u) round_piece(4u + m);
            // ---- the superblock's sums are complete: ((0.125 d_w) d_a) (128 hi + lo) ----
            if (m == 7u) {
#pragma unroll
                for (unsigned tb = 0; tb < NTB; ++tb)
#pragma unroll
                    for (unsigned i = 0; i < 16u; ++i) {
                        const int total = (sum_hi[tb][i] << 7) + sum_lo[tb][i];
                        const float term = scale[16u * tb + i] * (float)total;    // each product rounded to float
                        acc[tb][i] += (double)term;
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // ---- publish: the lane holds, for tokens 32 tb + r, rows 8 q + 4 h + j of its wave's 32
    // (j < 4): when fused, q 0-1 are gate rows and q 2-3 the matching up rows ----
    // The values go from the registers straight to memory, 16 bytes a lane: the two halves of a
    // wave complete 32 bytes of a token's row per store, the four (two) stores of a token block
    // a whole cache line (half of one), which the L2 merges before it writes them back. No LDS,
    // no barrier: the stores drain while the next row tile is worked on, those of a run's last one before the run ends.
    bool bad = false;
#pragma unroll
    for (unsigned tb = 0; tb < NTB; ++tb) {
        const unsigned token = tb * 32u + r;
        const uint2 info = lds_read_uint2(kPairInfoBase + token * 8u);   // (stale past the run's last token: not used)
        float *const out_row = pr.out + (unsigned long long)info.x * a.out_rows;
#pragma unroll
        for (unsigned q = 0; q < (FUSED_UP ? 2u : 4u); ++q) {
            const unsigned row = row_tile * kItemRows + wave * (FUSED_UP ? 16u : 32u) + 8u * q + 4u * h;
            float value[4];
            bool good = true;
            if constexpr (FUSED_UP) {
                const float route_weight = __uint_as_float(info.y);
#pragma unroll
                for (unsigned j = 0; j < 4u; ++j)
                    value[j] = swiglu_bf16_fast((float)acc[tb][4u * q + j], (float)acc[tb][4u * (q + 2u) + j], route_weight,
                                                a.limit, limit_f32);
            } else {
#pragma unroll
                for (unsigned j = 0; j < 4u; ++j) {
                    value[j] = (float)acc[tb][4u * q + j];
                    good &= finite_f32(value[j]);
                    if (!a.plain_output) value[j] = bf16_round(value[j]);   // (a NaN has just been noted)
                }
            }
#pragma unroll
            for (unsigned j = 0; j < 4u; ++j) {
                const bool finite = finite_f32(value[j]);
                good &= finite;
            }
            const bool live = (token < it.tokens) & (row < a.out_rows);
            bad |= live & !good;
            if (live & good) {
                if (whole_quads) {
                    *reinterpret_cast<float4 *>(out_row + row) = make_float4(value[0], value[1], value[2], value[3]);
                } else {
#pragma unroll
                    for (unsigned j = 0; j < 4u; ++j)
                        if (row + j < a.out_rows) out_row[row + j] = value[j];
                }
            }
        }
    }
    if (bad) raise_status(a.status, 1);
    }
    // Every run ends with all of its copies landed and all of its stores complete, whatever the next one looks like. A run with another
    // number of token blocks needs the former: it lays its stages out differently, so that its copies come from other waves than this run's
    // to the same bytes; the next run's opening barrier makes it hold for every wave.
    __builtin_amdgcn_s_waitcnt(0x0070u);   // vmcnt(0)
}

template <bool FUSED_UP, bool IMAGE>
__global__ __launch_bounds__(kRowThreads) void mfma_iq2_kernel(MfmaArgs a)
{
    extern __shared__ __align__(16) unsigned char mfma_lds[];
    if (lds_address_of(mfma_lds) != 0u) {   // the lookups address LDS by absolute byte offsets
        if (threadIdx.x == 0u) raise_status(a.status, 2);
        return;
    }
    const GroupedProblem &pr = a.pr;
    const unsigned tid = threadIdx.x;
    const bool fixed = pr.expert_ids == nullptr;
    const unsigned buckets = fixed ? 1u : (unsigned)pr.counts[0];

    // The buckets' populations are requested together (one round trip to memory instead of one per
    // bucket), and the tables built only where there is an item.
    // (a slot is read whether a bucket uses it or not: the number of buckets is on its way meanwhile)
    unsigned long long population_here = fixed ? pr.pairs : tid < 256u && tid < pr.experts ? pr.bucket_populations[tid] : 0ull;
    if (tid >= 256u || tid >= buckets) population_here = 0ull;
    // Full 64-pair tiles come first in the list of tiles, then the partial last tiles of more than 32
    // pairs, then those of fewer. Bucket b's first full tile is
    // the number of full tiles before it (a scan over the 256 bucket slots); its place in its
    // class of partial tiles (more than 32 pairs, or fewer) is its rank among the buckets of
    // that class, in bucket order, from ballots and per-wave totals.
    {
        const unsigned lane = tid & 63u, wave = tid >> 6;
        const unsigned full = tid < 256u ? (unsigned)(population_here / kTileTokens) : 0u;
        const unsigned rest = tid < 256u ? (unsigned)(population_here % kTileTokens) : 0u;
        const unsigned cls = rest <= few_pair_limit(a.few, population_here, kTrashBase + 48u) ? 2u : rest > 32u ? 0u : 1u;
        unsigned inclusive = wave_inclusive_sum_u32(full);
        unsigned rank[2];
#pragma unroll
        for (unsigned c = 0; c < 2u; ++c) {
            const unsigned long long members = __ballot(cls == c);
            rank[c] = (unsigned)__popcll(members & ((1ull << lane) - 1ull));
            if (lane == 0u && wave < 4u) lds_write_u32(kTrashBase + 16u + (c * 4u + wave) * 4u, (unsigned)__popcll(members));
        }
        if (lane == 63u && wave < 4u) lds_write_u32(kTrashBase + wave * 4u, inclusive);
        __syncthreads();
        if (tid < 256u) {
            unsigned before = 0u, class_before[2] = {0u, 0u};
            for (unsigned w = 0; w < wave; ++w) {
                before += lds_read_u32(kTrashBase + w * 4u);
                class_before[0] += lds_read_u32(kTrashBase + 16u + w * 4u);
                class_before[1] += lds_read_u32(kTrashBase + 16u + (4u + w) * 4u);
            }
            lds_write_u32(kTileStartBase + 4u * tid, before + inclusive - full);
            if (tid == 255u) lds_write_u32(kTileStartBase + 4u * 256u, before + inclusive);
            if (cls < 2u) lds_write_u16(kClassListBase + (cls * 256u + class_before[cls] + rank[cls]) * 2u, tid);
        }
        if (tid < 2u) {
            unsigned total = 0u;
            for (unsigned w = 0; w < 4u; ++w) total += lds_read_u32(kTrashBase + 16u + (tid * 4u + w) * 4u);
            lds_write_u32(kClassCountBase + 4u * tid, total);
        }
    }
    __syncthreads();
    if (buckets == 0u || buckets > 256u) {
        if (tid == 0u && buckets > 256u) raise_status(a.status, 2);
        return;
    }

    // The row tiles of all token tiles, a token tile's one after another, are dealt out in one piece of equal cost a
    // workgroup; a tile of 33 to 64 pairs costs four and one of fewer three (64 experts of 50 / 28 pairs: gate and up
    // 352 / 253 us, down 193 / 141). Where there are enough of the short ones, every workgroup has as many of the long ones as the
    // next, or one more, and short ones make up the difference (2048 uneven rows, gate and up: a workgroup in twenty
    // had 5 % more to do than the mean). Neighbouring pieces read the same weights where a bucket has several
    // token tiles, so they go to workgroups of one XCD (workgroups are dealt to the eight XCDs in turn; not so, 1231 -> 1270 us of 256
    // experts by 64).
    constexpr unsigned kItemRows = FUSED_UP ? 128u : 256u;
    constexpr unsigned kWide = 4u, kNarrow = 3u;                // costs of a row tile
    const unsigned row_tiles = (a.out_rows + kItemRows - 1u) / kItemRows;
    // (in 32 bits: the launch wrapper bounds the row tiles of all token tiles, and a division of 64 bits is a hundred instructions)
    const unsigned full_tiles = uniform32(lds_read_u32(kTileStartBase + 4u * buckets));
    const unsigned members[2] = {uniform32(lds_read_u32(kClassCountBase)), uniform32(lds_read_u32(kClassCountBase + 4u))};
    const unsigned wide = (full_tiles + members[0]) * row_tiles, narrow = members[1] * row_tiles, cost = kWide * wide + kNarrow * narrow;
    const unsigned who = gridDim.x % 8u ? blockIdx.x : (blockIdx.x % 8u) * (gridDim.x / 8u) + blockIdx.x / 8u;
    const unsigned cost_share = cost / gridDim.x, cost_rest = cost - cost_share * gridDim.x;
    const unsigned wide_share = wide / gridDim.x, wide_rest = wide - wide_share * gridDim.x;
    // what the workgroups before have
    auto cost_before = [&](unsigned workgroup) { return cost_share * workgroup + cost_rest * workgroup / gridDim.x; };
    auto wide_before = [&](unsigned workgroup) { return wide_share * workgroup + wide_rest * workgroup / gridDim.x; };
    const bool level = cost_share >= kWide * (wide_share + 1u);
    auto narrow_place = [&](unsigned workgroup) {
        return wide + (cost_before(workgroup) - kWide * wide_before(workgroup) + kNarrow - 1u) / kNarrow;
    };
    auto place_of = [&](unsigned workgroup) {                   // the first row tile of its piece, of its long ones
        const unsigned at = cost_before(workgroup);
        return level ? wide_before(workgroup)
             : at <= kWide * wide ? (at + kWide - 1u) / kWide : wide + (at - kWide * wide + kNarrow - 1u) / kNarrow;
    };
    auto uniform64 = [&](unsigned long long v) {
        return (unsigned long long)uniform32((unsigned)v) | ((unsigned long long)uniform32((unsigned)(v >> 32)) << 32);
    };
    unsigned at = uniform32(place_of(who)), end = uniform32(place_of(who + 1u));
    unsigned narrow_at = level ? uniform32(narrow_place(who)) : 0u;
    const unsigned narrow_end = level ? uniform32(narrow_place(who + 1u)) : 0u;
    if (at >= end && narrow_at >= narrow_end) return;
    mfma_tables_fill();
    __syncthreads();

    const bool ragged = a.out_rows % kItemRows != 0u;           // the last row tile is not whole
    while (at < end || narrow_at < narrow_end) {
        if (at >= end) {
            at = narrow_at;
            end = narrow_at = narrow_end;
        }
        const unsigned tile = uniform32(at / row_tiles);
        MfmaRun run;
        run.row_tile = at - tile * row_tiles;
        run.row_end = end - at < row_tiles - run.row_tile ? run.row_tile + (end - at) : row_tiles;
        if (ragged && run.row_end == row_tiles && run.row_end - run.row_tile > 1u) --run.row_end;
        at += run.row_end - run.row_tile;
        // which bucket the tile is of, and which of its tiles
        unsigned bucket, token_tile = 0u;
        const bool partial = tile >= full_tiles;                // the one behind the bucket's full tiles
        if (!partial) {
            unsigned low = 0u, high = buckets;                  // the last bucket whose first full tile is <= tile: it has it
            while (low + 1u < high) {
                const unsigned middle = (low + high) >> 1;
                if (lds_read_u32(kTileStartBase + 4u * middle) <= tile) low = middle;
                else high = middle;
            }
            bucket = low;
            token_tile = tile - lds_read_u32(kTileStartBase + 4u * low);
        } else {
            const unsigned rank = tile - full_tiles, c = rank < members[0] ? 0u : 1u;
            bucket = lds_read_u16(kClassListBase + (c * 256u + rank - (c ? members[0] : 0u)) * 2u);
        }
        bucket = uniform32(bucket);
        if (bucket >= buckets) {
            if (tid == 0u) raise_status(a.status, 2);
            continue;
        }
        const unsigned long long first = fixed ? 0ull : uniform64(pr.bucket_offsets[bucket]);
        const unsigned long long population = fixed ? pr.pairs : uniform64(pr.bucket_populations[bucket]);
        run.expert = fixed ? 0ull : uniform64(pr.expert_ids[bucket]);
        token_tile = uniform32(partial ? (unsigned)(population / kTileTokens) : token_tile);
        if (run.expert >= pr.experts || first + population > pr.pairs || (unsigned long long)token_tile * kTileTokens >= population) {
            if (tid == 0u) raise_status(a.status, 2);
            continue;
        }
        const unsigned long long tokens = population - (unsigned long long)token_tile * kTileTokens;
        run.pair0 = first + (unsigned long long)token_tile * kTileTokens;
        run.tokens = tokens < kTileTokens ? (unsigned)tokens : kTileTokens;
        if (run.tokens <= 32u) rows_run<FUSED_UP, 1u, IMAGE>(a, run);
        else rows_run<FUSED_UP, 2u, IMAGE>(a, run);
    }
}

template <bool FUSED_UP, bool IMAGE>
static int launch_mfma_variant(const MfmaArgs &a, hipStream_t stream)
{
    YVEX_ALLOW_DYNAMIC_LDS((mfma_iq2_kernel<FUSED_UP, IMAGE>), kMfmaLdsBytes);
    mfma_iq2_kernel<FUSED_UP, IMAGE><<<compute_units(), kRowThreads, kMfmaLdsBytes, stream>>>(a);
    return check_launch("moe_rows_mfma");
}

template <bool FUSED_UP>
static int launch_mfma(const MfmaArgs &a, hipStream_t stream)
{
    // (the kernel counts row tiles in 32 bits: whole tiles and one behind them a bucket, of which there are no more than pairs. The
    // outputs of so many are more than the card's memory)
    uint64_t buckets = 1u;
    if (a.pr.expert_ids) buckets = a.pr.experts < a.pr.pairs ? a.pr.experts : a.pr.pairs;
    const uint64_t token_tiles = a.pr.pairs / kTileTokens + (buckets < 256u ? buckets : 256u);
    if (token_tiles * ((uint64_t)a.out_rows / (FUSED_UP ? 128u : 256u) + 1u) >= 1ull << 30) return ST_BOUNDS;
    return a.image ? launch_mfma_variant<FUSED_UP, true>(a, stream)
                   : launch_mfma_variant<FUSED_UP, false>(a, stream);
}

// Expert matrices against the buckets of a worklist. The few-pair kernels (rows16.hip) take what a
// bucket holds behind its whole 64-pair tiles if that fits one of their tiles (12 pairs at width 7168, 16 up to about 5000; two tiles
// where few_pair_limit says so): such a tile takes them 1.3 us of the whole device for the 2 x 2048 x 4096 IQ2_XXS
// rows of an expert, and the 64-pair kernels, which pay for 32 token columns, 2.3 us; with two of theirs (2.6 us) it
// is the other way round. (Q4_K, and Q2_K down rows, without the few-pair kernels and with the present 64-pair ones: 150 / 420 even rows of
// 7168 by eight of 256 Q4_K experts 1442 / 1668 -> 1758 / 1899 us a layer, of 4096 by six in the model file's formats 577 / 660 -> 681 / 759; 2048 uneven rows 3460 -> 3519
// and 1523 -> 1534. Uneven rows of 4096 by six of Q4_K would gain: 1111 rows 1097 -> 1058.) A matrix that is alone (no worklist) is theirs where they come out at one round of
// their waves: 16 superblocks take 22 to 31 us then, and 45 us as 64-pair items, which are fewer than the
// compute units up to 1024 rows (4096 x 4096 IQ2_XXS by 128 rows 44 -> 24 us, 2048 x 7168 69 -> 35; 7168 x
// 7168 by 256 rows, two rounds, 102 us against 70).
struct RowsPlan {
    unsigned few;            // pairs of a full tile of the few-pair kernel, 0: it does not run
    bool many;               // the 64-pair kernel runs
};

static RowsPlan plan_rows(const GroupedProblem &pr, unsigned qtype, bool fused, int image, uint64_t width, uint64_t out_rows)
{
    const bool alone = pr.expert_ids == nullptr;
    unsigned few = rows16_tokens(pr, qtype, image != 0, fused, width, out_rows);
    if (alone && few && !rows16_one_round(pr, qtype, fused, few, out_rows)) few = 0u;
    return {few, !few || (!alone && pr.pairs > few)};
}

template <bool FUSED_UP>
static int launch_rows(MfmaArgs &a, unsigned qtype, hipStream_t stream, const GroupedProblem *beside = nullptr)
{
    const RowsPlan plan = plan_rows(a.pr, qtype, FUSED_UP, a.image, a.width, a.out_rows);
    a.few = plan.few;
    if (plan.many) {
        const int rc = qtype == QT_IQ2_XXS
            ? launch_mfma<FUSED_UP>(a, stream)
            : launch_q4k_rows_grouped(a.pr, qtype, FUSED_UP, a.width, a.out_rows, plan.few, beside, a.limit, a.status, stream);
        if (rc || !plan.few) return rc;
    }
    return launch_rows16_grouped(a.pr, qtype, a.image != 0, FUSED_UP, a.width, a.out_rows, a.pr.expert_ids ? kTileTokens : 0u,
                                 !a.plain_output, a.limit, a.status, stream);
}

// A plain projection through the row-batch kernel: every input row in one bucket of expert 0.
int launch_iq2_rows_dense(const uint8_t *encoded, uint64_t row_count, uint64_t row_width,
                          uint64_t row_bytes, const void *act_q8k, uint64_t input_rows, float *out,
                          bool round_bf16, int *status, hipStream_t stream, Publisher *publisher)
{
    int rc = check_matrix(QT_IQ2_XXS, row_width, row_bytes);
    if (rc) return rc;
    if (input_rows > 0xffffffffull || row_count > 0xffffffffull || row_count % 4u) return ST_BOUNDS;
    if (iq2_rows_small(row_count, row_width, input_rows))
        return launch_iq2_rows_small(encoded, row_count, row_width, row_bytes, act_q8k, input_rows, out, round_bf16, status, stream,
                                     publisher);
    yvex_hip_expert_weights w{};
    w.down = encoded;
    w.down_qtype = QT_IQ2_XXS;
    w.hidden = row_count;
    w.intermediate = row_width;
    w.down_row_bytes = row_bytes;
    w.down_expert_bytes = row_bytes * row_count;
    MfmaArgs a{};
    const WorklistView none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    fill_down_problem(a.pr, &w, act_q8k, 1, none, input_rows, 1u, out);
    a.width = (unsigned)row_width;
    a.out_rows = (unsigned)row_count;
    a.limit = 1.0;
    a.status = status;
    a.plain_output = round_bf16 ? 0 : 1;
    return launch_rows<false>(a, QT_IQ2_XXS, stream);
}

}  // namespace yvex

using namespace yvex;


extern "C" unsigned yvex_hip_moe_up_rows_launches(const yvex_hip_expert_weights *w, const void *act_q8k,
                                                  const uint64_t *expert_ids, uint64_t pairs, uint64_t topk,
                                                  uint64_t experts, float *intermediate)
{
    if (!w || pairs > 0xffffffffull) return 1u;
    GroupedProblem pr{};
    const WorklistView wl{nullptr, expert_ids, nullptr, nullptr, nullptr, nullptr};
    fill_up_problem(pr, w, act_q8k, 1, nullptr, wl, pairs, topk, experts, intermediate);
    const RowsPlan plan = plan_rows(pr, w->gate_qtype, true, w->gate_up_image, w->hidden, w->intermediate);
    return (plan.few ? 1u : 0u) + (plan.many ? 1u : 0u);
}

extern "C" unsigned yvex_hip_moe_down_rows_launches(const yvex_hip_expert_weights *w, const void *intermediate_q8k,
                                                    const uint64_t *expert_ids, uint64_t pairs, uint64_t experts,
                                                    float *pair_outputs)
{
    if (!w || pairs > 0xffffffffull) return 1u;
    GroupedProblem pr{};
    const WorklistView wl{nullptr, expert_ids, nullptr, nullptr, nullptr, nullptr};
    fill_down_problem(pr, w, intermediate_q8k, 1, wl, pairs, experts, pair_outputs);
    const RowsPlan plan = plan_rows(pr, w->down_qtype, false, w->down_image, w->intermediate, w->hidden);
    return (plan.few ? 1u : 0u) + (plan.many ? 1u : 0u);
}

// A shared expert's rows go along with the routed ones' where both are the 64-pair Q4_K and Q2_K kernel's, in the same shape.
static bool rows_join(const GroupedProblem &routed, const GroupedProblem &alone, const yvex_hip_expert_weights *w,
                      const yvex_hip_expert_weights *shared, bool fused)
{
    const unsigned qtype = fused ? w->gate_qtype : w->down_qtype;
    if (qtype == QT_IQ2_XXS || qtype != (fused ? shared->gate_qtype : shared->down_qtype) || w->hidden != shared->hidden ||
        w->intermediate != shared->intermediate)
        return false;
    const uint64_t width = fused ? w->hidden : w->intermediate, out_rows = fused ? w->intermediate : w->hidden;
    const RowsPlan plan = plan_rows(routed, qtype, fused, 0, width, out_rows);
    const RowsPlan other = plan_rows(alone, qtype, fused, 0, width, out_rows);
    return plan.many && other.many && !other.few && (uint64_t)routed.pairs + alone.pairs <= 1ull << 21;      // (the grid's second side)
}

static int prepare_up_rows(MfmaArgs &a, const yvex_hip_expert_weights *w, const void *act_q8k, const float *route_weights,
                           const WorklistView &wl, uint64_t pairs, uint64_t topk, uint64_t experts, double limit,
                           float *intermediate, int *status)
{
    if (!w || !w->gate || !w->up || !act_q8k || !intermediate || !status || !pairs || !topk ||
        !experts || !(limit > 0.0) || (wl.expert_ids && (!wl.bucket_offsets || !wl.bucket_populations || !wl.counts)))
        return ST_INVALID_ARG;
    if (w->gate_qtype != w->up_qtype || (w->gate_qtype != QT_IQ2_XXS && w->gate_qtype != QT_Q4_K))
        return ST_UNSUPPORTED;
    int rc = w->gate_up_image
        ? check_image_matrix(w->gate_qtype, w->hidden, w->gate_row_bytes, w->gate, w->gate_expert_bytes)
        : check_matrix(w->gate_qtype, w->hidden, w->gate_row_bytes);
    if (rc) return rc;
    if (w->up_row_bytes != w->gate_row_bytes) return ST_BOUNDS;
    if (w->gate_up_image && (((uintptr_t)w->up & 3u) || (w->up_expert_bytes & 3u))) return ST_INVALID_ARG;
    if (pairs > 0xffffffffull || w->intermediate > 0xffffffffull || w->intermediate % 4u) return ST_BOUNDS;
    fill_up_problem(a.pr, w, act_q8k, 1, route_weights, wl, pairs, topk, experts, intermediate);
    a.width = (unsigned)w->hidden;
    a.out_rows = (unsigned)w->intermediate;
    a.limit = limit;
    a.status = status;
    a.image = w->gate_up_image != 0;
    return ST_OK;
}

static int prepare_down_rows(MfmaArgs &a, const yvex_hip_expert_weights *w, const void *intermediate_q8k, const WorklistView &wl,
                             uint64_t pairs, uint64_t experts, float *pair_outputs, int *status)
{
    if (!w || !w->down || !intermediate_q8k || !pair_outputs || !status || !pairs || !experts ||
        (wl.expert_ids && (!wl.bucket_offsets || !wl.bucket_populations || !wl.counts)))
        return ST_INVALID_ARG;
    if (w->down_qtype != QT_IQ2_XXS && w->down_qtype != QT_Q4_K && w->down_qtype != QT_Q2_K) return ST_UNSUPPORTED;
    int rc = w->down_image
        ? check_image_matrix(w->down_qtype, w->intermediate, w->down_row_bytes, w->down, w->down_expert_bytes)
        : check_matrix(w->down_qtype, w->intermediate, w->down_row_bytes);
    if (rc) return rc;
    if (pairs > 0xffffffffull || w->hidden > 0xffffffffull || w->hidden % 4u) return ST_BOUNDS;
    fill_down_problem(a.pr, w, intermediate_q8k, 1, wl, pairs, experts, pair_outputs);
    a.width = (unsigned)w->intermediate;
    a.out_rows = (unsigned)w->hidden;
    a.limit = 1.0;
    a.status = status;
    a.image = w->down_image != 0;
    return ST_OK;
}

static const WorklistView kNoWorklist{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};

extern "C" int yvex_hip_moe_up_rows(const yvex_hip_expert_weights *w, const void *act_q8k,
                                    const float *route_weights, const uint64_t *order,
                                    const uint64_t *expert_ids, const uint64_t *bucket_offsets,
                                    const uint64_t *bucket_populations, const uint64_t *counts,
                                    uint64_t pairs, uint64_t topk, uint64_t experts, double limit,
                                    float *intermediate, int *status, yvex_hip_stream stream)
{
    MfmaArgs a{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, nullptr, counts};
    const int rc = prepare_up_rows(a, w, act_q8k, route_weights, wl, pairs, topk, experts, limit, intermediate, status);
    return rc ? rc : launch_rows<true>(a, w->gate_qtype, as_stream(stream));
}

extern "C" int yvex_hip_moe_down_rows(const yvex_hip_expert_weights *w, const void *intermediate_q8k,
                                      const uint64_t *order, const uint64_t *expert_ids,
                                      const uint64_t *bucket_offsets,
                                      const uint64_t *bucket_populations, const uint64_t *counts,
                                      uint64_t pairs, uint64_t experts, float *pair_outputs,
                                      int *status, yvex_hip_stream stream)
{
    MfmaArgs a{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, nullptr, counts};
    const int rc = prepare_down_rows(a, w, intermediate_q8k, wl, pairs, experts, pair_outputs, status);
    return rc ? rc : launch_rows<false>(a, w->down_qtype, as_stream(stream));
}

extern "C" int yvex_hip_moe_rows_join(const yvex_hip_expert_weights *w, const uint64_t *expert_ids, uint64_t pairs, uint64_t topk,
                                      uint64_t experts, const yvex_hip_expert_weights *shared, uint64_t shared_rows, int down)
{
    if (!w || !shared || !expert_ids || pairs > 0xffffffffull || shared_rows > 0xffffffffull || !shared_rows) return 0;
    GroupedProblem routed{}, alone{};
    const WorklistView wl{nullptr, expert_ids, nullptr, nullptr, nullptr, nullptr};
    if (down) {
        fill_down_problem(routed, w, nullptr, 1, wl, pairs, experts, nullptr);
        fill_down_problem(alone, shared, nullptr, 1, kNoWorklist, shared_rows, 1u, nullptr);
    } else {
        fill_up_problem(routed, w, nullptr, 1, nullptr, wl, pairs, topk, experts, nullptr);
        fill_up_problem(alone, shared, nullptr, 1, nullptr, kNoWorklist, shared_rows, 1u, 1u, nullptr);
    }
    return rows_join(routed, alone, w, shared, !down);
}

extern "C" int yvex_hip_moe_up_rows_joined(const yvex_hip_expert_weights *w, const void *act_q8k, const float *route_weights,
                                           const uint64_t *order, const uint64_t *expert_ids, const uint64_t *bucket_offsets,
                                           const uint64_t *bucket_populations, const uint64_t *counts, uint64_t pairs,
                                           uint64_t topk, uint64_t experts, double limit, float *intermediate,
                                           const yvex_hip_expert_weights *shared, uint64_t shared_rows,
                                           float *shared_intermediate, int *status, yvex_hip_stream stream)
{
    MfmaArgs a{}, alone{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, nullptr, counts};
    int rc = prepare_up_rows(a, w, act_q8k, route_weights, wl, pairs, topk, experts, limit, intermediate, status);
    if (!rc) rc = prepare_up_rows(alone, shared, act_q8k, nullptr, kNoWorklist, shared_rows, 1u, 1u, limit, shared_intermediate, status);
    if (!rc && (!expert_ids || !rows_join(a.pr, alone.pr, w, shared, true))) rc = ST_UNSUPPORTED;
    return rc ? rc : launch_rows<true>(a, w->gate_qtype, as_stream(stream), &alone.pr);
}

extern "C" int yvex_hip_moe_down_rows_joined(const yvex_hip_expert_weights *w, const void *intermediate_q8k, const uint64_t *order,
                                             const uint64_t *expert_ids, const uint64_t *bucket_offsets,
                                             const uint64_t *bucket_populations, const uint64_t *counts, uint64_t pairs,
                                             uint64_t experts, float *pair_outputs, const yvex_hip_expert_weights *shared,
                                             const void *shared_intermediate_q8k, uint64_t shared_rows, float *shared_outputs,
                                             int *status, yvex_hip_stream stream)
{
    MfmaArgs a{}, alone{};
    const WorklistView wl{order, expert_ids, bucket_offsets, bucket_populations, nullptr, counts};
    int rc = prepare_down_rows(a, w, intermediate_q8k, wl, pairs, experts, pair_outputs, status);
    if (!rc) rc = prepare_down_rows(alone, shared, shared_intermediate_q8k, kNoWorklist, shared_rows, 1u, shared_outputs, status);
    if (!rc && (!expert_ids || !rows_join(a.pr, alone.pr, w, shared, false))) rc = ST_UNSUPPORTED;
    return rc ? rc : launch_rows<false>(a, w->down_qtype, as_stream(stream), &alone.pr);
}
