// Expert projections of row batches whose buckets hold few pairs, on the int8 matrix cores of
// gfx950: IQ2_XXS rows (canonical bytes or the sweep image), Q4_K rows and the Q2_K rows of a down projection
// (src/backend/cuda/tensorcore.cu:378-702 is the reference's counterpart, for its own formats).
//
// With a handful of pairs to an expert the cost of the row-batch kernels (prefill.hip,
// rows_q4k.hip) is a tile's 32 token columns and the latency of two waves a SIMD in step behind
// a barrier a superblock: 256 experts with eight pairs each cost what they cost with 32. Here a
// tile is up to sixteen pairs of one bucket, and
//   * their whole Q8_K rows are resident in LDS, so nothing is staged inside the loop and no
//     wave waits for another: twelve waves a workgroup (eight for Q4_K and Q2_K rows) cover each
//     other's latency;
//   * a wave owns 32 weight rows (16 gate rows and the matching up rows when the SwiGLU is
//     fused) and walks them superblock by superblock, records coming straight into registers
//     ahead of their use, across row units as well;
//   * the products are V_MFMA_I32_16X16X64_I8: lane (r, q) = (lane % 16, lane / 16) owns weight
//     row r and a quarter of the superblock, four K chunks of sixteen values, in an order of K
//     that is the format's own (both operands follow it). One B fragment serves both row tiles.
//   * tiles times row units, in order, are cut into one piece of equal length a workgroup (short
//     ones end with their tiles); the waves of a workgroup draw units of its piece from a counter.
// Measured (256 experts, uniform routing; the row-batch kernels before, these after): gate/up of 4096 x 2048
// IQ2_XXS, eight pairs an expert, 620 -> 357 us, Q2_K down 358 -> 196; 7168 x 2048 IQ2_XXS, six pairs, 890 ->
// 608 and 503 -> 307; Q4_K 1115 -> 950 and 624 -> 509 (4.5 TB/s). IQ2_XXS has no pipe full (counters, 4096 x 2048 by
// eight pairs, 358 us: 1.21 GB or 3.4 TB/s, vector ALU 62 % busy, LDS 31 %, matrix cores 16 %; a wave waits for data
// 38 % of its time and for its turn to issue 29 %): load latency that three waves a SIMD do not cover, and
// more do not fit the registers. Coalescing four lanes to a row and passing
// the records through LDS, requesting four superblocks ahead, eight or sixteen waves (spills) were no faster.
// The arithmetic is that of the kernels named above, term by term: int8 limbs whose product sums
// are exact, one float term a superblock, added in double in superblock order, rounded to float
// once, so all kernel families publish the same bits.
#include "common.hpp"
#include "launch.hpp"
#include "grouped.hpp"
#include "lds_copy.hpp"
#include "iq2_limbs.hpp"
#include "kquant_limbs.hpp"

namespace yvex {

namespace {

typedef v4i v4i_dword __attribute__((aligned(4)));       // 16 bytes on a dword boundary

constexpr unsigned kSlots16 = 16u;                        // token columns of a tile
constexpr unsigned kMaxBlocks16 = 32u;                    // superblocks of a row
constexpr unsigned kBatchTiles = 8u;                      // tiles in LDS at a time
constexpr unsigned kLds16 = 160u * 1024u;
constexpr unsigned kIq2Image = 0x100u;                    // IQ2_XXS rows as the sweep image (no format number)

// LDS map (byte addresses; the dynamic block starts at LDS address 0). The IQ2_XXS tables come
// first: entry e owns the 256 bytes at 256 e, sixteen replicas of the level codes of codebook
// entry e in the first half; the second halves hold the sign selectors of fields 0-127, then the
// waves' row scales; sixteen replicas of the limb words of the sixteen scales follow. Last come the
// areas of the tiles at hand, each {out row, route weight} of its tokens, the activation scales
// [superblock][token], the minimum operands and the int8 payload.
//
// LDS reads: 64 banks, and a 16-byte read takes lanes 0-3, 12-15, 20-23 and 24-27 (and so on)
// together. With the image the table lookups of eight bytes use all banks: the lanes of odd quarters read
// the sign selectors with the instruction that reads codes for the even ones, and the codes with
// the other (the two are OR-ed): 2.3 cycles an instruction instead of 4.0, measured in a loop of such
// reads. The payload stands piece-major, [superblock][piece][token slot] with a multiple of four
// slots: 4.1 cycles instead of the 8.0 of token rows with XOR-ed piece positions.
template <unsigned QT> struct Map16 {
    static constexpr bool kIq2 = QT == QT_IQ2_XXS || QT == kIq2Image;
    static constexpr unsigned kWaves = kIq2 ? 12u : 8u;
    static constexpr unsigned kThreads = 64u * kWaves;
    static constexpr unsigned kLimbs = 65536u;
    static constexpr unsigned kStarts = kIq2 ? kLimbs + 4096u : 0u;       // first tile of a bucket (257 words)
    static constexpr unsigned kMisc = kStarts + 1040u;                    // wave totals, the counters below
    static constexpr unsigned kDrawn = kMisc + 64u, kBatch = kMisc + 68u; // units drawn; {tiles, units, units passed}
    static constexpr unsigned kTiles = kMisc + 112u;                      // Tile16 of every tile at hand
    static constexpr unsigned kScratch = kTiles + kBatchTiles * 32u;      // Q4_K, Q2_K: [wave][tile][d, dmin][16] f32
    static constexpr unsigned kAreas = (kScratch + (kIq2 ? 0u : kWaves * 256u) + 255u) & ~255u;
    // minimum operands of a superblock: Q4_K lo | hi limbs of a token's pair sums, Q2_K three pieces a token
    static constexpr unsigned kSumBytes = kIq2 ? 0u : QT == QT_Q4_K ? 256u : 768u;
    __host__ __device__ static constexpr unsigned area_bytes(unsigned blocks, unsigned slots)
    {
        return 128u + blocks * (64u + kSumBytes + 256u * slots);
    }
};

struct Rows16Args {
    GroupedProblem pr;
    unsigned blocks;         // superblocks per weight row
    unsigned out_rows;       // weight rows per expert
    unsigned tokens;         // of a full tile
    bool round;              // a plain projection's sums are rounded to bfloat16
    unsigned behind;         // what is served of a bucket: all of it (0), or its pairs behind whole tiles of
                             // this many, where they fit one tile here
    double limit;
    int *status;
};

struct Lane16 {
    unsigned r, q;           // weight row (token column) of the tile, quarter
};

// A tile at hand: units `start` .. of the batch are its row units from `first_unit` on.
struct Tile16 {
    unsigned start, first_unit, expert, pair0, live, area;
};

// ---- formats: a lane's bytes of one row's superblock ----
template <unsigned QT> struct Record16;

template <> struct Record16<kIq2Image> {
    static constexpr unsigned kBytes = 72u;
    unsigned head;           // fp16 scale | the four group scales of the lane's half << 16
    v4i body;                // groups 2 q and 2 q + 1: codebook bytes, sign bytes
    __device__ __forceinline__ void load(const unsigned char *base, unsigned row, bool, const Lane16 &l)
    {
        head = *reinterpret_cast<const unsigned *>(base + (row + 36u * (l.q >> 1)));
        body = *reinterpret_cast<const v4i_dword *>(base + (row + (36u * (l.q >> 1) + 16u * (l.q & 1u) + 4u)));
    }
};

// Canonical superblocks are 66 bytes and rows whole dwords, so the lane's sixteen bytes start two bytes
// into a dword in even superblocks and on one in odd ones: a window of five dwords, of which the odd
// superblocks use four (their fifth, which may lie behind the matrix, repeats the fourth).
template <> struct Record16<QT_IQ2_XXS> {
    static constexpr unsigned kBytes = 66u;
    v4i window;
    unsigned fifth;
    unsigned short scale;
    __device__ __forceinline__ void load(const unsigned char *base, unsigned row, bool odd, const Lane16 &l)
    {
        const unsigned at = row + (odd ? 2u : 0u) + 16u * l.q;
        window = *reinterpret_cast<const v4i_dword *>(base + at);
        fifth = *reinterpret_cast<const unsigned *>(base + (at + (odd ? 12u : 16u)));
        scale = *reinterpret_cast<const unsigned short *>(base + row);
    }
};

template <> struct Record16<QT_Q4_K> {
    static constexpr unsigned kBytes = 144u;
    v4i head;                // d | dmin << 16, the 12 scale bytes
    v4i codes[2];            // the 32 bytes of sub-blocks 2 q (low nibbles) and 2 q + 1
    __device__ __forceinline__ void load(const unsigned char *base, unsigned row, bool, const Lane16 &l)
    {
        head = *reinterpret_cast<const v4i_dword *>(base + row);
        codes[0] = *reinterpret_cast<const v4i_dword *>(base + (row + (32u * l.q + 16u)));
        codes[1] = *reinterpret_cast<const v4i_dword *>(base + (row + (32u * l.q + 32u)));
    }
    __device__ __forceinline__ unsigned scales_word() const { return (unsigned)head[0]; }
};

template <> struct Record16<QT_Q2_K> {
    static constexpr unsigned kBytes = 84u;
    v4i scales;              // (scale | minimum << 4) of the sixteen sub-blocks
    v4i codes;               // bytes 16 (q % 2) .. + 15 of code half q / 2
    unsigned dd;             // d | dmin << 16
    __device__ __forceinline__ void load(const unsigned char *base, unsigned row, bool, const Lane16 &l)
    {
        scales = *reinterpret_cast<const v4i_dword *>(base + row);
        codes = *reinterpret_cast<const v4i_dword *>(base + (row + (16u * l.q + 16u)));
        dd = *reinterpret_cast<const unsigned *>(base + (row + 80u));
    }
    __device__ __forceinline__ unsigned scales_word() const { return dd; }
};

template <unsigned QT, bool FUSED>
__global__ __launch_bounds__(Map16<QT>::kThreads) void rows16_kernel(Rows16Args a)
{
    using M = Map16<QT>;
    constexpr bool kIq2 = M::kIq2;
    extern __shared__ __align__(16) unsigned char rows16_lds[];
    if (lds_address_of(rows16_lds) != 0u) {      // operands are addressed by absolute LDS offsets
        if (threadIdx.x == 0u) raise_status(a.status, 2);
        return;
    }
    const GroupedProblem &pr = a.pr;
    auto uniform = [](unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); };
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = uniform(tid >> 6);
    const Lane16 l{lane & 15u, lane >> 4};
    const bool fixed = pr.expert_ids == nullptr;
    const unsigned buckets = fixed ? 1u : uniform((unsigned)pr.counts[0]);

    // ---- the first tile of every bucket (a scan over the 256 bucket slots) ----
    unsigned long long population_here = 0ull;
    if (tid < 256u && tid < buckets) population_here = fixed ? pr.pairs : pr.bucket_populations[tid];
    {
        const unsigned long long served = a.behind ? population_here % a.behind : population_here;
        const unsigned tiles = tid >= 256u || (a.behind && served > a.tokens) ? 0u
                                                                             : (unsigned)((served + a.tokens - 1u) / a.tokens);
        unsigned inclusive = tiles;
#pragma unroll
        for (int offset = 1; offset < 64; offset <<= 1) {
            const unsigned below = (unsigned)__shfl_up((int)inclusive, offset, kWave);
            if ((int)lane >= offset) inclusive += below;
        }
        if (lane == 63u && wave < 4u) lds_write_u32(M::kMisc + 4u * wave, inclusive);
        __syncthreads();
        if (tid < 256u) {
            for (unsigned w = 0; w < wave; ++w) inclusive += lds_read_u32(M::kMisc + 4u * w);
            lds_write_u32(M::kStarts + 4u * tid, inclusive - tiles);
            if (tid == 255u) lds_write_u32(M::kStarts + 1024u, inclusive);
        }
        __syncthreads();
    }
    if (buckets == 0u || buckets > 256u) {
        if (tid == 0u && buckets > 256u) raise_status(a.status, 2);
        return;
    }

    // ---- this workgroup's piece of the tiles' row units ----
    constexpr unsigned kUnitRows = FUSED ? 16u : 32u;
    const unsigned units = (a.out_rows + kUnitRows - 1u) / kUnitRows;
    const unsigned all_tiles = uniform(lds_read_u32(M::kStarts + 4u * buckets));
    if (!all_tiles) return;
    // A short piece that runs into a second tile takes twice its time where the two do not fit the LDS
    // together. So where a tile has several workgroups to itself and they come out at two rounds of
    // their waves or less, pieces end with their tiles (4096 x 4096 by 48 rows, three tiles: 39 -> 23 us);
    // longer ones are cut to equal lengths across tiles.
    const unsigned shares = gridDim.x / all_tiles;              // workgroups a tile
    unsigned long long at, end;
    if (shares && (units + shares - 1u) / shares <= 2u * M::kWaves) {
        const unsigned tile = blockIdx.x / shares, share = blockIdx.x % shares;
        if (tile >= all_tiles) return;
        at = (unsigned long long)tile * units + (unsigned long long)units * share / shares;
        end = (unsigned long long)tile * units + (unsigned long long)units * (share + 1u) / shares;
    } else {
        const unsigned long long total = (unsigned long long)all_tiles * units;
        at = total * blockIdx.x / gridDim.x;
        end = total * (blockIdx.x + 1u) / gridDim.x;
    }
    if (at == end) return;
    if constexpr (kIq2) {
        for (unsigned index = tid; index < 256u * 16u; index += M::kThreads)
            lds_write_uint2((index >> 4) * 256u + (index & 15u) * 8u, iq2_level_codes(index >> 4));
        for (unsigned index = tid; index < 128u * 16u; index += M::kThreads)
            lds_write_uint2((index >> 4) * 256u + 128u + (index & 15u) * 8u, iq2_sign_selectors(index >> 4));
        if (tid < 256u)
            lds_write_uint4(M::kLimbs + 16u * tid, iq2_limb_words(tid >> 4));
    }
    const unsigned scratch = kIq2 ? (160u + wave) * 256u + 128u : M::kScratch + wave * 256u;
    auto source_of = [&](unsigned long long ordered) { return pr.order ? pr.order[ordered] : ordered; };

    while (at < end) {
        // ---- the next tiles of the piece, as many as fit the LDS together: between them nobody
        // waits for anybody ----
        lds_barrier();       // every wave is done with the previous tiles
        if (wave == 0u) {
            const unsigned tile = (unsigned)(at / units) + lane;
            const unsigned first_unit = lane ? 0u : (unsigned)(at % units);
            const unsigned long long from = (unsigned long long)tile * units + first_unit;
            const bool mine = lane < kBatchTiles && from < end;
            unsigned count = 0u, passed = 0u, bytes = 0u;
            Tile16 t{0u, first_unit, 0u, 0u, 0u, 0u};
            if (mine) {
                passed = end - from < units - first_unit ? (unsigned)(end - from) : units - first_unit;
                unsigned low = 0u, high = buckets;       // the last bucket whose first tile is <= tile: it holds it
                while (low + 1u < high) {
                    const unsigned middle = (low + high) >> 1;
                    if (lds_read_u32(M::kStarts + 4u * middle) <= tile) low = middle;
                    else high = middle;
                }
                const unsigned long long population = fixed ? pr.pairs : pr.bucket_populations[low];
                const unsigned long long inside = a.behind ? population - population % a.behind
                    : (unsigned long long)(tile - lds_read_u32(M::kStarts + 4u * low)) * a.tokens;
                const unsigned long long pair0 = (fixed ? 0ull : pr.bucket_offsets[low]) + inside;
                const unsigned long long expert = fixed ? 0ull : pr.expert_ids[low];
                if (inside >= population || expert >= pr.experts || pair0 + (population - inside) > pr.pairs) {
                    raise_status(a.status, 2);
                } else {
                    count = passed;
                    t.expert = (unsigned)expert;
                    t.pair0 = (unsigned)pair0;
                    t.live = population - inside < a.tokens ? (unsigned)(population - inside) : a.tokens;
                    bytes = M::area_bytes(a.blocks, (t.live + 3u) & ~3u);
                }
            }
            // running totals over the eight lanes: area bytes, units, units passed
            unsigned bytes_to = bytes, count_to = count, passed_to = passed;
#pragma unroll
            for (int offset = 1; offset < (int)kBatchTiles; offset <<= 1) {
                const unsigned x = (unsigned)__shfl_up((int)bytes_to, offset, kWave), y = (unsigned)__shfl_up((int)count_to, offset, kWave),
                               z = (unsigned)__shfl_up((int)passed_to, offset, kWave);
                if ((int)lane >= offset) {
                    bytes_to += x;
                    count_to += y;
                    passed_to += z;
                }
            }
            const bool fits = mine && M::kAreas + bytes_to <= kLds16;        // (a tile of any size does alone)
            const unsigned tiles = (unsigned)__popcll(__ballot(fits));
            if (fits) {
                t.start = count_to - count;
                t.area = M::kAreas + bytes_to - bytes;
                lds_write_uint4(M::kTiles + 32u * lane, make_uint4(t.start, t.first_unit, t.expert, t.pair0));
                lds_write_uint2(M::kTiles + 32u * lane + 16u, make_uint2(t.live, t.area));
                if (lane + 1u == tiles) {
                    lds_write_u32(M::kBatch, tiles);
                    lds_write_u32(M::kBatch + 4u, count_to);
                    lds_write_u32(M::kBatch + 8u, passed_to);
                    lds_write_u32(M::kDrawn, M::kWaves);             // the unit drawn after every wave's first
                }
            }
        }
        __syncthreads();
        const unsigned tiles = uniform(lds_read_u32(M::kBatch)), drawable = uniform(lds_read_u32(M::kBatch + 4u));
        at += uniform(lds_read_u32(M::kBatch + 8u));
        auto tile_of = [&](unsigned index) {
            const unsigned from = M::kTiles + 32u * index;
            return Tile16{uniform(lds_read_u32(from)), uniform(lds_read_u32(from + 4u)), uniform(lds_read_u32(from + 8u)),
                          uniform(lds_read_u32(from + 12u)), uniform(lds_read_u32(from + 16u)), uniform(lds_read_u32(from + 20u))};
        };
        // parts of a tile's area
        const unsigned scales_at = 128u, sums_at = 128u + 64u * a.blocks, payload_at = sums_at + a.blocks * M::kSumBytes;

        // ---- their activation rows into LDS ----
        for (unsigned n = 0; n < tiles; ++n) {
            const Tile16 t = tile_of(n);
            if (!t.live) continue;
            auto token_row = [&](unsigned token) {
                const unsigned long long ordered = t.pair0 + token;
                const unsigned long long row = pr.act_by_ordered_pair ? ordered : source_of(ordered) / pr.topk;
                return (const unsigned char *)pr.activations + row * pr.act_stride;
            };
            const unsigned slots = (t.live + 3u) & ~3u;             // of a piece
            for (unsigned s = wave; s < slots * a.blocks / 4u; s += M::kWaves) {       // 64 pieces an instruction
                const unsigned piece = 64u * s + lane, column = piece / slots, slot = piece - column * slots;
                copy_to_lds_16(token_row(slot < t.live ? slot : 0u) + (unsigned long long)(column >> 4) * kQ8KBytes + 4u + 16u * (column & 15u),
                               uniform(t.area + payload_at + s * 1024u));
            }
            for (unsigned index = tid; index < kSlots16 * a.blocks; index += M::kThreads) {
                const unsigned sb = index >> 4, token = index & 15u;
                if (token >= t.live) continue;
                const unsigned char *block = token_row(token) + (unsigned long long)sb * kQ8KBytes;
                lds_write_u32(t.area + scales_at + 4u * index, *reinterpret_cast<const unsigned *>(block));
                if constexpr (!kIq2) {
                    const v4i first = *reinterpret_cast<const v4i_dword *>(block + 260u);
                    const v4i second = *reinterpret_cast<const v4i_dword *>(block + 276u);
                    const uint4 sums[2] = {make_uint4((unsigned)first[0], (unsigned)first[1], (unsigned)first[2], (unsigned)first[3]),
                                           make_uint4((unsigned)second[0], (unsigned)second[1], (unsigned)second[2], (unsigned)second[3])};
                    if constexpr (QT == QT_Q4_K) {
                        uint2 lo, hi;
                        q4k_bsum_limbs(sums, lo, hi);
                        lds_write_uint4(t.area + sums_at + 16u * index, make_uint4(lo.x, lo.y, hi.x, hi.y));
                    } else {
                        v4i piece[3];
                        q2k_bsum_pieces(sums, piece);
#pragma unroll
                        for (unsigned p = 0; p < 3u; ++p)
                            lds_write_uint4(t.area + sums_at + sb * 768u + p * 256u + token * 16u,
                                            make_uint4((unsigned)piece[p][0], (unsigned)piece[p][1], (unsigned)piece[p][2],
                                                       (unsigned)piece[p][3]));
                    }
                }
            }
            if (tid < t.live) {
                const unsigned long long ordered = t.pair0 + tid, source = source_of(ordered);
                lds_write_uint2(t.area + 8u * tid, make_uint2((unsigned)(pr.out_by_source_pair ? source : ordered),
                                                              __float_as_uint(pr.route_weights ? pr.route_weights[source] : 1.0f)));
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();

        // ---- units, one after another; the next one is known while this one runs, so that its
        // first records are requested with this one's last superblocks ----
        auto draw = [&]() {
            unsigned drawn = 0u;
            if (lane == 0u) drawn = atomicAdd(reinterpret_cast<unsigned *>(rows16_lds + M::kDrawn), 1u);
            return uniform(drawn);
        };
        // where a unit's rows lie: its expert's matrices and the lane's row of either row tile
        struct Rows {
            const unsigned char *base[2];
            unsigned row[2];
        };
        unsigned tile_index = 0u;                               // of the unit drawn last (they ascend)
        Tile16 drawn_tile = tile_of(0u);
        auto locate = [&](unsigned unit) {
            while (tile_index + 1u < tiles && uniform(lds_read_u32(M::kTiles + 32u * (tile_index + 1u))) <= unit) ++tile_index;
            drawn_tile = tile_of(tile_index);
            Rows rows;
            rows.base[0] = pr.gate + drawn_tile.expert * pr.expert_bytes;
            rows.base[1] = FUSED ? pr.up + drawn_tile.expert * pr.up_expert_bytes : rows.base[0];
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u) {
                unsigned row = (drawn_tile.first_unit + unit - drawn_tile.start) * kUnitRows + (FUSED ? 0u : 16u * u) + l.r;
                if (row >= a.out_rows) row = a.out_rows - 1u;       // a ragged edge repeats the last row
                rows.row[u] = row * (unsigned)pr.row_bytes;
            }
            return rows;
        };
        unsigned unit = wave;
        if (unit >= drawable) continue;
        Rows here = locate(unit);
        Tile16 tile = drawn_tile;
        unsigned next = draw();
        Rows ahead = here;
        if (next < drawable) ahead = locate(next);
        Record16<QT> rec[2][2];                  // [parity of the stream][row tile]
        auto request = [&](Record16<QT> (&into)[2], unsigned sb) {
            const bool past = sb >= a.blocks;
            const unsigned block = (past ? sb - a.blocks : sb) * Record16<QT>::kBytes;
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u)
                into[u].load(past ? ahead.base[u] : here.base[u], (past ? ahead.row[u] : here.row[u]) + block,
                             ((past ? sb - a.blocks : sb) & 1u) != 0u, l);
        };
        request(rec[0], 0u);
        request(rec[1], 1u);

        unsigned column, frag_pitch, frag_step, frag_at, sb = 0u;
        double acc[2][4];
        auto begin = [&]() {                     // the unit at hand, `tile`
            column = l.r < tile.live ? l.r : 0u;                    // padding repeats the first token
            frag_pitch = 16u * ((tile.live + 3u) & ~3u);            // from piece to piece
            frag_step = QT == QT_Q2_K ? 2u * frag_pitch : frag_pitch;       // from K chunk to K chunk
            frag_at = tile.area + payload_at + column * 16u + frag_pitch * (QT == QT_Q2_K ? 8u * (l.q >> 1) + (l.q & 1u) : 4u * l.q);
            sb = 0u;
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u)
#pragma unroll
                for (unsigned i = 0; i < 4u; ++i) acc[u][i] = 0.0;
        };
        begin();
        const v4i zero = {0, 0, 0, 0};

        auto superblock = [&](Record16<QT> (&w)[2]) {
            v4i lo[2] = {zero, zero}, hi[2] = {zero, zero};
            if constexpr (kIq2) {
                // lanes of odd quarters look signs up first
                const bool odd = QT == kIq2Image && (l.q & 1u) != 0u;
                const unsigned first_lane = l.r * 8u + (odd ? 128u : 0u), second_lane = first_lane ^ 128u;
                const unsigned lut_lane = M::kLimbs + l.r * 16u;
                const unsigned nibble = 8u + 8u * (l.q & 1u);
                unsigned first[2][2], second[2][2];              // [tile][group]: codebook and sign words
                unsigned scale16[2];
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    if constexpr (QT == kIq2Image) {
                        scale16[u] = w[u].head & 0xffffu;
#pragma unroll
                        for (unsigned g = 0; g < 2u; ++g) {
                            const unsigned grids = (unsigned)w[u].body[2u * g], aux = (unsigned)w[u].body[2u * g + 1u];
                            first[u][g] = odd ? aux : grids;
                            second[u][g] = odd ? grids : aux;
                        }
                    } else {
                        scale16[u] = w[u].scale;
                        const unsigned shift = sb & 1u ? 0u : 2u;
                        const unsigned d[5] = {(unsigned)w[u].window[0], (unsigned)w[u].window[1], (unsigned)w[u].window[2],
                                               (unsigned)w[u].window[3], w[u].fifth};
#pragma unroll
                        for (unsigned g = 0; g < 2u; ++g) {
                            first[u][g] = __builtin_amdgcn_alignbyte(d[2u * g + 1u], d[2u * g], shift);
                            second[u][g] = __builtin_amdgcn_alignbyte(d[2u * g + 2u], d[2u * g + 1u], shift);
                        }
                    }
                }
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u)
                    lds_write_u32(scratch + 64u * u + 4u * l.r, __float_as_uint(0.125f * f16_bits_to_float(scale16[u])));
                uint2 codes[2][2][2], signs[2][2][2];            // [chunk & 1][tile][subgroup]
                uint4 limbs[2][2];                               // [group & 1][tile]
                v4i frag[2];
                // the scale of a group in bits 8-11
                auto limb_field = [&](unsigned u, unsigned g) -> unsigned {
                    if constexpr (QT == kIq2Image) return w[u].head >> (nibble + 4u * g);
                    else return second[u][g] >> 20;
                };
                auto lookup = [&](unsigned m) {
                    frag[m & 1u] = lds_read_v4i(frag_at + m * frag_step);
#pragma unroll
                    for (unsigned u = 0; u < 2u; ++u) {
#pragma unroll
                        for (unsigned i = 0; i < 2u; ++i) {
                            const unsigned pick = 0x0c0c0400u + ((2u * (m & 1u) + i) << 8);
                            codes[m & 1u][u][i] =
                                lds_read_uint2(__builtin_amdgcn_perm(first[u][m >> 1], first_lane, pick));
                            // (the image's sign fields have bytes of their own, the canonical ones seven bits each)
                            const unsigned j = 2u * (m & 1u) + i, word = second[u][m >> 1];
                            signs[m & 1u][u][i] = lds_read_uint2(
                                QT == kIq2Image ? __builtin_amdgcn_perm(word, second_lane, pick)
                                                : ((j == 0u ? word << 8 : j == 1u ? word << 1 : word >> (7u * j - 8u)) & 0x7f00u) | second_lane);
                        }
                        if ((m & 1u) == 0u)
                            limbs[(m >> 1) & 1u][u] = lds_read_uint4((limb_field(u, m >> 1) & 0xf00u) | lut_lane);
                    }
                };
                lookup(0u);
#pragma unroll
                for (unsigned m = 0; m < 4u; ++m) {
                    if (m < 3u) lookup(m + 1u);
#pragma unroll
                    for (unsigned u = 0; u < 2u; ++u) {
                        const uint4 lw = limbs[(m >> 1) & 1u][u];
                        v4i a_lo, a_hi;
#pragma unroll
                        for (unsigned i = 0; i < 4u; ++i) {
                            const uint2 c = codes[m & 1u][u][i >> 1], s = signs[m & 1u][u][i >> 1];
                            const unsigned selector = i & 1u ? c.y | s.y : c.x | s.x;
                            a_lo[i] = (int)__builtin_amdgcn_perm(lw.y, lw.x, selector);
                            a_hi[i] = (int)__builtin_amdgcn_perm(lw.w, lw.z, selector);
                        }
                        lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, frag[m & 1u], lo[u], 0, 0, 0);
                        hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, frag[m & 1u], hi[u], 0, 0, 0);
                    }
                }
                request(w, sb + 2u);
                const float ts = __uint_as_float(lds_read_u32(tile.area + scales_at + 64u * sb + 4u * column));
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    const v4i rs = lds_read_v4i(scratch + 64u * u + 16u * l.q);
#pragma unroll
                    for (unsigned i = 0; i < 4u; ++i) {
                        const int sum = (hi[u][i] << 7) + lo[u][i];
                        const float term = __int_as_float(rs[i]) * ts * (float)sum;      // each product rounded to float
                        acc[u][i] += (double)term;
                    }
                }
            } else {
                // d and dmin of the rows, for the lanes that hold their sums
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    const unsigned dd = w[u].scales_word();
                    lds_write_u32(scratch + 128u * u + 4u * l.r, __float_as_uint(f16_bits_to_float(dd & 0xffffu)));
                    lds_write_u32(scratch + 128u * u + 64u + 4u * l.r, __float_as_uint(f16_bits_to_float(dd >> 16)));
                }
                v4i min_lo[2], min_hi[2];
                if constexpr (QT == QT_Q4_K) {
                    const v4i sums = lds_read_v4i(tile.area + sums_at + 256u * sb + 16u * column);
                    unsigned scales[2];
#pragma unroll
                    for (unsigned u = 0; u < 2u; ++u) {
                        const unsigned s0 = (unsigned)w[u].head[1], s1 = (unsigned)w[u].head[2], s2 = (unsigned)w[u].head[3];
                        const unsigned pack = l.q >> 1 ? (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u) : s0 & 0x3f3f3f3fu;
                        scales[u] = pack >> (16u * (l.q & 1u));          // of sub-blocks 2 q and 2 q + 1
                        // the minimums stand on the first quarter's lanes: against the low limbs of the
                        // pair sums (dwords 0-1 of `sums`), then against the high ones (dwords 2-3)
                        const int mn0 = l.q ? 0 : (int)(s1 & 0x3f3f3f3fu);
                        const int mn1 = l.q ? 0 : (int)(((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u));
                        min_lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{mn0, mn1, 0, 0}, sums, zero, 0, 0, 0);
                        min_hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{0, 0, mn0, mn1}, sums, zero, 0, 0, 0);
                    }
#pragma unroll
                    for (unsigned m = 0; m < 4u; ++m) {
                        const v4i frag = lds_read_v4i(frag_at + m * frag_step);
#pragma unroll
                        for (unsigned u = 0; u < 2u; ++u) {
                            const unsigned sc = (scales[u] >> (8u * (m >> 1))) & 255u;
                            v4i a_lo, a_hi;
#pragma unroll
                            for (unsigned i = 0; i < 4u; ++i) {
                                unsigned low_limbs, high_limbs;
                                q4k_limbs((unsigned)w[u].codes[m & 1u][i] >> (4u * (m >> 1)), sc, low_limbs, high_limbs);
                                a_lo[i] = (int)low_limbs;
                                a_hi[i] = (int)high_limbs;
                            }
                            lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, frag, lo[u], 0, 0, 0);
                            hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, frag, hi[u], 0, 0, 0);
                        }
                    }
                } else {
                    // quarter 0 holds the minimums against the sums' low three bits, quarters 1 and 2 hold
                    // eight times the minimums against the two halves of the rest
                    const v4i sums = lds_read_v4i(tile.area + sums_at + 768u * sb + 256u * (l.q < 2u ? l.q : 2u) + 16u * column);
                    unsigned scales[2][2];
#pragma unroll
                    for (unsigned u = 0; u < 2u; ++u) {
                        v4i mn;
#pragma unroll
                        for (unsigned i = 0; i < 4u; ++i) {
                            const unsigned four = ((unsigned)w[u].scales[i] >> 4) & 0x0f0f0f0fu;
                            mn[i] = (int)(l.q == 3u ? 0u : four << (l.q ? 3u : 0u));
                        }
                        min_lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mn, sums, zero, 0, 0, 0);
                        min_hi[u] = zero;
#pragma unroll
                        for (unsigned i = 0; i < 2u; ++i)      // sub-blocks 8 (q / 2) + 4 i .. + 3: every other byte from q % 2 on
                            scales[u][i] = (unsigned)(l.q >> 1 ? w[u].scales[2u + i] : w[u].scales[i]) >> (8u * (l.q & 1u));
                    }
#pragma unroll
                    for (unsigned m = 0; m < 4u; ++m) {
                        const v4i frag = lds_read_v4i(frag_at + m * frag_step);
#pragma unroll
                        for (unsigned u = 0; u < 2u; ++u) {
                            const unsigned sc = (scales[u][m >> 1] >> (16u * (m & 1u))) & 15u;
                            v4i limb;
#pragma unroll
                            for (unsigned i = 0; i < 4u; ++i) limb[i] = (int)q2k_limb((unsigned)w[u].codes[i] >> (2u * m), sc);
                            lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(limb, frag, lo[u], 0, 0, 0);
                        }
                    }
                }
                request(w, sb + 2u);
                const float ts = __uint_as_float(lds_read_u32(tile.area + scales_at + 64u * sb + 4u * column));
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    const v4i d = lds_read_v4i(scratch + 128u * u + 16u * l.q);
                    const v4i dmin = lds_read_v4i(scratch + 128u * u + 64u + 16u * l.q);
#pragma unroll
                    for (unsigned i = 0; i < 4u; ++i) {
                        const int dot = QT == QT_Q2_K ? lo[u][i] : (hi[u][i] << 3) + lo[u][i];
                        const int low = QT == QT_Q2_K ? min_lo[u][i] : (min_hi[u][i] << 7) + min_lo[u][i];
                        const float left = (ts * __int_as_float(d[i])) * (float)dot;
                        const float right = (ts * __int_as_float(dmin[i])) * (float)low;
                        acc[u][i] += (double)(left - right);
                    }
                }
            }
        };
        // Lane (token, q) holds the sums of rows 4 q .. 4 q + 3 of either row tile: sixteen bytes a store.
        auto publish = [&]() {
            const uint2 info = lds_read_uint2(tile.area + 8u * column);
            float *const out_row = pr.out + (unsigned long long)info.x * a.out_rows;
            const float limit_f32 = (float)a.limit;
            bool bad = false;
#pragma unroll
            for (unsigned u = 0; u < (FUSED ? 1u : 2u); ++u) {
                const unsigned row = (tile.first_unit + unit - tile.start) * kUnitRows + 16u * u + 4u * l.q;
                float value[4];
                bool good = true;
#pragma unroll
                for (unsigned i = 0; i < 4u; ++i) {
                    if constexpr (FUSED) {
                        value[i] = swiglu_bf16_fast((float)acc[0][i], (float)acc[1][i], __uint_as_float(info.y), a.limit,
                                                    limit_f32);
                    } else {
                        value[i] = (float)acc[u][i];
                        good &= finite_f32(value[i]);
                        if (a.round) value[i] = bf16_round_number(value[i]);      // (a NaN has just been noted)
                    }
                    good &= finite_f32(value[i]);
                }
                const bool kept = (l.r < tile.live) & (row < a.out_rows);
                bad |= kept & !good;
                if (kept & good) *reinterpret_cast<float4 *>(out_row + row) = make_float4(value[0], value[1], value[2], value[3]);
            }
            if (bad) raise_status(a.status, 1);
        };
        // Behind a superblock: on to the next, at a unit's end its results and the unit drawn before.
        // False when there is none.
        auto advance = [&]() -> bool {
            frag_at += 16u * frag_pitch;
            if (++sb < a.blocks) return true;
            publish();
            if (next >= drawable) return false;
            unit = next;
            here = ahead;
            tile = drawn_tile;
            begin();
            next = draw();
            if (next < drawable) ahead = locate(next);
            return true;
        };
        for (;;) {
            superblock(rec[0]);
            if (!advance()) break;
            superblock(rec[1]);
            if (!advance()) break;
        }
    }
}

template <unsigned QT, bool FUSED>
int launch_rows16(const Rows16Args &a, hipStream_t stream)
{
    YVEX_ALLOW_DYNAMIC_LDS((rows16_kernel<QT, FUSED>), kLds16);
    rows16_kernel<QT, FUSED><<<compute_units(), Map16<QT>::kThreads, kLds16, stream>>>(a);
    return check_launch("moe_rows16");
}

// Pairs of a full tile: as many Q8_K rows as the LDS holds, at most sixteen.
template <unsigned QT> unsigned tile_tokens16(unsigned blocks)
{
    unsigned tokens = kSlots16;
    while (tokens && Map16<QT>::kAreas + Map16<QT>::area_bytes(blocks, tokens) > kLds16) tokens -= 4u;
    return tokens;
}

}  // namespace

unsigned rows16_tokens(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, uint64_t width,
                       uint64_t out_rows)
{
    const uint64_t blocks = width / 256u, superblock = qtype == QT_IQ2_XXS ? (image ? 72u : 66u) : qtype == QT_Q4_K ? 144u : 84u;
    // superblocks are requested two ahead, across one unit's end
    if (width % 256u || blocks < 2u || blocks > kMaxBlocks16 || (qtype == QT_Q2_K && fused)) return 0u;
    // a lane addresses its rows with 32-bit offsets inside an expert and stores four rows at a time
    if (!out_rows || out_rows % 4u || problem.row_bytes != blocks * superblock || (problem.row_bytes & 3u) ||
        (fused && problem.up_row_bytes != problem.row_bytes) || out_rows * problem.row_bytes > 0xffffffffull)
        return 0u;
    if ((((uintptr_t)problem.gate | (uintptr_t)problem.up | (uintptr_t)problem.activations | problem.expert_bytes |
          problem.up_expert_bytes | problem.act_stride) & 3u) || ((uintptr_t)problem.out & 15u))
        return 0u;
    if (problem.experts > 256u && problem.expert_ids) return 0u;
    return qtype == QT_IQ2_XXS ? tile_tokens16<QT_IQ2_XXS>((unsigned)blocks)
         : qtype == QT_Q4_K    ? tile_tokens16<QT_Q4_K>((unsigned)blocks)
         : qtype == QT_Q2_K    ? tile_tokens16<QT_Q2_K>((unsigned)blocks) : 0u;
}

bool rows16_one_round(const GroupedProblem &problem, unsigned qtype, bool fused, unsigned tokens, uint64_t out_rows)
{
    const uint64_t units = (out_rows + (fused ? 15u : 31u)) / (fused ? 16u : 32u);
    const unsigned waves = qtype == QT_IQ2_XXS ? Map16<QT_IQ2_XXS>::kWaves : Map16<QT_Q4_K>::kWaves;
    return (problem.pairs + (uint64_t)tokens - 1u) / tokens * units <= (uint64_t)waves * compute_units();
}

int launch_rows16_grouped(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, unsigned width,
                          unsigned out_rows, unsigned behind, bool round, double limit, int *status, hipStream_t stream)
{
    const Rows16Args a{problem, width / 256u, out_rows, rows16_tokens(problem, qtype, image, fused, width, out_rows), round,
                       behind, limit, status};
    if (!a.tokens) return ST_UNSUPPORTED;
    if (qtype == QT_Q2_K) return launch_rows16<QT_Q2_K, false>(a, stream);
    if (qtype == QT_Q4_K)
        return fused ? launch_rows16<QT_Q4_K, true>(a, stream) : launch_rows16<QT_Q4_K, false>(a, stream);
    if (image)
        return fused ? launch_rows16<kIq2Image, true>(a, stream) : launch_rows16<kIq2Image, false>(a, stream);
    return fused ? launch_rows16<QT_IQ2_XXS, true>(a, stream) : launch_rows16<QT_IQ2_XXS, false>(a, stream);
}

}  // namespace yvex
