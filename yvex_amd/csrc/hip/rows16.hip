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
//     fused) and walks them superblock by superblock, their bytes loaded in runs ahead of their use (Run16 below),
//     across row units as well;
//   * the products are V_MFMA_I32_16X16X64_I8: lane (r, q) = (lane % 16, lane / 16) owns weight
//     row r and a quarter of the superblock, four K chunks of sixteen values, in an order of K
//     that is the format's own (both operands follow it). One B fragment serves both row tiles.
//   * IQ2_XXS table lookups run one step (a K chunk of a row tile) ahead of their use, the next superblock's
//     first ones ahead of this one's scaling; the scaling starts from sums that are floats already (kBias);
//   * tiles times row units, in order, are cut into one piece of equal length a workgroup (short
//     ones end with their tiles); the waves of a workgroup draw units of its piece from a counter.
// Measured (256 experts, uniform routing; lanes loading their own records before, runs after): gate/up of 4096 x 2048
// IQ2_XXS, nine pairs an expert, 370 -> 325 us, Q2_K down 208 -> 198; 7168 x 2048 IQ2_XXS, eight pairs, 592 -> 580 and
// 312 -> 292; Q4_K 947 -> 860 and 535 -> 505. Loads of the old kind with nothing computed took 314 us for the first of
// these (3.8 TB/s), in runs 209 (5.8). What bounds the IQ2_XXS rows now is the vector ALU: 237 instructions a wave and
// superblock at 4.7 cycles each with three waves a SIMD, 1190 of 1310 to 1490 cycles; the rest is the
// ends of tiles that do not fit the LDS together, where waves wait for each other. (Eight waves: two a SIMD, 5.0 cycles an
// instruction, 3 % behind; units cut at whole rounds of the waves: 1 % behind.)
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

// How weight bytes arrive: a run is the bytes of S superblocks of a row: pieces of sixteen bytes that hold codes, at the
// offsets that a lane's record begins at, and what else the superblocks have. The lanes of a load take consecutive
// pieces of consecutive rows, few cache lines an instruction (a lane loading its own record touches another
// row's lines than its neighbour, and the memory pipeline takes about two cycles a line). The pieces of sixteen
// rows pass through a window of LDS of the wave's own, piece k of row r at slot r ^ swizzle(k) of line k: writes of
// neighbouring rows and reads of sixteen both spread over the banks.
// IQ2_XXS runs of one superblock have their windows in the halves of the table entries from 128 on that hold no sign
// selectors, half the banks: without LDS of their own twelve pairs fit behind the tables at width 7168 (eight with it). Up to
// width 4096, where sixteen fit either way, the image comes two superblocks at a time through windows of their own:
// a load touches half the lines and all banks serve it (256 experts of nine pairs, gate/up of 4096 x 2048 325 us, 349
// one at a time; the other way round at 7168, ten pairs: 585, and 924 in the 64-pair kernels).
template <unsigned QT, unsigned S> struct Run16 {
    static constexpr bool kIq2 = QT == QT_IQ2_XXS || QT == kIq2Image, kAmongTables = kIq2 && S == 1u;
    static constexpr unsigned kPieces = (QT == QT_Q4_K ? 8u : 4u) * S;
    static constexpr unsigned kRows = 64u / kPieces, kLoads = 16u / kRows;      // of a load, for sixteen rows
    // behind the codes: Q4_K the superblock's first sixteen bytes, Q2_K scales, then d and dmin, of both row tiles
    static constexpr unsigned kExtra = 256u * kPieces, kWords = kExtra + 512u * S;
    static constexpr unsigned kWindow = kIq2 ? 2048u : kExtra + (QT == QT_Q4_K ? 512u : 640u * S);
    // Canonical IQ2_XXS superblocks are 66 bytes and rows whole dwords: an odd one's codes start on a dword, an even
    // one's two bytes into one, where the pieces start on the dword before.
    __device__ static __forceinline__ unsigned offset(unsigned run)
    {
        if constexpr (QT == QT_IQ2_XXS) return 66u * run + 2u * (run & 1u);
        else return S * (QT == QT_Q4_K ? 144u : QT == QT_Q2_K ? 84u : 72u) * run;
    }
    __device__ static __forceinline__ unsigned piece(unsigned k)
    {
        if constexpr (QT == kIq2Image) return 36u * (k >> 1) + 16u * (k & 1u) + 4u;
        else if constexpr (QT == QT_IQ2_XXS) return 16u * k;
        else if constexpr (QT == QT_Q4_K) return 16u * k + 16u;
        else return 84u * (k >> 2) + 16u * (k & 3u) + 16u;
    }
    __device__ static __forceinline__ unsigned place(unsigned window, unsigned k, unsigned row)
    {
        if constexpr (kAmongTables) {
            const unsigned slot = row ^ (4u * k);
            return window + 512u * k + 256u * (slot >> 3) + 16u * (slot & 7u);
        } else {
            // (a Q4_K lane reads pieces 2 q and 2 q + 1)
            const unsigned swizzle = QT == QT_Q4_K ? 8u * (k >> 2) + 4u * (k & 1u) + (k & 2u) : 16u / kPieces * k;
            return window + 256u * k + 16u * (row ^ swizzle);
        }
    }
};

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
template <unsigned QT, unsigned S> struct Map16 {
    static constexpr bool kIq2 = QT == QT_IQ2_XXS || QT == kIq2Image;
    static constexpr unsigned kWaves = kIq2 ? 12u : 8u;
    static constexpr unsigned kThreads = 64u * kWaves;
    static constexpr unsigned kLimbs = 65536u;
    static constexpr unsigned kStarts = kIq2 ? kLimbs + 4096u : 0u;       // first tile of a bucket (257 words)
    static constexpr unsigned kMisc = kStarts + 1040u;                    // wave totals, the counters below
    static constexpr unsigned kDrawn = kMisc + 64u, kBatch = kMisc + 68u; // units drawn; {tiles, units, units passed}
    static constexpr unsigned kTiles = kMisc + 112u;                      // Tile16 of every tile at hand
    static constexpr unsigned kScratch = kTiles + kBatchTiles * 32u;      // Q4_K, Q2_K: [wave][tile][d, dmin][16] f32
    // a run of the waves' rows
    static constexpr bool kAmongTables = Run16<QT, S>::kAmongTables;
    static constexpr unsigned kUnused = 128u * 256u + 128u;               // first of the unused half entries of the tables
    static constexpr unsigned kBehind = (kScratch + (kIq2 ? 0u : kWaves * 256u) + 255u) & ~255u;
    static constexpr unsigned kWindows = kAmongTables ? kUnused : kBehind;
    // IQ2_XXS, in unused half entries: the words before the halves of the image's records (canonical: the one dword of
    // a superblock that its pieces leave out), [row][half]; then the waves' row scales, [tile][16] f32
    static constexpr unsigned kHeads = kUnused + (kAmongTables ? kWaves * 2048u : 0u), kRowScales = kHeads + kWaves * S * 256u;
    static constexpr unsigned kAreas = kBehind + (kAmongTables ? 0u : kWaves * Run16<QT, S>::kWindow);
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
                             // this many, where few_pair_limit admits them
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

// ---- formats: a lane's bytes of one row's superblock, out of the wave's window ----
template <unsigned QT, unsigned S> struct Record16;

template <unsigned S> struct Record16<kIq2Image, S> {
    unsigned head;           // fp16 scale | the four group scales of the lane's half << 16
    v4i body;                // groups 2 q and 2 q + 1: codebook bytes, sign bytes
    __device__ __forceinline__ void read(unsigned window, unsigned heads, unsigned, unsigned s, const Lane16 &l)
    {
        const unsigned word = 2u * (S * l.r + s) + (l.q >> 1);
        head = lds_read_u32(heads + 256u * (word >> 5) + 4u * (word & 31u));
        body = lds_read_v4i(Run16<kIq2Image, S>::place(window, 4u * s + l.q, l.r));
    }
};

// A window of five dwords of which odd superblocks use four.
template <unsigned S> struct Record16<QT_IQ2_XXS, S> {
    v4i window;
    unsigned fifth;
    unsigned scale;
    __device__ __forceinline__ void read(unsigned at, unsigned heads, unsigned, unsigned parity, const Lane16 &l)
    {
        using Run = Run16<QT_IQ2_XXS, S>;
        window = lds_read_v4i(Run::place(at, l.q, l.r));
        fifth = parity ? 0u : lds_read_u32(l.q == 3u ? heads + 4u * l.r : Run::place(at, l.q + 1u, l.r));
        scale = parity ? lds_read_u16(heads + 4u * l.r + 2u) : lds_read_u16(Run::place(at, 0u, l.r));
    }
};

template <unsigned S> struct Record16<QT_Q4_K, S> {
    v4i head;                // d | dmin << 16, the 12 scale bytes
    v4i codes[2];            // the 32 bytes of sub-blocks 2 q (low nibbles) and 2 q + 1
    __device__ __forceinline__ void read(unsigned window, unsigned, unsigned u, unsigned, const Lane16 &l)
    {
        using Run = Run16<QT_Q4_K, S>;
        head = lds_read_v4i(window + Run::kExtra + 256u * u + 16u * l.r);
        codes[0] = lds_read_v4i(Run::place(window, 2u * l.q, l.r));
        codes[1] = lds_read_v4i(Run::place(window, 2u * l.q + 1u, l.r));
    }
    __device__ __forceinline__ unsigned scales_word() const { return (unsigned)head[0]; }
};

template <unsigned S> struct Record16<QT_Q2_K, S> {
    v4i scales;              // (scale | minimum << 4) of the sixteen sub-blocks
    v4i codes;               // bytes 16 (q % 2) .. + 15 of code half q / 2
    unsigned dd;             // d | dmin << 16
    __device__ __forceinline__ void read(unsigned window, unsigned, unsigned u, unsigned s, const Lane16 &l)
    {
        using Run = Run16<QT_Q2_K, S>;
        scales = lds_read_v4i(window + Run::kExtra + 256u * (S * u + s) + 16u * l.r);
        codes = lds_read_v4i(Run::place(window, 4u * s + l.q, l.r));
        dd = lds_read_u32(window + Run::kWords + 64u * (S * u + s) + 4u * l.r);
    }
    __device__ __forceinline__ unsigned scales_word() const { return dd; }
};

template <unsigned QT, bool FUSED, unsigned S>
__global__ __launch_bounds__((Map16<QT, S>::kThreads)) void rows16_kernel(Rows16Args a)
{
    using M = Map16<QT, S>;
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
    // ---- the first tile of every bucket (a scan over the 256 bucket slots; a slot is read whether a bucket uses it or not:
    // the number of buckets is on its way meanwhile) ----
    const unsigned long long held = fixed ? pr.pairs : tid < 256u && tid < pr.experts ? pr.bucket_populations[tid] : 0ull;
    const unsigned buckets = fixed ? 1u : uniform((unsigned)pr.counts[0]);
    const unsigned long long population_here = tid < 256u && tid < buckets ? held : 0ull;
    {
        const unsigned long long served = a.behind ? population_here % a.behind : population_here;
        const unsigned limit = a.behind ? few_pair_limit(a.tokens, population_here, M::kMisc + 16u) : 0u;
        const unsigned tiles = tid >= 256u || (a.behind && served > limit) ? 0u
                                                                             : (unsigned)((served + a.tokens - 1u) / a.tokens);
        unsigned inclusive = wave_inclusive_sum_u32(tiles);
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
    const unsigned scratch = (kIq2 ? M::kRowScales : M::kScratch) + wave * 256u;
    auto source_of = [&](unsigned long long ordered) { return pr.order ? pr.order[ordered] : ordered; };

    using Run = Run16<QT, S>;
    const unsigned window = uniform(M::kWindows + wave * Run::kWindow), heads = uniform(M::kHeads + wave * S * 256u);
    // the lane's pieces of sixteen rows' run: piece lane % kPieces of every kRows-th row; the rest of its bytes
    unsigned place[Run::kLoads], piece_at[Run::kLoads], head_at = 0u;
#pragma unroll
    for (unsigned i = 0; i < Run::kLoads; ++i) {
        const unsigned k = lane % Run::kPieces, row = Run::kRows * i + lane / Run::kPieces;
        place[i] = Run::place(window, k, row);
        piece_at[i] = row * (unsigned)pr.row_bytes + Run::piece(k);
    }
    if constexpr (QT == kIq2Image) head_at = (lane / (2u * S) & 15u) * (unsigned)pr.row_bytes + 36u * (lane % (2u * S));
    if constexpr (QT == QT_IQ2_XXS) head_at = l.r * (unsigned)pr.row_bytes;
    if constexpr (QT == QT_Q4_K) head_at = (FUSED ? l.r : lane & 31u) * (unsigned)pr.row_bytes;
    if constexpr (QT == QT_Q2_K) head_at = (l.r + 16u * (lane / (16u * S) & 1u)) * (unsigned)pr.row_bytes + 84u * (l.q & (S - 1u));
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
                const unsigned long long inside = (a.behind ? population - population % a.behind : 0ull) +
                                                  (unsigned long long)(tile - lds_read_u32(M::kStarts + 4u * low)) * a.tokens;
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
        // where the row tiles of a unit lie (a ragged edge takes rows that the unit before has, too: the same bits)
        struct Rows {
            const unsigned char *base[2];
        };
        auto first_row = [&](const Tile16 &t, unsigned unit) {
            return min((t.first_unit + unit - t.start) * kUnitRows, a.out_rows - kUnitRows);
        };
        unsigned tile_index = 0u;                               // of the unit drawn last (they ascend)
        Tile16 drawn_tile = tile_of(0u);
        unsigned tile_end = tiles > 1u ? uniform(lds_read_u32(M::kTiles + 32u)) : drawable;
        auto locate = [&](unsigned unit) {
            while (unit >= tile_end) {
                drawn_tile = tile_of(++tile_index);
                tile_end = tile_index + 1u < tiles ? uniform(lds_read_u32(M::kTiles + 32u * (tile_index + 1u))) : drawable;
            }
            const unsigned long long row = (unsigned long long)first_row(drawn_tile, unit) * pr.row_bytes;
            Rows rows;
            rows.base[0] = pr.gate + drawn_tile.expert * pr.expert_bytes + row;
            rows.base[1] = FUSED ? pr.up + drawn_tile.expert * pr.up_expert_bytes + row : rows.base[0] + 16u * pr.row_bytes;
            return rows;
        };
        unsigned unit = wave;
        if (unit >= drawable) continue;
        Rows here = locate(unit);
        Tile16 tile = drawn_tile;
        unsigned next = draw();
        Rows ahead = here;
        if (next < drawable) ahead = locate(next);
        // the run that comes next
        struct Staged {
            v4i piece[2][Run::kLoads], head;
            unsigned word[2];
        } staged;
        const unsigned runs = a.blocks / S;
        auto request = [&](unsigned run) {       // of the unit at hand, or behind its end of the one drawn before
            const bool past = run >= runs;
            const unsigned here_run = past ? run - runs : run, from = Run::offset(here_run);
            const unsigned char *const base[2] = {(past ? ahead.base[0] : here.base[0]) + from,
                                                  (past ? ahead.base[1] : here.base[1]) + from};
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u) {
                if constexpr (kIq2)
                    staged.word[u] = *reinterpret_cast<const unsigned *>(base[u] + (QT == kIq2Image ? 0 : here_run & 1u ? -4 : 64) + head_at);
#pragma unroll
                for (unsigned i = 0; i < Run::kLoads; ++i)
                    staged.piece[u][i] = *reinterpret_cast<const v4i_dword *>(base[u] + piece_at[i]);
            }
            if constexpr (QT == QT_Q4_K) {
                // gate heads on the lanes of the even quarters, up heads on the others (plain rows: of both row tiles)
                const unsigned long long to_up = FUSED && (l.q & 1u) ? (unsigned long long)(base[1] - base[0]) : 0ull;
                staged.head = *reinterpret_cast<const v4i_dword *>(base[0] + to_up + head_at);
            }
            if constexpr (QT == QT_Q2_K) {
                staged.head = *reinterpret_cast<const v4i_dword *>(base[0] + head_at);
                staged.word[0] = *reinterpret_cast<const unsigned *>(base[0] + (head_at + 80u));
            }
        };
        request(0u);

        // where a tile's activations stand for a lane. Lanes behind the last token, whose results nobody takes, read
        // what their neighbours read, with which they share the banks' cycle.
        struct Columns {
            unsigned column, pitch, frag_at, scale_at;     // pitch: from piece to piece
        };
        auto columns_of = [&](const Tile16 &t) {
            const bool lives = l.r < t.live;
            const unsigned q = lives ? l.q : l.q & 2u;
            Columns c;
            c.column = lives ? l.r : 0u;
            c.pitch = 16u * ((t.live + 3u) & ~3u);
            c.frag_at = t.area + payload_at + (lives ? l.r : l.r & 3u) * 16u + c.pitch * (QT == QT_Q2_K ? 8u * (q >> 1) + (q & 1u) : 4u * q);
            c.scale_at = t.area + scales_at + 4u * c.column;
            return c;
        };
        Columns c = columns_of(tile), c_ahead = columns_of(drawn_tile);
        unsigned sb = 0u;
        double acc[2][4];
        auto begin = [&]() {                     // the unit at hand
            sb = 0u;
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u)
#pragma unroll
                for (unsigned i = 0; i < 4u; ++i) acc[u][i] = 0.0;
        };
        begin();
        // The IQ2_XXS limbs' sums start from the bits of 1.5 * 2^23: |sum| stays below 2^22 (low limbs 256 * 64 * 127), so
        // a result's bits are the float 1.5 * 2^23 + sum.
        constexpr float kBias = 12582912.0f;
        const int start_bits = kIq2 ? __float_as_int(kBias) : 0;
        const v4i start = {start_bits, start_bits, start_bits, start_bits}, zero = {0, 0, 0, 0};

        // A superblock's sums (int32, exact) and the scales that make its float terms of them.
        struct Sums {
            v4i lo[2], hi[2], min_lo[2], min_hi[2];
        };
        struct Scales {
            float token;
            v4i d[2], dmin[2];
        };
        auto scales_here = [&]() {
            Scales r;
            r.token = __uint_as_float(lds_read_u32(c.scale_at + 64u * sb));
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u) {
                r.d[u] = lds_read_v4i(scratch + (kIq2 ? 64u : 128u) * u + 16u * l.q);
                if constexpr (!kIq2) r.dmin[u] = lds_read_v4i(scratch + 128u * u + 64u + 16u * l.q);
            }
            return r;
        };
        auto settle = [&](const Sums &x, const Scales &r) {
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u)
#pragma unroll
                for (unsigned i = 0; i < 4u; ++i) {
                    if constexpr (kIq2) {
                        // 128 hi - kBias is exact, and so the float of 128 hi + lo comes from one rounding
                        const float sum = __builtin_fmaf(__int_as_float(x.hi[u][i]), 128.0f, -129.0f * kBias) + __int_as_float(x.lo[u][i]);
                        const float term = __int_as_float(r.d[u][i]) * r.token * sum;      // each product rounded to float
                        acc[u][i] += (double)term;
                    } else {
                        const int dot = QT == QT_Q2_K ? x.lo[u][i] : (x.hi[u][i] << 3) + x.lo[u][i];
                        const int low = QT == QT_Q2_K ? x.min_lo[u][i] : (x.min_hi[u][i] << 7) + x.min_lo[u][i];
                        const float left = (r.token * __int_as_float(r.d[u][i])) * (float)dot;
                        const float right = (r.token * __int_as_float(r.dmin[u][i])) * (float)low;
                        acc[u][i] += (double)(left - right);
                    }
                }
        };

        // IQ2_XXS: a superblock's table words and the lookups in flight.
        // Lanes of odd quarters look signs up first.
        const bool odd_quarter = QT == kIq2Image && (l.q & 1u) != 0u;
        const unsigned first_lane = l.r * 8u + (odd_quarter ? 128u : 0u), second_lane = first_lane ^ 128u;
        const unsigned lut_lane = M::kLimbs + l.r * 16u;
        const unsigned nibble = 8u + 8u * (l.q & 1u);
        unsigned first[2][2], second[2][2], words[2];            // [tile][group]: codebook and sign words
        uint2 codes[2][2], signs[2][2];                          // [row tile][subgroup]
        v4i limbs[2][2];                                         // [group & 1][tile]
        v4i frag[kIq2 ? 2 : 4];
        unsigned frag_at = c.frag_at, pitch = c.pitch;           // of the superblock that is ready
        const unsigned chunk_pieces = QT == QT_Q2_K ? 2u : 1u;   // from K chunk to K chunk
        auto lookup = [&](unsigned step) {                       // K chunk step / 2 of row tile step % 2
            const unsigned m = step >> 1, u = step & 1u;
            if (u == 0u) frag[m & 1u] = lds_read_v4i(frag_at + m * pitch);
            // the scale of a group in bits 8-11
            if ((m & 1u) == 0u) {
                const unsigned field = QT == kIq2Image ? words[u] >> (nibble + 4u * (m >> 1)) : second[u][m >> 1] >> 20;
                limbs[(m >> 1) & 1u][u] = lds_read_v4i((field & 0xf00u) | lut_lane);
            }
#pragma unroll
            for (unsigned i = 0; i < 2u; ++i) {
                const unsigned j = 2u * (m & 1u) + i, pick = 0x0c0c0400u + (j << 8), word = second[u][m >> 1];
                codes[u][i] = lds_read_uint2(__builtin_amdgcn_perm(first[u][m >> 1], first_lane, pick));
                // (the image's sign fields have bytes of their own, the canonical ones seven bits each)
                signs[u][i] = lds_read_uint2(
                    QT == kIq2Image ? __builtin_amdgcn_perm(word, second_lane, pick)
                                    : ((j == 0u ? word << 8 : j == 1u ? word << 1 : word >> (7u * j - 8u)) & 0x7f00u) | second_lane);
            }
        };
        // A superblock is next: its row scales where the lanes that will hold its sums find them, its first lookups.
        auto ready = [&](const Record16<QT, S> (&w)[2], unsigned parity) {
            if constexpr (kIq2) {
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    unsigned scale16;
                    if constexpr (QT == kIq2Image) {
                        words[u] = w[u].head;
                        scale16 = w[u].head & 0xffffu;
#pragma unroll
                        for (unsigned g = 0; g < 2u; ++g) {
                            const unsigned grids = (unsigned)w[u].body[2u * g], aux = (unsigned)w[u].body[2u * g + 1u];
                            first[u][g] = odd_quarter ? aux : grids;
                            second[u][g] = odd_quarter ? grids : aux;
                        }
                    } else {
                        scale16 = w[u].scale;
                        const unsigned d[5] = {(unsigned)w[u].window[0], (unsigned)w[u].window[1], (unsigned)w[u].window[2],
                                               (unsigned)w[u].window[3], w[u].fifth};
#pragma unroll
                        for (unsigned g = 0; g < 2u; ++g) {
                            first[u][g] = parity ? d[2u * g] : __builtin_amdgcn_alignbyte(d[2u * g + 1u], d[2u * g], 2u);
                            second[u][g] = parity ? d[2u * g + 1u] : __builtin_amdgcn_alignbyte(d[2u * g + 2u], d[2u * g + 1u], 2u);
                        }
                    }
                    lds_write_u32(scratch + 64u * u + 4u * l.r, __float_as_uint(0.125f * f16_bits_to_float(scale16)));
                }
                lookup(0u);
            } else {
#pragma unroll
                for (unsigned u = 0; u < 2u; ++u) {
                    const unsigned dd = w[u].scales_word();
                    lds_write_u32(scratch + 128u * u + 4u * l.r, __float_as_uint(f16_bits_to_float(dd & 0xffffu)));
                    lds_write_u32(scratch + 128u * u + 64u + 4u * l.r, __float_as_uint(f16_bits_to_float(dd >> 16)));
                }
            }
        };

        // The staged run through the window into the lanes' records, and the one behind it requested.
        Record16<QT, S> rec[S][2];
        unsigned run = 0u;                       // of the unit at hand
        auto turn_over = [&](unsigned behind, [[maybe_unused]] unsigned parity) {
            if constexpr (QT == QT_Q4_K) lds_write_v4i(window + Run::kExtra + 16u * (lane & 31u), staged.head);
            if constexpr (QT == QT_Q2_K) {
                lds_write_v4i(window + Run::kExtra + 16u * (lane % (32u * S)), staged.head);
                lds_write_u32(window + Run::kWords + 4u * (lane % (32u * S)), staged.word[0]);
            }
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u) {
#pragma unroll
                for (unsigned i = 0; i < Run::kLoads; ++i) lds_write_v4i(place[i], staged.piece[u][i]);
                if constexpr (kIq2) lds_write_u32(heads + 256u * (S - 1u) * (lane >> 5) + 4u * (lane & (QT == kIq2Image ? 31u : 15u)), staged.word[u]);
#pragma unroll
                for (unsigned s = 0; s < S; ++s) rec[s][u].read(window, heads, u, QT == QT_IQ2_XXS ? parity : s, l);
            }
            request(behind);
        };
        // One superblock, an odd one by `parity`; `turn` if it is its run's last.
        auto superblock = [&](const Record16<QT, S> (&record)[2], bool turn, unsigned parity) {
            [[maybe_unused]] const Record16<QT, S> w[2] = {record[0], record[1]};
            Sums x;
#pragma unroll
            for (unsigned u = 0; u < 2u; ++u) {
                x.lo[u] = x.hi[u] = start;
                x.min_lo[u] = x.min_hi[u] = zero;
            }
            if constexpr (kIq2) {
#pragma unroll
                for (unsigned step = 0; step < 8u; ++step) {
                    const unsigned m = step >> 1, u = step & 1u;
                    if (step < 7u) lookup(step + 1u);
                    else if (turn) turn_over(run + 2u, parity ^ 1u);
                    __builtin_amdgcn_sched_barrier(0);
                    const v4i lw = limbs[(m >> 1) & 1u][u];
                    v4i a_lo, a_hi;
#pragma unroll
                    for (unsigned i = 0; i < 4u; ++i) {
                        const uint2 code = codes[u][i >> 1], sign = signs[u][i >> 1];
                        const unsigned selector = i & 1u ? code.y | sign.y : code.x | sign.x;
                        a_lo[i] = (int)__builtin_amdgcn_perm((unsigned)lw[1], (unsigned)lw[0], selector);
                        a_hi[i] = (int)__builtin_amdgcn_perm((unsigned)lw[3], (unsigned)lw[2], selector);
                    }
                    x.lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, frag[m & 1u], x.lo[u], 0, 0, 0);
                    x.hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, frag[m & 1u], x.hi[u], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                const v4i sums = lds_read_v4i(tile.area + sums_at + M::kSumBytes * sb + (QT == QT_Q2_K ? 256u * (l.q < 2u ? l.q : 2u) : 0u)
                                              + 16u * c.column);
#pragma unroll
                for (unsigned m = 0; m < 4u; ++m) frag[m] = lds_read_v4i(frag_at + m * chunk_pieces * pitch);
                if (turn) turn_over(run + 2u, parity ^ 1u);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (QT == QT_Q4_K) {
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
                        x.min_lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{mn0, mn1, 0, 0}, sums, zero, 0, 0, 0);
                        x.min_hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{0, 0, mn0, mn1}, sums, zero, 0, 0, 0);
                    }
#pragma unroll
                    for (unsigned m = 0; m < 4u; ++m) {
#pragma unroll
                        for (unsigned u = 0; u < 2u; ++u) {
                            const unsigned sc = (scales[u] >> (8u * (m >> 1))) & 255u;
                            v4i a_lo, a_hi;
#pragma unroll
                            for (unsigned i = 0; i < 4u; ++i) {
                                unsigned low_limbs, high_limbs;
                                q4k_limbs((unsigned)w[u].codes[m & 1u][i] >> (4u * (m >> 1)), (unsigned short)(sc & 7u),
                                          (unsigned short)(sc >> 3), low_limbs, high_limbs);
                                a_lo[i] = (int)low_limbs;
                                a_hi[i] = (int)high_limbs;
                            }
                            x.lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_lo, frag[m], x.lo[u], 0, 0, 0);
                            x.hi[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_hi, frag[m], x.hi[u], 0, 0, 0);
                        }
                    }
                } else {
                    // quarter 0 holds the minimums against the sums' low three bits, quarters 1 and 2 hold
                    // eight times the minimums against the two halves of the rest
                    unsigned scales[2][2];
#pragma unroll
                    for (unsigned u = 0; u < 2u; ++u) {
                        v4i mn;
#pragma unroll
                        for (unsigned i = 0; i < 4u; ++i) {
                            const unsigned four = ((unsigned)w[u].scales[i] >> 4) & 0x0f0f0f0fu;
                            mn[i] = (int)(l.q == 3u ? 0u : four << (l.q ? 3u : 0u));
                        }
                        x.min_lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mn, sums, zero, 0, 0, 0);
#pragma unroll
                        for (unsigned i = 0; i < 2u; ++i)      // sub-blocks 8 (q / 2) + 4 i .. + 3: every other byte from q % 2 on
                            scales[u][i] = (unsigned)(l.q >> 1 ? w[u].scales[2u + i] : w[u].scales[i]) >> (8u * (l.q & 1u));
                    }
#pragma unroll
                    for (unsigned m = 0; m < 4u; ++m) {
#pragma unroll
                        for (unsigned u = 0; u < 2u; ++u) {
                            const unsigned sc = (scales[u][m >> 1] >> (16u * (m & 1u))) & 15u;
                            v4i limb;
#pragma unroll
                            for (unsigned i = 0; i < 4u; ++i) limb[i] = (int)q2k_limb((unsigned)w[u].codes[i] >> (2u * m), sc);
                            x.lo[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(limb, frag[m], x.lo[u], 0, 0, 0);
                        }
                    }
                }
            }
            return x;
        };
        // Lane (token, q) holds the sums of rows 4 q .. 4 q + 3 of either row tile: sixteen bytes a store.
        auto publish = [&]() {
            const uint2 info = lds_read_uint2(tile.area + 8u * c.column);
            float *const out_row = pr.out + (unsigned long long)info.x * a.out_rows;
            const float limit_f32 = (float)a.limit;
            bool bad = false;
#pragma unroll
            for (unsigned u = 0; u < (FUSED ? 1u : 2u); ++u) {
                const unsigned row = first_row(tile, unit) + 16u * u + 4u * l.q;
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
                        if (a.round) value[i] = bf16_round(value[i]);      // (a NaN has just been noted)
                    }
                    good &= finite_f32(value[i]);
                }
                const bool kept = l.r < tile.live;
                bad |= kept & !good;
                if (kept & good) *reinterpret_cast<float4 *>(out_row + row) = make_float4(value[0], value[1], value[2], value[3]);
            }
            if (bad) raise_status(a.status, 1);
        };
        // Behind a run's last superblock: its successor made ready while the sums settle, at a unit's end that of the
        // next unit; the results go out then. False when no unit is left.
        auto advance = [&](const Sums &x, unsigned parity) -> bool {
            const bool ends = ++run == runs;
            const Scales r = scales_here();
            frag_at = ends ? c_ahead.frag_at : frag_at + 16u * pitch;
            pitch = ends ? c_ahead.pitch : pitch;
            ready(rec[0], parity);
            settle(x, r);
            ++sb;
            if (ends) {
                publish();
                if (next >= drawable) return false;
                unit = next;
                here = ahead;
                tile = drawn_tile;
                c = c_ahead;
                run = 0u;
                begin();
                next = draw();
                if (next < drawable) {
                    ahead = locate(next);
                    c_ahead = columns_of(drawn_tile);
                }
            }
            return true;
        };
        turn_over(1u, 0u);
        ready(rec[0], 0u);
        for (;;) {
            const Sums x = superblock(rec[0], S == 1u, 0u);
            if constexpr (S == 1u) {
                if (!advance(x, 1u)) break;
            } else {
                const Scales r = scales_here();
                frag_at += 16u * pitch;
                ready(rec[1], 1u);
                settle(x, r);
                ++sb;
            }
            if (!advance(superblock(rec[S - 1u], true, 1u), 0u)) break;
        }
    }
}

template <unsigned QT, bool FUSED, unsigned S>
int launch_rows16(const Rows16Args &a, hipStream_t stream)
{
    YVEX_ALLOW_DYNAMIC_LDS((rows16_kernel<QT, FUSED, S>), kLds16);
    rows16_kernel<QT, FUSED, S><<<compute_units(), (Map16<QT, S>::kThreads), kLds16, stream>>>(a);
    return check_launch("moe_rows16");
}

// Pairs of a full tile: as many Q8_K rows as the LDS holds, at most sixteen.
template <unsigned QT, unsigned S> unsigned tile_tokens16(unsigned blocks)
{
    using M = Map16<QT, S>;
    unsigned tokens = kSlots16;
    while (tokens && M::kAreas + M::area_bytes(blocks, tokens) > kLds16) tokens -= 4u;
    return tokens;
}

// Image rows that come two superblocks a run.
bool two_at_a_time(uint64_t blocks) { return blocks % 2u == 0u && blocks >= 4u && blocks <= 16u; }

}  // namespace

unsigned rows16_tokens(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, uint64_t width,
                       uint64_t out_rows)
{
    const uint64_t blocks = width / 256u, superblock = qtype == QT_IQ2_XXS ? (image ? 72u : 66u) : qtype == QT_Q4_K ? 144u : 84u;
    // two runs are asked for ahead of their use, the second of them at a unit's end of the unit behind it
    if (width % 256u || blocks < (qtype == QT_Q2_K && !(blocks & 1u) ? 4u : 2u) || blocks > kMaxBlocks16 || (qtype == QT_Q2_K && fused)) return 0u;
    // a lane addresses its rows with 32-bit offsets inside an expert and stores four rows at a time
    if (out_rows < (fused ? 16u : 32u) || out_rows % 4u || problem.row_bytes != blocks * superblock || (problem.row_bytes & 3u) ||
        (fused && problem.up_row_bytes != problem.row_bytes) || out_rows * problem.row_bytes > 0xffffffffull)
        return 0u;
    if ((((uintptr_t)problem.gate | (uintptr_t)problem.up | (uintptr_t)problem.activations | problem.expert_bytes |
          problem.up_expert_bytes | problem.act_stride) & 3u) || ((uintptr_t)problem.out & 15u))
        return 0u;
    if (problem.experts > 256u && problem.expert_ids) return 0u;
    return qtype == QT_IQ2_XXS && image && two_at_a_time(blocks) ? tile_tokens16<kIq2Image, 2u>((unsigned)blocks)
         : qtype == QT_IQ2_XXS ? tile_tokens16<kIq2Image, 1u>((unsigned)blocks)
         : qtype == QT_Q4_K    ? tile_tokens16<QT_Q4_K, 1u>((unsigned)blocks)
         : qtype == QT_Q2_K    ? tile_tokens16<QT_Q2_K, 2u>((unsigned)blocks) : 0u;
}

bool rows16_one_round(const GroupedProblem &problem, unsigned qtype, bool fused, unsigned tokens, uint64_t out_rows)
{
    const uint64_t units = (out_rows + (fused ? 15u : 31u)) / (fused ? 16u : 32u);
    const unsigned waves = qtype == QT_IQ2_XXS ? Map16<kIq2Image, 1u>::kWaves : Map16<QT_Q4_K, 1u>::kWaves;
    return (problem.pairs + (uint64_t)tokens - 1u) / tokens * units <= (uint64_t)waves * compute_units();
}

int launch_rows16_grouped(const GroupedProblem &problem, unsigned qtype, bool image, bool fused, unsigned width,
                          unsigned out_rows, unsigned behind, bool round, double limit, int *status, hipStream_t stream)
{
    const Rows16Args a{problem, width / 256u, out_rows, rows16_tokens(problem, qtype, image, fused, width, out_rows), round,
                       behind, limit, status};
    if (!a.tokens) return ST_UNSUPPORTED;
    // (a run of two Q2_K superblocks fills a load; a row of an odd number of them comes one at a time)
    if (qtype == QT_Q2_K)
        return a.blocks & 1u ? launch_rows16<QT_Q2_K, false, 1u>(a, stream) : launch_rows16<QT_Q2_K, false, 2u>(a, stream);
    if (qtype == QT_Q4_K)
        return fused ? launch_rows16<QT_Q4_K, true, 1u>(a, stream) : launch_rows16<QT_Q4_K, false, 1u>(a, stream);
    if (image && two_at_a_time(a.blocks))
        return fused ? launch_rows16<kIq2Image, true, 2u>(a, stream) : launch_rows16<kIq2Image, false, 2u>(a, stream);
    if (image)
        return fused ? launch_rows16<kIq2Image, true, 1u>(a, stream) : launch_rows16<kIq2Image, false, 1u>(a, stream);
    return fused ? launch_rows16<QT_IQ2_XXS, true, 1u>(a, stream) : launch_rows16<QT_IQ2_XXS, false, 1u>(a, stream);
}

}  // namespace yvex
