// Kernel parameter blocks and LDS layouts of the library, shared by the gfx950 kernels
// (gllmq_kernels.hip) and the host launcher (gllmq_host.cpp): one definition, so the bytes the
// host hands to hipModuleLaunchKernel are the struct the kernel reads.
#ifndef GQ_PARAMS_H
#define GQ_PARAMS_H

#include <stdint.h>

#if defined(__HIP__)
#define GQ_HD __host__ __device__
#else
#define GQ_HD
#endif

namespace gq {

struct GemvParams {
    const uint8_t *w;
    const float *x;
    float *y;
    uint32_t n;          // weight rows = outputs
    uint32_t k;          // elements per row (activations beyond k read as zero)
    uint32_t groups;     // 256-element groups per row = ceil(k / 256)
    uint32_t row_bytes;  // bytes between rows
    uint32_t ks;         // waves that share one row (K split)
    uint32_t rps;        // rows side by side in one wave (1 when a row fills the wave)
    uint32_t rows_per_wg;
    uint32_t ldx;        // elements between activation rows
    uint32_t ldy;        // elements between output rows
    uint32_t x_vec;      // activation rows are 16-byte aligned: vector loads allowed
    uint32_t accumulate; // add to y instead of overwriting it (K handled in several launches)
    uint32_t prep_words; // integer-dot kernels: 32-bit words of LDS holding the prepared activations
    uint32_t act_bf16;   // integer-dot kernels: round activations to bf16 before use
    uint32_t elem;       // integer-dot kernels: element type of x and y (ELEM_F32 / ELEM_F16 / ELEM_BF16)
    uint32_t glu, glu_off; // integer-dot kernels: x[i] = act(x[i]) * x[i + glu_off] (0 off, 1 SiLU, 2 SiLU behind a ReLU)
    // kernels that end in the greedy token choice: one candidate per workgroup (argmax_key); the
    // workgroup that finishes last (ticket counts them and is left at 0) picks among them
    uint64_t *keys;
    uint32_t *ticket;
    uint32_t *token; // the choice (ARGMAX_NONE: no candidate)
    float *value;    // null, or the chosen logit (NaN: none)
};

struct Mm8Params {
    const uint8_t *w;
    const float *x;
    float *y;
    uint32_t n;         // weight rows
    uint32_t k;         // elements per row
    uint32_t groups;    // 256-element blocks per row
    uint32_t row_bytes; // bytes between rows
    uint32_t m;         // activation rows (<= 2 * PAIRS of the kernel)
    uint32_t ldx, ldy;
    uint32_t tiles;     // ceil(n / 32)
    uint32_t grid;      // workgroups launched (kept beside the other fields so one kernarg line holds all)
    uint32_t act_bf16;  // round activations to bf16 before use
    const uint32_t *xrows; // row of x (in units of ldx) behind each of the m activation rows: 0..m-1, or gathered rows
    // gated form only (gq_mm8_glu_*): the up rows, and whether the gate passes a ReLU ahead of the SiLU
    const uint8_t *w2;
    uint32_t glu_relu;
    // K split (plain kernels only; 0 or 1 = off): `ksplit` consecutive workgroups share a tile list,
    // workgroup s of them multiplies blocks [s * kslice_groups, (s + 1) * kslice_groups) of every
    // row and writes its sums to part[s][m][n]; the one that finishes last adds the slices up in
    // order (arrive[tile list] counts the finished ones and is left at 0).
    uint32_t ksplit, kslice_groups;
    uint32_t elem;      // element type of x and y (ELEM_F32 / ELEM_F16 / ELEM_BF16); the slice sums stay f32
    float *part;
    uint32_t *arrive;
    // streamed kernels (mm8s.hip.inc) only, all worked out by the host so that a loader wave's
    // way to its first load is short: weight rows per workgroup, rows per tile (<= 32: a
    // workgroup's rows are cut into tiles of equal height), item slots of the LDS ring (a
    // multiple of the loader waves unless the ring holds every item), tiles of a full
    // workgroup and of the last one, rows of the last one, the LDS offsets of the counters
    // and of the ring, and the items a loader keeps unconfirmed (1 .. MM8S_MAX_DEPTH)
    uint32_t rows_per_wg, tile_rows, ring_slots, wg_tiles, last_wg_tiles, last_wg_rows, lds_ctrl, lds_ring, depth;
    // activations that are the gated product of two f32 vectors (the input of a feed-forward
    // block's down projection): x[i] = act(x[i]) * x[i + glu_off]; glu = 0 off, 1 SiLU, 2 SiLU behind a ReLU
    uint32_t glu, glu_off;
    // streamed kernels: null, or the word that says which launch of the context has started (the
    // weight prefetch of the launch behind this one waits for it): workgroup 0 raises it to
    // `progress_seq` on its way in
    unsigned long long *progress;
    unsigned long long progress_seq;
};

// The launch that ends in the greedy token (gq_mm8s_*_token): the workgroups' candidates (argmax_key), how many workgroups have left
// theirs (zero between launches), the token, and (or null) its value.
struct Mm8sTokenParams {
    Mm8Params p;
    uint64_t *keys;
    uint32_t *ticket;
    uint32_t *token;
    float *value;
};

// Several weight matrices over the same activations in one streamed launch: the row ranges of a matrix are
// those of workgroups first_wg .. up to the next matrix's; p.w, p.y, p.n and p.ldy are each workgroup's own.
constexpr int MM8S_MAX_SEGS = 3;
struct Mm8sSeg {
    const uint8_t *w;
    float *y;
    uint32_t n, first_wg;
};
struct Mm8sGroupParams {
    Mm8Params p;
    Mm8sSeg seg[MM8S_MAX_SEGS];
    uint32_t segs;
};

// The weight prefetch that runs beside a sequence of dependent launches (touch.hip.inc): for each
// entry, in order, wait until launch number `seq - 1` of the context has started (`progress`, see
// Mm8Params), then pull the entry's bytes into the memory-side cache by reading one word of every
// 128-byte line.  An entry whose own launch has already started, or whose wait runs out after
// `timeout_ticks` of the 100 MHz clock, is skipped: the prefetch never holds anything up.
constexpr uint32_t TOUCH_MAX_ENTRIES = 32;
struct TouchEntry {
    const uint8_t *w;
    unsigned long long bytes;
    unsigned long long seq;
};
struct TouchParams {
    const unsigned long long *progress;
    uint32_t *sink;          // null (a place the words read would go to if they were ever needed)
    uint32_t count, timeout_ticks;
    uint32_t flags, pad;     // bit 0: wait as usual but read nothing (for measurements)
    TouchEntry e[TOUCH_MAX_ENTRIES];
};

constexpr uint32_t MM8_SPLIT_MAX_LISTS = 256;        // tile lists (workgroups per slice) of a K-split launch
constexpr uint32_t MM8_SPLIT_PART_FLOATS = 1u << 20; // slices * activation rows * n of a K-split launch (4 MiB)

constexpr int MM8_WAVES = 8;
constexpr int MM8_THREADS = 64 * MM8_WAVES;
constexpr int MM8_LOADS = 5;            // 16-byte loads per lane for one 32-row block tile (4.5 used)
constexpr int MM8_STAGE_BYTES = 5120;   // 32 rows x 144 bytes, rounded up to whole wave loads

// What differs between the two formats of mm8.hip.inc.  Q5_K is Q4_K with a fifth bit per quant
// (32 bytes of qh between the header and the nibbles): same sub-blocks, scales and mins.
template <int FMT> struct Mm8Format;
template <> struct Mm8Format<0> { // Q4_K
    static constexpr uint32_t BLOCK = 144, CHUNKS = 9, QS = 16, STAGE = MM8_STAGE_BYTES;
    static constexpr int LOADS = MM8_LOADS;
};
template <> struct Mm8Format<1> { // Q5_K
    static constexpr uint32_t BLOCK = 176, CHUNKS = 11, QS = 48, STAGE = 6144; // 32 rows x 176 bytes, rounded up
    static constexpr int LOADS = 6;                                           // 5.5 used
};

// What the streamed kernels (mm8s.hip.inc) need to know of a format: bytes of a block in memory,
// 16-byte pieces a block's row is fetched as (Q6_K blocks are 210 bytes and only 2-byte aligned:
// 13 pieces at 16 p and a fourteenth at 194, so no load runs past a block), wave-loads of a
// 32-row item, sub-block sums the preparation keeps per block.  In LDS a row of an item is its
// pieces side by side, PIECES * 16 bytes.
template <int FMT> struct Mm8sFormat;
template <> struct Mm8sFormat<0> { static constexpr uint32_t BLOCK = 144, PIECES = 9, SUBS = 8, ZEROS = 0; };   // Q4_K
template <> struct Mm8sFormat<1> { static constexpr uint32_t BLOCK = 176, PIECES = 11, SUBS = 8, ZEROS = 0; };  // Q5_K
template <> struct Mm8sFormat<2> { static constexpr uint32_t BLOCK = 210, PIECES = 14, SUBS = 0, ZEROS = 256; }; // Q6_K (ZEROS: bytes of zeros ahead of the ring, a block of an operand's unused elements)
template <> struct Mm8sFormat<3> { static constexpr uint32_t BLOCK = 272, PIECES = 17, SUBS = 0, ZEROS = 0; };   // Q8_0: a group of 8 blocks of 34 bytes (K a multiple of 256)
GQ_HD constexpr uint32_t mm8s_piece_offset(int fmt, uint32_t piece) { return (fmt == 2 && piece == 13u) ? 194u : 16u * piece; }

// LDS carve-up (bytes) of the int8 matrix-core kernels.
struct Mm8Lds {
    uint32_t plane_stride; // bytes between digit planes
    uint32_t planes;       // offset of [3 * m][plane_stride]
    uint32_t sums;         // offset of float [m][groups][8]: sum of X per sub-block
    uint32_t scales;       // offset of float [m][groups]: 2^e per block (NaN if poisoned)
    uint32_t red;          // offset of float [2][MM8_WAVES][PAIRS][64]
    uint32_t stage;        // offset of [MM8_WAVES][MM8_STAGE_BYTES]: one weight block tile per wave
    uint32_t total;
};

// `subs`: sub-block sums kept per 256-element block (8 of 32 elements for Q4_K and Q5_K, none for
// Q6_K and Q8_0); `stage_bytes`: one wave's weight stage.
GQ_HD inline Mm8Lds mm8_lds_layout(uint32_t groups, uint32_t m, uint32_t pairs, uint32_t subs = 8u,
                                   uint32_t stage_bytes = MM8_STAGE_BYTES)
{
    Mm8Lds L;
    L.plane_stride = groups * 256u + 16u; // +16 staggers the planes over the LDS banks
    L.planes = 0;
    L.sums = L.planes + 3u * m * L.plane_stride;
    L.scales = L.sums + m * groups * subs * 4u;
    L.red = (L.scales + m * groups * 4u + 15u) & ~15u;
    L.stage = L.red + 2u * MM8_WAVES * pairs * 64u * 4u;
    L.total = L.stage + MM8_WAVES * stage_bytes;
    return L;
}

// Streamed form of the int8 matrix-core kernels (mm8s.hip.inc): loader waves and arithmetic waves.
constexpr int MM8S_CWAVES = 8;      // arithmetic waves
#ifndef GQ_MM8S_LOADERS
#define GQ_MM8S_LOADERS 4
#endif
constexpr int MM8S_LOADERS = GQ_MM8S_LOADERS; // loader waves
constexpr int MM8S_RED_BUFS = 4;    // tiles whose partial sums can be waiting in LDS
// Items a loader keeps unconfirmed (its depth D, chosen per launch: what is in flight per CU,
// not the item count, is what keeps the memory system busy, and items of low tiles are small).
// A loader's outstanding wave-loads are counted by a 6-bit counter: D times the wave-loads of
// an item (at most 7) stays below 64.
constexpr uint32_t MM8S_MAX_DEPTH = 6;
constexpr uint32_t MM8S_DEPTH_BYTES = 8192; // a loader keeps about this much unconfirmed
// A consumer sees item i once its loader has requested D more items of its own, that is item
// i + D * MM8S_LOADERS, and that request waits for the slot of item i + D * MM8S_LOADERS - slots
// to be free: with slots > D * MM8S_LOADERS every wait is for an item with a smaller number and
// the chain ends.  Half as many again keep the stream going while items are being multiplied.
inline GQ_HD uint32_t mm8s_min_slots(uint32_t depth) { return depth * MM8S_LOADERS + MM8S_LOADERS * ((depth + 1u) / 2u); }

struct Mm8sCtrl {                    // counters in LDS, all start at zero
    uint32_t landed[8];              // per loader: items whose bytes are in LDS
    uint32_t done[MM8S_CWAVES];      // per arithmetic wave: items consumed
    uint32_t arrived[MM8S_RED_BUFS]; // per partial-sum buffer: waves that left their sums
    uint32_t reduced;                // tiles summed and stored
    uint32_t finished;               // K split: arithmetic waves whose slice sums have reached coherent memory; token choice: that are through
    union {
        uint32_t pad[2];
        uint64_t best;               // token choice: the workgroup's largest candidate
    };
};

// LDS carve-up of the streamed kernels: the preparation's planes, sums and scales as in
// mm8_lds_layout, then the counters, the partial sums and the ring of item slots.
struct Mm8sLds {
    Mm8Lds prep;
    uint32_t ctrl, red, ring, total;
};

// The folded form of the streamed kernels (one activation row, tiles of at most 16 weight rows):
// an item is a pair of blocks of the tile, blocks 16 q + i and 16 q + 8 + i (i < 8) being pair
// 8 q + i, so that the arithmetic wave of a pair (pair mod 8) is the wave of both of its blocks
// (block mod 8), as in the form that goes block by block: the same wave prepares the activations
// of a block either way.  A row whose last group of 16 blocks has 8 or fewer ends in pairs without
// a second block.
GQ_HD inline uint32_t mm8s_fold_pairs(uint32_t groups) { return 8u * (groups / 16u) + (groups % 16u < 8u ? groups % 16u : 8u); }
GQ_HD inline uint32_t mm8s_fold_first(uint32_t pair) { return 16u * (pair >> 3) + (pair & 7u); }

// `glu`: the gated kernels keep the sums of a gate tile (pairs x 64 floats) behind the partial sums
// until the up tile of the same rows is summed.
GQ_HD inline Mm8sLds mm8s_lds_layout(uint32_t groups, uint32_t m, uint32_t pairs, uint32_t item_bytes, uint32_t slots,
                                     uint32_t subs, bool glu, uint32_t zeros)
{
    Mm8sLds L;
    L.prep = mm8_lds_layout(groups, m, pairs, subs, 0u);
    L.ctrl = (L.prep.red + 15u) & ~15u; // the area of mm8.hip.inc's partial sums and stages is not used here
    L.red = L.ctrl + static_cast<uint32_t>(sizeof(Mm8sCtrl));
    L.ring = (L.red + MM8S_RED_BUFS * MM8S_CWAVES * pairs * 64u * 4u + (glu ? pairs * 64u * 4u : 0u) + zeros + 1023u) & ~1023u;
    L.total = L.ring + slots * item_bytes;
    return L;
}

// Ring and loader depth of a streamed launch for `m` activation rows (1..4) whose items, `items`
// per workgroup of `item_bytes` each, share `lds_bytes` of LDS with the preparation of `groups`
// blocks: one or two rows keep one item per loader unconfirmed, three and four about
// MM8S_DEPTH_BYTES.  False when the ring would be too short for the loaders to run ahead.
// `want_depth` != 0: that many items per loader instead (a long stream gains from more of them).
GQ_HD inline bool mm8s_ring(uint32_t groups, uint32_t m, uint32_t item_bytes, uint32_t items, uint32_t subs, bool glu, uint32_t zeros,
                            uint32_t lds_bytes, uint32_t want_depth, Mm8sLds &L, uint32_t &slots, uint32_t &depth)
{
    const uint32_t pairs = m <= 2u ? 1u : 2u;
    L = mm8s_lds_layout(groups, m, pairs, item_bytes, 0u, subs, glu, zeros);
    if (L.total + item_bytes > lds_bytes) return false;
    slots = (lds_bytes - L.total) / item_bytes;
    if (slots >= items) slots = items;
    else slots -= slots % MM8S_LOADERS; // a reused ring is a whole number of rounds of the loaders
    depth = 1u;
    if (pairs > 1u) {
        depth = (MM8S_DEPTH_BYTES + item_bytes / 2u) / item_bytes;
        depth = depth < 2u ? 2u : (depth > MM8S_MAX_DEPTH ? MM8S_MAX_DEPTH : depth);
    }
    if (want_depth) depth = want_depth > MM8S_MAX_DEPTH ? MM8S_MAX_DEPTH : want_depth;
    while (depth > (pairs > 1u ? 2u : 1u) && slots < items && slots < mm8s_min_slots(depth)) --depth;
    return slots >= items || slots >= mm8s_min_slots(depth);
}

// Q6_K flavour (mm8_q6k.hip.inc)
constexpr int MM8Q6_LOADS = 7;             // 16-byte loads per lane for one 32-row block tile (32 x 14 pieces)
constexpr int MM8Q6_ROW_STRIDE = 240;      // bytes between rows in the stage: 224 used, padded against bank conflicts
constexpr int MM8Q6_STAGE_BYTES = 32 * MM8Q6_ROW_STRIDE;

// Q8_0 flavour (mm8_q8_0.hip.inc): 8 blocks of 34 bytes per 256 elements
constexpr int MM8Q8_LOADS = 9;             // 16-byte loads per lane for one 32-row group tile (32 x 17 pieces, 8.5 used)
constexpr int MM8Q8_ROW_STRIDE = 272;      // bytes between rows in the stage: the 8 blocks as they lie in memory
constexpr int MM8Q8_STAGE_BYTES = 32 * MM8Q8_ROW_STRIDE;

struct MmfParams {
    const uint8_t *w;
    const float *x;
    float *y;
    uint8_t *ximg;       // [groups] images of the prepared activations, MmfLds<MT>::image bytes apart
    float *partial;      // [ksplit][m][n] when ksplit > 1
    uint32_t n, k, groups, row_bytes, m, ldx, ldy;
    uint32_t row_tiles;        // ceil(n / 256)
    uint32_t ksplit;           // workgroups per row tile
    uint32_t blocks_per_split; // 256-element blocks of K per workgroup
    uint32_t act_bf16;
    uint32_t elem;             // element type of y (ELEM_F32 / ELEM_F16 / ELEM_BF16); partial sums stay f32
};

constexpr int MMF_WAVES = 8;
constexpr int MMF_ST = 1;                                  // 32-row sub-tiles per wave
constexpr int MMF_THREADS = 64 * MMF_WAVES;
constexpr int MMF_TILE_ROWS = 32 * MMF_ST * MMF_WAVES;     // weight rows per workgroup
constexpr int MMF_PREP_THREADS = 1024;                     // threads that prepare one block of K
constexpr int MMF_XROW_BYTES = 256 * 2 + 16;   // one activation row of a block in LDS (f16), padded
constexpr int MMF_STAGE_BYTES = 5120;          // one 32-row sub-tile of one block, as fetched

// FMT: 0 = Q4_K (144-byte blocks, 5 KiB per wave stage), 1 = Q5_K (176 bytes, 6 KiB), 2 = Q6_K, 3 = Q8_0.
template <int FMT> struct MmfFormat;
template <> struct MmfFormat<0> { static constexpr uint32_t BLOCK = 144, CHUNKS = 9, QS = 16, STAGE = 5120; static constexpr int LOADS = 5; };
template <> struct MmfFormat<1> { static constexpr uint32_t BLOCK = 176, CHUNKS = 11, QS = 48, STAGE = 6144; static constexpr int LOADS = 6; };
template <> struct MmfFormat<2> { static constexpr uint32_t STAGE = MM8Q6_STAGE_BYTES; }; // Q6_K (mmf_q6k.hip.inc): 7.5 KiB
template <> struct MmfFormat<3> { static constexpr uint32_t STAGE = MM8Q8_STAGE_BYTES; }; // Q8_0 (mmf_q8_0.hip.inc): 8.5 KiB

// LDS carve-up for MT 32-row activation tiles.  The first `image` bytes are the block image
// that gq_mmf_prep_* writes and the GEMM copies verbatim: hi plane, sub-block sums, inverse
// scales, lo plane, padded to whole rounds of one 16-byte chunk per thread.
template <int MT, int FMT = 0>
struct MmfLds {
    static constexpr uint32_t rows = 32u * MT;
    static constexpr uint32_t hi = 0;
    static constexpr uint32_t sums = hi + rows * MMF_XROW_BYTES; // [rows][16] f16: 8 hi, 8 lo
    static constexpr uint32_t inv = sums + rows * 32u;           // [rows] f32
    static constexpr uint32_t lo = inv + rows * 4u;
    static constexpr uint32_t round = MMF_THREADS * 16u;
    static constexpr uint32_t loads_hi = (lo + round - 1u) / round;                           // copy rounds without the lo plane
    static constexpr uint32_t loads_all = (lo + rows * MMF_XROW_BYTES + round - 1u) / round;  // with it
    static constexpr uint32_t image = loads_all * round;
    static constexpr uint32_t stages = MMF_WAVES * MMF_ST * MmfFormat<FMT>::STAGE; // one weight stage per wave
    // One image and one set of stages, or (when two of each fit the 160 KiB of a CU) two that
    // take turns: image p at p * image, stage set p behind the images.
    static constexpr bool twice = 2u * (image + stages) <= 160u * 1024u;
    static constexpr uint32_t stage = (twice ? 2u : 1u) * image; // [twice ? 2 : 1][waves][MMF_ST][MMF_STAGE_BYTES]
    static constexpr uint32_t total = stage + (twice ? 2u : 1u) * stages;
};

// A chain of streamed one- or two-row matmuls in one launch (mm8c.hip.inc).
constexpr int MM8C_CWAVES = 8;             // arithmetic waves (MM8_WAVES: the preparation is the same code)
constexpr int MM8C_LOADERS = 4;            // loader waves
constexpr int MM8C_RED_BUFS = 4;           // tiles whose partial sums can be waiting in LDS
constexpr uint32_t MM8C_MAX_SLOTS = 32;    // ring slots (a counter each)
constexpr uint32_t MM8C_MAX_ENTRIES = 32;  // matmuls per launch
struct Mm8ChainEntry {
    const uint8_t *w;
    const float *x;
    float *y;
    uint32_t n, ldy;
    // the entry's geometry, worked out by the host as for the streamed kernels: weight rows per
    // workgroup, workgroups that take part, tile height, tiles of a full and of the last
    // workgroup, rows of the last workgroup; flags: bit 0 = its x is (part of) the y of the entry
    // before it, read from the mailbox, bit 1 = the entry behind it reads this one's y (so this one
    // posts its outputs there), bit 2 = its items are pairs of blocks (one activation row, tiles
    // of at most 16 rows)
    uint32_t rows_per_wg, grid, tile_rows, wg_tiles, last_wg_tiles, last_wg_rows, flags;
    // mailbox places (in pairs, see Mm8ChainParams::box): where this entry posts output row 0 (rows
    // `n` apart), and where its own activation row 0 was posted by the entry before (rows `x_ld` apart)
    uint32_t box_at, x_at, x_ld, pad;
};
struct Mm8ChainParams {
    uint32_t count, launched;     // entries, workgroups of the launch (the largest `grid`)
    uint32_t k, groups, row_bytes, m, ldx, act_bf16;
    uint32_t ring_slots, slot_bytes, depth, lds_ctrl, lds_ring, spin_limit;
    // Entries that read the output of the one before them inside the launch: every output of such
    // a producer is also posted as one 64-bit word (epoch << 32 | value bits) with a device-scope
    // store, entry e under epoch `epoch0 + e`; a reader loads the words it needs until all carry the
    // producer's epoch.  A word says by itself that its value is there, so nobody waits for stores
    // to be acknowledged, nothing is counted, and nothing is set back: epochs are the context's own
    // count of chained entries, no earlier launch used them, and every entry of a launch has places
    // of its own.  Null when no entry waits.
    unsigned long long *box;
    uint32_t epoch0, pad0;
    uint32_t *error;              // host-visible word, set to 1 when a reader's wait ran out
    unsigned long long *progress; // as in Mm8Params
    unsigned long long progress_seq;
    Mm8ChainEntry e[MM8C_MAX_ENTRIES];
};

// Streamed form of the Q4_K / Q5_K GEMM (mmfs.hip.inc): takes Mm8Params like the streamed int8
// kernels, whose loader it shares (x holds the activation images, groups all blocks of K,
// kslice_groups the blocks of a workgroup's slice of K, grid the row ranges).
// Its activation image of one block of K and 32 rows, in the order the lanes hold it: for each of
// the 16 K steps of the block the 64 lanes' 16-byte operands (lane = row + 32 * half of the step)
// one after the other, hi plane then lo plane; the sub-block sums as the operand of the min term
// (hi sums for the lanes of half 0, lo sums for half 1); the rows' inverse scales.  Every register
// of a wave is then one contiguous 1 KiB load.
struct MmfLanes {
    static constexpr uint32_t hi = 0, lo = 16u * 1024u, sums = 32u * 1024u, inv = 33u * 1024u, image = 34u * 1024u;
};
constexpr int MMFS_CWAVES = 4;  // arithmetic waves = blocks of K per workgroup
constexpr int MMFS_LOADERS = 4; // loader waves (MM8S_LOADERS: the loader is the same code)
constexpr int MMFS_RED_BUFS = 3; // tiles whose block sums can be waiting in LDS
static_assert(MMFS_LOADERS == MM8S_LOADERS, "mm8s_min_slots() is worked out for that many loaders");

// The streamed GEMM whose waves prepare their own activations (mmfr.hip.inc).
constexpr int MMFR_CWAVES = 8;   // arithmetic waves
constexpr int MMFR_LOADERS = 4;  // loader waves (MM8S_LOADERS: the loader is the same code)
constexpr int MMFR_RED_BUFS = 3; // tiles whose block sums can be waiting in LDS
constexpr uint32_t MMFR_RED_WAVE = 2u * 64u * 16u; // bytes of a tile's sums in LDS per wave: [column tile][lane] float4

// The GEMM for prompts and larger batches (mmfw.hip.inc).  A workgroup is eight waves of 32 weight
// rows each and MT tiles of 32 activation rows; the activations come as images in the order the
// lanes hold them (MmfwImage), the weight matrices of one launch share the activations.
constexpr int MMFW_WAVES = 8;
constexpr int MMFW_TILE_ROWS = 32 * MMFW_WAVES; // weight rows per workgroup
// What a launch multiplies: activation tiles, experts' jobs, or experts' jobs of one and two tiles in workgroups of four waves, two a CU
// (moe_wide_few).
constexpr int MMFW_DENSE = 0, MMFW_EXPERTS = 1, MMFW_EXPERTS_FEW = 2;
constexpr int mmfw_waves(int grouped) { return grouped == MMFW_EXPERTS_FEW ? MMFW_WAVES / 2 : MMFW_WAVES; }
constexpr int MMFW_MAX_SEGS = 3;                // weight matrices of one launch
constexpr int MMFW_MAX_MT = 4;
constexpr bool mmfw_runs(int mt) { return mt <= 3; } // Q6_K, Q8_0: registers for sums of runs (MmfwParams::run_mask)
constexpr uint32_t MMFW_PREP_WAVES = 16;        // of a workgroup that prepares an image
constexpr uint32_t MMFW_PREP16_WAVES = 8;       // ... from 16-bit elements, four rows a wave

// Four tiles of Q4_K and Q5_K: no registers for sums of the lo plane's products, which therefore come ahead of the hi
// plane's (a block's weights are unpacked twice).  In turn with them, where each costs the sum a rounding at its full size,
// the error was 2.43e-7 (512 f32 rows of 14336 x 4096 Q4_K; so 1.92e-7, the 64-row form 2.17e-7) and the call 3 % shorter
// (123 us, so 126; three tiles, which have the registers, 177, two 143).
constexpr bool mmfw_lo_first(int fmt, int planes, int mt) { return fmt <= 1 && planes == 2 && mt == 4; }

// Q8_0 against two planes: quants two units of 32 elements ahead, a unit's last sums scaled behind the next one's products.  A unit
// is a chain of LDS read, unpacking, products and scaling that two waves a SIMD do not hide: 512 rows of 14336 x 4096 in two
// tiles 172 us, so 165, in three 212, 206; 64 rows of 28672 x 4096 59.2, 57.7.  One plane 1 to 3 % longer (64 rows 48.4, 49.2), four
// tiles have no registers for it.
constexpr bool mmfw_q8_ahead(int planes, int mt) { return planes == 2 && mt <= 3; }

// Image of 32 activation rows x 256 elements of K: [K step 0..15][plane][lane] 16 bytes (lo first: [lo, hi][K step]), then
// [lane] 16 bytes of sub-block sums (lanes 0..31 hi, 32..63 lo); images lie [row tile][block].
// The inverse scales are an array of their own: [block][padded rows] f32.
template <int PL> struct MmfwImage {
    static constexpr uint32_t sums = 16u * PL * 1024u, bytes = sums + 1024u;
};

// FMT: 0 = Q4_K, 1 = Q5_K, 2 = Q6_K, 3 = Q8_0.  A wave's weights of a block come in parts, each
// requested again (for the next block) as soon as it has been read: the header (scales) and `PARTS`
// equal shares of the quants, `PART` wave-loads each.
template <int FMT> struct MmfwFormat;
template <> struct MmfwFormat<0> { // 32 rows x 32 bytes per part, headers 16 bytes a row
    static constexpr uint32_t BLOCK = 144, STAGE = 5u * 1024u;
    static constexpr int PARTS = 4, PART = 1, HEAD = 1;
    static constexpr bool SUMS = true;
};
template <> struct MmfwFormat<1> { // the fifth bits come with the header
    static constexpr uint32_t BLOCK = 176, STAGE = 6u * 1024u;
    static constexpr int PARTS = 4, PART = 1, HEAD = 2;
    static constexpr bool SUMS = true;
};
template <> struct MmfwFormat<2> { // half blocks: two 32-byte pieces of low nibbles a row, one of high bits
    static constexpr uint32_t BLOCK = 210, STAGE = 7u * 1024u;
    static constexpr int PARTS = 2, PART = 3, HEAD = 1;
    static constexpr bool SUMS = false;
};
template <> struct MmfwFormat<3> { // half groups: 136 bytes a row
    static constexpr uint32_t BLOCK = 272, STAGE = 10u * 1024u;
    static constexpr int PARTS = 2, PART = 5, HEAD = 0;
    static constexpr bool SUMS = false;
};

template <int FMT, int PL, int MT, bool LO_FIRST = false, bool OWN = false, int NWAVES = MMFW_WAVES>
struct MmfwShape {
    using F = MmfwFormat<FMT>;
    static constexpr int WAVES = NWAVES;
    static_assert(WAVES == MMFW_WAVES || MT <= 2, "workgroups of four waves: one and two tiles");
    static_assert(!LO_FIRST || mmfw_lo_first(FMT, PL, MT), "");
    static_assert(!OWN || MT == 1, "");
    // Activations move in chunks of UC units (32 elements of K) through a ring of R chunk slots in LDS.
    static constexpr int UC = (MT == 4 ? (PL == 2 ? 1 : 2) : MT == 3 ? (PL == 2 ? 2 : 4) : MT == 2 ? (PL == 2 ? 2 : 4) : (PL == 2 ? 4 : 8)) * WAVES / MMFW_WAVES;
    static constexpr int R = MT == 3 ? 3 : 4;
    static constexpr int C = 8 / UC;                   // chunks per block
    static constexpr int PIECES = MT * PL * 2 * UC;    // KiB per chunk
    static constexpr int NA = OWN ? 0 : PIECES / WAVES; // wave-loads per wave and chunk
    static_assert(PIECES % WAVES == 0, "every wave requests the same number of pieces");
    static constexpr uint32_t CHUNK = PIECES * 1024u;
    static constexpr uint32_t TILE_CHUNK = 2u * UC * PL * 1024u; // a row tile's share: contiguous in its image
    static constexpr uint32_t extra = 0;               // [4][sums of MT tiles, inverse scales]
    static constexpr uint32_t EXTRA = ((F::SUMS ? MT : 0) + 1) * 1024u;
    static constexpr uint32_t SLOTS = OWN ? 8u : 4u;
    static constexpr uint32_t stage = SLOTS * EXTRA;
    static constexpr uint32_t ring = stage + WAVES * F::STAGE;
    // OWN: the images of a slice's blocks are made here, all of them ahead of the first product, and take the ring's place
    // (eight places of sums and scales: more than blocks, the next one is read past the last)
    static constexpr int OWN_FIT = (160u * 1024u - ring) / (C * CHUNK), OWN_BLOCKS = OWN_FIT < 4 ? OWN_FIT : 4;
    static constexpr uint32_t RING = OWN ? OWN_BLOCKS * C * CHUNK : R * CHUNK;
    static constexpr uint32_t total = ring + RING;
    static_assert(total <= 160u * 1024u, "LDS");

    // ---- A block is NS stages of SG operand slots (a K step of one plane) for all row tiles; Q6_K, Q8_0:
    // a stage is a unit.  What stage s + 1 multiplies is read from LDS during stage s.
    static constexpr int SG = MT >= 3 ? 1 : MT == 2 ? 2 : 4;
    static constexpr int NS = FMT >= 2 ? 8 : 16 * PL / SG;
    static constexpr int SPC = NS / C;                 // stages per chunk
    static constexpr int PASS = LO_FIRST ? NS / 2 : NS; // stages in which the block's weights are read once
    static constexpr int QL = PASS / F::PARTS;         // stages per weight part
    // Q8_0 reads the quants of stage s + 1 (s + 2) in stage s, so a part is free a stage (two) before the next one starts
    static constexpr int FREE = FMT == 3 ? QL - (mmfw_q8_ahead(PL, MT) ? 2 : 1) : 0; // a part is requested again that far behind its first stage
    static constexpr int requested(int p) { return NS - PASS + p * QL + FREE; } // (lo first: behind its second read)
    static constexpr int part_of(int s) { return s >= requested(0) && (s - requested(0)) % QL == 0 ? (s - requested(0)) / QL : -1; }

    // ---- the wave's sequence of loads, one block being a period: stage s requests its weights (and
    // stage 0 the extra of the block after next, first); then, in the last stage of a chunk, the
    // next chunk is acquired: its arrival is waited for and NA pieces of the chunk R - 1 further on
    // are requested.
    static constexpr int stage_loads(int s) { return (s == 0 ? (OWN ? 0 : 1) + F::HEAD : 0) + (part_of(s) >= 0 ? F::PART : 0); }
    static constexpr int after_weights(int s) // position behind stage s's weight requests
    {
        int p = 0;
        for (int i = 0; i <= s; ++i) p += stage_loads(i) + (i < s && (i + 1) % SPC == 0 ? NA : 0);
        return p;
    }
    static constexpr int period = after_weights(NS - 1) + NA;
    static constexpr int acquired(int c) // position of the acquisition of chunk c, ahead of its requests
    {
        int blk = 0;
        while (c < 0) { c += C; --blk; }
        return blk * period + (c ? after_weights(c * SPC - 1) : -NA);
    }
    static constexpr int limit(int n) { return n < 0 ? 0 : n < 63 ? n : 63; }
    // loads that may be outstanding: at the acquisition of chunk c (with chunk 0 of a block its extra
    // has to be there, requested two blocks ago)
    static constexpr int chunk_wait(int c)
    {
        int n = acquired(c) - (acquired(c - R + 1) + NA);
        if (c == 0 && 2 * period - NA - 1 < n) n = 2 * period - NA - 1;
        return limit(n);
    }
    // ... when stage s has made its requests and reads what the weight requests of stage `at`, `blocks` blocks
    // ago (0: this block), brought
    static constexpr int weight_wait(int s, int at, int blocks)
    {
        return limit(after_weights(s) + ((s + 1) % SPC == 0 ? NA : 0) - (after_weights(at) - blocks * period));
    }
};

// Few row tiles: a wave's weights come in units, whole rows of one block of K, or of two (Q4_K and Q5_K against one tile of one
// plane), and a unit is read into registers before the next one is requested into the same place.  What that is for is the
// CU's requests, which take longer the more lines a wave-load touches, 32 rows x 32 bytes as the parts have them
// (a stream of 28672 x 4096 Q4_K weights alone, eight waves a CU: 17.5 us so, whole rows 14.3, two blocks of a row 13.0).
// us a launch, parts, units of one block, of two (bits are the same):
//   Q4_K 16 rows 28672 x 4096, one plane        26.9, 27.1, 25.1     Q5_K 16 rows 13824 x 5120, one plane  21.5, 21.2, 19.8
//   Q4_K 16 rows 57344 x 8192, one plane        85.9, 86.1, 76.7     Q5_K 32 rows, two planes              23.7, 23.8, 24.1
//   Q4_K 32 rows 14336 x 4096, two planes       18.2, 17.9, 18.9     Q5_K 48 rows, two planes              31.5, 31.1, 32.9
//   Q4_K 64 rows 28672 x 4096, two planes       43.2, 40.8, 44.1     Q4_K 64 rows, one plane               32.8, 33.2, 33.4
//   Q6_K 16 rows 4096 x 14336, two planes       26.2, 24.5           Q6_K 64 rows 14336 x 4096, one plane  31.4, 28.5
//   Q6_K 2048 rows 4096 x 14336, two planes     610, 585             Q6_K 48 rows 14336 x 4096, two planes 35.3, 32.6
//   Q8_0 64 rows 28672 x 4096, one plane        48.4, 50.6           (both while its quants were read off any alignment; not timed since)
// Q5_K against two planes keeps the parts: calls of 160 drawn shapes of 9 to 130 rows are level (in the mean up to 16 rows parts 0.5 %
// shorter, above within 0.2 %; single ones 5 % either way).
// Experts, all of whose CUs stream weights at once, take units against two tiles of one plane as well (512 tokens, top 8 of 128 experts of
// 4096 x 1536, the call: Q4_K 589 us, so 585, Q5_K 628, 619; with workgroups of four waves 581, 572 and 622, 605).
constexpr bool mmfw_units(int fmt, int planes, int mt, int grouped)
{
    if (grouped && fmt <= 1 && planes == 1 && mt == 2) return true;
    return fmt == 2 ? mt <= 2 : fmt == 1 ? planes == 1 && mt == 1 : fmt == 0 && mt <= planes;
}
template <int FMT, int PL, int MT, int NWAVES = MMFW_WAVES>
struct MmfwUnitShape {
    using F = MmfwFormat<FMT>;
    using W = MmfwShape<FMT, PL, MT, false, false, NWAVES>;
    static constexpr int WAVES = NWAVES;
    static constexpr int UB = FMT <= 1 && PL == 1 ? 2 : 1;                            // blocks of K in a unit
    static constexpr uint32_t ROW = FMT == 2 ? 224u : UB * F::BLOCK;                  // bytes of a row in LDS (Q6_K: 208 and a window of 16 that ends with the block)
    static constexpr int ROW_PIECES = ROW / 16u;
    static constexpr int LW = (32 * ROW_PIECES + 63) / 64;                            // wave-loads of a unit
    static constexpr uint32_t STAGE = LW * 1024u;
    static constexpr int UC = W::UC, R = FMT == 1 && UB == 2 ? 3 : 4, C = W::C, NA = W::NA;      // the activations' ring, as above
    static constexpr uint32_t CHUNK = W::CHUNK, TILE_CHUNK = W::TILE_CHUNK, EXTRA = W::EXTRA, extra = 0;
    static_assert(NA == 2 && TILE_CHUNK % (NA * 1024u) == 0, "a wave's pieces of a chunk are two neighbours");
    static constexpr uint32_t stage = 4u * EXTRA;
    static constexpr uint32_t ring = stage + WAVES * STAGE;
    static constexpr uint32_t total = ring + R * CHUNK;
    static_assert(total <= 160u * 1024u, "LDS");
    static constexpr int SG = W::SG, NS = W::NS, SPC = W::SPC;
    static constexpr int T = UB * NS;              // stages of a unit
    static constexpr int REQUEST = 1;              // first stage that requests of the next unit; the last reads of this one are in stage 0
    static constexpr int SPREAD = T - 2 - REQUEST > LW ? LW : T - 2 - REQUEST; // stages that share the requests
    static constexpr int asked(int t) { return t <= REQUEST ? 0 : t - REQUEST >= SPREAD ? LW : (t - REQUEST) * LW / SPREAD; } // wave-loads requested ahead of stage t

    // ---- the wave's sequence of loads, a unit being a period: stage t requests weights (t = REQUEST), then the extra of the
    // block after next (first stage of a block); then, in the last stage of a chunk, the next chunk is acquired: its arrival is
    // waited for and NA pieces of the chunk R - 1 further on are requested.
    static constexpr int own(int t) { return asked(t + 1) - asked(t) + (t % NS == 0 ? 1 : 0); }
    static constexpr bool acquires(int t) { return (t + 1) % SPC == 0; }
    static constexpr int ahead_of(int t) // loads ahead of stage t
    {
        int blk = 0, n = 0;
        while (t < 0) { t += T; --blk; }
        for (int i = 0; i < t; ++i) n += own(i) + (acquires(i) ? NA : 0);
        int period = 0;
        for (int i = 0; i < T; ++i) period += own(i) + (acquires(i) ? NA : 0);
        return n + blk * period;
    }
    static constexpr int own_at(int t) { return own((t + T) % T); }
    static constexpr int limit(int n) { return n < 0 ? 0 : n < 63 ? n : 63; }
    // loads that may be outstanding at stage t's acquisition; with the first chunk of a block its extra has to be there,
    // requested in the first stage of the block before this one
    static constexpr int chunk_wait(int t)
    {
        const int now = ahead_of(t) + own(t), from = t - (R - 1) * SPC;
        int n = now - (ahead_of(from) + own_at((from % T + T) % T) + NA);
        const int ex = t - (NS - 1) - NS;
        if ((t + 1) % NS == 0 && now - (ahead_of(ex) + own_at((ex % T + T) % T)) < n) n = now - (ahead_of(ex) + own_at((ex % T + T) % T));
        return limit(n);
    }
    // ... in stage t, behind its acquisition, where the unit requested in stage REQUEST of this period is read
    static constexpr int weight_wait(int t)
    {
        const int last = REQUEST + SPREAD - 1;
        return limit(ahead_of(t) + own(t) + (acquires(t) ? NA : 0) - (ahead_of(last) + asked(last + 1) - asked(last)));
    }
};

// Q6_K weights decoded once per call (mmfx.hip.inc).  A record: 32 weight rows x one block of K, [K step 0..15][lane] 16 bytes of
// f16 operands (q - 32; lane = row + 32 half, elements 16 step + 8 half .. + 7), the rows' sixteen scales each, their d as f32; records lie
// [32 rows][block].
struct MmfxRecord {
    static constexpr uint32_t scales = 16u * 1024u, d = scales + 512u, bytes = d + 128u;
};
constexpr int MMFX_DECODE_WAVES = 4; // records of a workgroup that decodes
struct MmfxDecodeParams {
    const uint8_t *w; // first row of the slab
    uint8_t *out;
    uint32_t n, groups, row_bytes; // rows of the slab
};
template <int PL, int MT>
struct MmfxShape {
    using W = MmfwShape<2, PL, MT>; // the activations' ring is as it is there
    static constexpr int UC = W::UC, R = W::R, C = W::C, NA = W::NA, SPC = W::SPC;
    static constexpr uint32_t CHUNK = W::CHUNK, TILE_CHUNK = W::TILE_CHUNK, EXTRA = W::EXTRA, extra = 0, ring = 4u * EXTRA, total = ring + R * CHUNK;
    static constexpr int AHEAD = 8;  // K steps that weights are requested ahead
    static constexpr int BEHIND = 1; // of those ahead of the loop, steps requested behind the last chunk, as a unit has it
    static constexpr int SCALES = 4; // unit that requests the next block's scales
    // ---- the wave's sequence of loads, a block being a period: unit u requests the extra of the block after next (u = 0), scales and d (u =
    // SCALES) and, behind its first step, a step's weights; then, in the last unit of a chunk, the next chunk is acquired, and NA pieces of
    // the one R - 1 further on are requested; then the second step's weights.
    static constexpr int own(int u) { return (u == 0 ? 1 : 0) + (u == SCALES ? 2 : 0) + 1; }
    static constexpr bool acquires(int u) { return (u + 1) % SPC == 0; }
    static constexpr int all(int u) { return own(u) + (acquires(u) ? NA : 0) + 1; }
    static constexpr int ahead_of(int u) // loads ahead of unit u
    {
        int blk = 0, n = 0, period = 0;
        while (u < 0) { u += 8; --blk; }
        for (int i = 0; i < u; ++i) n += all(i);
        for (int i = 0; i < 8; ++i) period += all(i);
        return n + blk * period;
    }
    // loads that may be outstanding at unit u's acquisition (a block's extra is older than any chunk that is waited for before it is read)
    static_assert((R - 1) * SPC <= 15, "extra");
    static constexpr int chunk_wait(int u)
    {
        const int from = u - (R - 1) * SPC, n = ahead_of(u) + own(u) - (ahead_of(from) + own((from % 8 + 8) % 8) + NA);
        return n < 63 ? n : 63;
    }
    // Every load of a wave in its order, the ones ahead of the loop and three blocks': is there any acquisition whose chunk could still be
    // on its way by its wait alone?  (The compiler's waits for weights, which it puts ahead of a step's products, are tighter today; nothing
    // promises that.)
    static constexpr bool waits_cover()
    {
        int issued = 0, behind[3 * 8 / SPC + R] = {}; // behind[q]: loads up to the last piece of chunk q
        issued += 2 + 2 + AHEAD - BEHIND; // scales and d, extras, weights
        for (int q = 0; q < R - 1; ++q) behind[q] = issued += NA;
        const int landed = issued;
        behind[R - 1] = issued += NA;
        issued += BEHIND;
        for (int u = 0; u < 3 * 8; ++u) {
            issued += own(u % 8);
            if (acquires(u % 8)) {
                const int q = (u + 1) / SPC;
                if (behind[q] > landed && issued - behind[q] < chunk_wait(u % 8)) return false;
                behind[q + R - 1] = issued += NA;
            }
            ++issued;
        }
        return true;
    }
};
static_assert(MmfxShape<1, 2>::waits_cover() && MmfxShape<1, 3>::waits_cover() && MmfxShape<1, 4>::waits_cover() && MmfxShape<2, 2>::waits_cover() &&
              MmfxShape<2, 3>::waits_cover() && MmfxShape<2, 4>::waits_cover(), "a chunk is read before it is sure to have arrived");

// A workgroup may take several weight tiles against its activation rows one after the other: the requests go on into the next
// tile, so its first loads, the arguments and the way in are not waited for again.  Prompts of 16-bit elements: 2048 rows of 28672 x
// 4096 Q4_K, seven rounds of workgroups 532 us, seven tiles a workgroup 502; of 6144 x 4096 141, 133 (three).  Two planes and
// Q6_K lose 1 to 3 % to the registers it takes, for experts (tiles of unequal length) it came to nothing: 645, 642.
constexpr bool mmfw_may_run(int fmt, int planes, int mt, bool grouped) { return fmt <= 1 && planes == 1 && mt >= 2 && !grouped; }

// A workgroup of one row tile whose slice of K is this short makes its images itself.
template <int FMT, int PL> constexpr uint32_t mmfw_own_blocks() { return MmfwShape<FMT, PL, 1, false, true>::OWN_BLOCKS; }
template <int FMT, int PL> constexpr uint32_t mmfw_own_lds() { return MmfwShape<FMT, PL, 1, false, true>::total; }

template <int FMT, int PL, int MT, int GROUPED = MMFW_DENSE> constexpr uint32_t mmfw_lds()
{
    using W = MmfwShape<FMT, PL, MT, false, false, mmfw_waves(GROUPED)>;
    using U = MmfwUnitShape<FMT, PL, MT, mmfw_waves(GROUPED)>;
    if constexpr (mmfw_units(FMT, PL, MT, GROUPED)) return U::total > W::total ? U::total : W::total;
    else return W::total;
}
// ... of a grouped launch, whose jobs have any number of tiles
template <int FMT, int PL, int GROUPED> constexpr uint32_t mmfw_grouped_lds()
{
    constexpr uint32_t one = mmfw_lds<FMT, PL, 1, GROUPED>(), two = mmfw_lds<FMT, PL, 2, GROUPED>(), few = one > two ? one : two;
    if constexpr (GROUPED == MMFW_EXPERTS_FEW) {
        static_assert(few <= 80u * 1024u, "two workgroups a CU");
        return few;
    } else {
        constexpr uint32_t three = mmfw_lds<FMT, PL, 3, GROUPED>(), four = mmfw_lds<FMT, PL, 4, GROUPED>(), many = three > four ? three : four;
        return few > many ? few : many;
    }
}

struct MmfwSeg {
    const uint8_t *w;
    float *y;
    float *partial;    // [ksplit][m][n] when ksplit > 1
    uint32_t n, tile0; // weight rows; index of the matrix's first 256-row tile in the launch
    uint32_t first_record_row; // decoded weights: rows of 32 ahead of the first that `w` holds
    uint64_t expert_stride; // grouped: bytes between the experts' matrices
};

struct MmfwParams {
    MmfwSeg seg[MMFW_MAX_SEGS];
    const uint8_t *ximg;
    const float *inv;          // [groups][inv_ld]
    uint32_t segs, groups, row_bytes, m, k;
    uint32_t row_tiles;        // images per block of K = ceil(m / 32)
    uint32_t inv_ld;
    uint32_t m_tiles, n_tiles; // workgroup tiles of activation rows and of weight rows (all matrices)
    uint32_t ksplit, blocks_per_split;
    uint32_t run_mask;         // blocks whose sums are taken in one run, less one (a power of two less one; all ones: a slice's all)
    uint32_t run_tiles;        // weight tiles that a workgroup multiplies one after the other (more than one: all of K, four or more blocks)
    uint32_t n_runs;           // runs of them: ceil(n_tiles / run_tiles)
    uint32_t items;            // m_tiles * n_runs * ksplit
    uint32_t band;             // activation tiles that neighbouring workgroups share a weight tile over
    uint32_t elem;             // element type of y
    // Grouped launch (experts): jobs[0 .. counters[2]) take the place of the activation tiles, row r of job J
    // is output row J.p0 + r.  Or, where a workgroup makes its images itself: the activations, bytes between their rows, their
    // element type.
    union {
        const struct MoeWideJob *jobs;
        const uint8_t *x;
    };
    union {
        const uint32_t *counters;
        struct { uint32_t x_row_bytes, x_elem; };
    };
    uint32_t max_jobs;         // entries of `jobs` that exist at most
};

struct MmfwPrepParams {
    const float *x;
    uint8_t *ximg;
    float *inv;
    uint32_t m, k, ldx, groups, inv_ld;
    uint32_t act_bf16, elem;
    // grouped launch: image t (below counters[3]) holds the rows tiles[t].p0 + r; their activations are row
    // row_of[that], or that row itself
    const struct MoeTile *tiles;
    const uint32_t *row_of, *counters;
    uint32_t lo_first;     // two planes: see mmfw_lo_first
    uint32_t natural;      // K order inside 32 elements: 1: step s, half h = 16 s + 8 h; 0: 16 h + 8 s
    uint32_t glu, glu_off; // x[i] = act(x[i]) * x[i + glu_off] (0 off, 1 SiLU, 2 SiLU behind a ReLU)
    uint32_t slices;       // ... where both are sums of K slices, `slice_ld` elements apart, that nobody has added up yet (0, 1: they are whole)
    uint32_t slice_ld;
};

struct MmfPrepParams {
    const float *x;
    uint8_t *ximg;
    uint32_t m, k, ldx, act_bf16;
    uint32_t elem; // element type of x
    uint32_t glu, glu_off; // x[i] = act(x[i]) * x[i + glu_off] (0 off, 1 SiLU, 2 SiLU behind a ReLU)
};

struct MmfReduceSeg {
    const float *partial; // [ksplit][m][n]
    float *y;             // [m][n]
    uint32_t n, first_wg; // the matrix's first workgroup
};

struct MmfReduceParams {
    MmfReduceSeg seg[MMFW_MAX_SEGS];
    uint32_t segs, m, ksplit;
    uint32_t elem; // element type of y
};

struct GatherParams {
    const uint8_t *table;   // [vocab] rows of row_bytes
    const uint32_t *ids;    // [count]
    float *out;             // [count][hidden]
    uint32_t vocab, hidden, row_bytes;
    uint32_t quads_per_row; // hidden / 4
    uint32_t count;
    float scale;            // 1.0f when the lookup is not scaled
    uint32_t elem;          // the 16-bit kernels: element type of out (ELEM_F16 / ELEM_BF16)
    uint32_t rows;          // looked-up rows per workgroup, at most GATHER_ROWS
};
constexpr uint32_t GATHER_ROWS = 2;

struct GluActParams {
    const float *g; // gate results, row r at g + r * ld
    const float *u; // up results, row r at u + r * ld
    float *h;       // [m][ffn]
    uint32_t m, ffn, ld, relu_gate;
};

struct ConvertParams {
    const void *src;
    void *dst;
    uint64_t count;  // elements
    uint32_t elem;   // the 16-bit type (ELEM_F16 / ELEM_BF16); gq_finish_elem: any element type
    uint32_t widen;  // 1: 16-bit -> f32, 0: f32 -> 16-bit
    uint32_t accumulate, pad; // gq_finish_elem: dst = round(dst + src) instead of round(src)
};

struct ArgmaxParams {
    const float *logits; // [rows][ld]
    uint32_t *token;     // [rows]
    float *value;        // [rows] or null: the winning logit
    uint64_t *keys;      // [rows][parts] scratch between the two launches
    uint32_t n, ld;      // entries per row, elements between rows
    uint32_t parts;      // workgroups per row
    uint32_t chunk;      // entries per part
};

constexpr uint32_t ARGMAX_NONE = 0xFFFFFFFFu; // the row has no entry that is not NaN
constexpr uint32_t ARGMAX_MAX_PARTS = 128, ARGMAX_MAX_ROWS = 64; // scratch keys per launch pair

struct MoeJob {
    uint32_t expert;
    uint32_t p0;     // sorted position of the job's first pair
    uint32_t m;      // pairs in the job: 1 or 2
    uint32_t t0, t1; // their tokens (t1 = t0 when m = 1)
};

// All tokens of one expert, up to eight (or four) at a time: a job of the int8 matrix-core kernels.
struct MoeJob8 {
    uint32_t expert;
    uint32_t p0;     // sorted position of the job's first pair
    uint32_t m;      // pairs in the job: 1..8
    uint32_t pad;
    uint32_t tok[8]; // their tokens (entries past m repeat the last one)
};

// The GEMM's view of the sorted pairs (mmfw.hip.inc): a tile is up to 32 of them, of one expert; a job
// is an expert's consecutive tiles that a workgroup multiplies together.
struct MoeTile {
    uint32_t p0, rows; // first sorted position, pairs
};
struct MoeWideJob {
    uint32_t expert, tile0, p0, rows;
};

constexpr int MOE_PLAN_THREADS = 1024;
constexpr uint32_t MOE_PLAN_FEW = 192, MOE_PLAN_FEW_THREADS = 256; // most pairs of gq_moe_plan_few, a thread each
static_assert(MOE_PLAN_FEW <= 255, "counts of a byte");

struct MoePlanParams {
    const uint32_t *route_expert; // [tokens][top_k]
    const uint32_t *route_len;    // [tokens]
    uint32_t *pair_src;
    uint32_t *pair_pos;
    MoeJob *jobs;
    MoeJob8 *jobs8;
    MoeTile *tiles;     // null, or the GEMM's tables are written instead of the two job lists
    MoeWideJob *wide;
    uint32_t *token;    // [pairs] token of each sorted position
    uint32_t *counters; // [0] jobs, [1] routed pairs, [2] matrix-core (or GEMM) jobs, [3] tiles of 32
    uint32_t tokens, top_k, experts, pairs;
    uint32_t top_k_inverse; // 2^32 / top_k, rounded down
    uint32_t experts_per_thread; // rounded up
    uint32_t job_shift; // a matrix-core job takes up to 1 << job_shift tokens of an expert
    uint32_t in_lds;    // the pairs' experts and the sorted order fit the LDS
};

constexpr uint32_t MOE_NONE = 0xFFFFFFFFu;

struct MoeGemvParams {
    GemvParams g;            // shape, split and LDS fields; w/x/y are the bases
    const MoeJob *jobs;
    const uint32_t *counters;
    uint64_t expert_stride;  // bytes between experts in g.w
    uint32_t wgs_per_job;
    uint32_t x_by_token;     // 1: activation row = token index, 0: sorted position
    uint32_t x_stride;       // elements between activation rows
    uint32_t y_stride;       // elements between output rows (by sorted position)
};

struct MoeMm8Params {
    Mm8Params g;             // shape of one expert's matrix; w, x, y are the bases
    const MoeJob8 *jobs;
    const uint32_t *counters;
    uint64_t expert_stride;  // bytes between experts in g.w
    const uint8_t *up;       // gated form: the up rows of expert 0 (g.w then holds the gate rows)
    uint64_t up_stride;      // bytes between experts in `up`
    uint32_t slices;         // workgroups that share one job's tiles (the streamed kernels cut runs of tiles across jobs instead)
    uint32_t y_stride;       // elements between output rows (by sorted position)
    const uint32_t *rows;    // null: the activation rows are the job's tokens; else this table (0, 1, ...)
                             // counts from the job's first sorted position
};

// Router (route.hip.inc): gate logits -> route table.
struct MoeRouteParams {
    const float *logits;     // [tokens][experts]
    uint32_t *route_expert;  // [tokens][top_k]
    float *route_weight;     // [tokens][top_k]
    uint32_t *route_len;     // [tokens]
    uint32_t *route_pos;     // [tokens][top_k] or null: the token's place in its expert's list
    uint32_t *expert_counts; // [experts] or null
    uint32_t *overflow;      // [1] or null: choices dropped because their expert was full
    uint32_t tokens, experts, top_k;
    uint32_t capacity;       // tokens an expert takes
    uint32_t phases;         // bit 0: softmax and top-k, bit 1: capacity filter (one workgroup)
};

constexpr int ROUTE_WAVES = 8;
constexpr int ROUTE_THREADS = 64 * ROUTE_WAVES;
constexpr uint32_t ROUTE_MAX_EXPERTS = 4096, ROUTE_MAX_TOP_K = 64;
constexpr uint32_t ROUTE_FUSED_MAX_TOKENS = 64; // up to here both phases are one launch

struct MoeActParams {
    const float *gu; // [pairs][2 * ffn]
    float *h;        // [pairs][ffn]
    const uint32_t *counters;
    uint32_t ffn, relu_gate;
};

struct MoeCombineParams {
    const float *o;               // [pairs][hidden] by sorted position
    const float *route_weight;    // [tokens][top_k]
    const uint32_t *route_len;    // [tokens]
    const uint32_t *pair_pos;     // [tokens][top_k]
    float *out;                   // [tokens][hidden]
    uint32_t tokens, top_k, hidden;
    uint32_t elem;                // element type of out
};

} // namespace gq

#endif
