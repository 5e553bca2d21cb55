// wtc_kernels.h -- device data layout shared by the HIP kernels and the host
// code that launches them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wtc {

constexpr int kWave = 64;               // CDNA wavefront
constexpr int kWavesPerBlock = 4;       // counting-kernel block = 256 lanes
constexpr int kBlock = kWave * kWavesPerBlock;
constexpr int kCountWavesMax = 8;       // counting-kernel block: 1..8 waves, chosen per launch
constexpr uint32_t kChunkMax = 16;      // wedges per lane staged in LDS at once
constexpr int kTreeLevels = 12;         // cached levels of the wedge-prefix search tree
constexpr uint32_t kTreeSize = (1u << kTreeLevels) - 1u;
constexpr int kScanItems = 16;          // vertices per thread in the prefix scan
constexpr uint32_t kScanChunk = kBlock * kScanItems;  // vertices per scan block
constexpr uint32_t kSentinel = 0xffffffffu;           // empty LDS wedge slot
constexpr int kSmallBlock = 512;        // small-graph kernel block: one graph per block
// Largest LDS footprint, in 32-bit words, of a graph the small-graph kernel
// takes: 2(n+1) + m <= 2^16 keeps m < 2^16, so W <= C(m,2) < 2^31 and every
// wedge index of such a graph fits 32 bits.
constexpr uint32_t kSmallWordsMax = 1u << 16;

// Wedges per block the host aims at when it splits a graph of a small-graph
// set over several blocks of the small-graph kernel.
constexpr uint64_t kSmallBlockWedges = 16384;

// One block of the small-graph kernel: wedges [wcount*part/parts,
// wcount*(part+1)/parts) of graph g's range.
struct SmallPart {
    uint32_t g;
    uint16_t part, parts;
};
static_assert(sizeof(SmallPart) == 8, "SmallPart layout");

// GraphDesc::mode
enum : uint32_t {
    kModeTiles = 0,  // counted by k_count in tiles of 64*s wedges
    kModeSmall = 1,  // counted by k_count_small, one block with the CSR in LDS
    kModeInvalid = 2,  // failed the device-side CSR check: nothing is read
                       // beyond rowPtr, and its count is set to kCountInvalid
};

// Count of a graph whose CSR failed the device-side check.
constexpr unsigned long long kCountInvalid = ~0ull;

// A tile of edges, in-edges or packed chunks goes through the rows it spans in
// windows of one row a thread.  After this many windows, where most rows are
// empty, it finds the rows of its positions instead, one search a thread: some
// ten windows' time, for any number of empty rows between.  (Three million
// vertices without out-edges between the triangles and a dense core: row count
// 3.6 -> 0.22 ms, split count 14.4 -> 0.48.)
constexpr uint32_t kRowWindows = 16;

// Edges per tile of the row count (wtc_rows.hip).
constexpr uint32_t kRowsTile = 512, kRowsTileMin = 256;

// One graph of a graph set.  A graph set is any number of oriented CSRs
// resident in HBM (ids local to each graph, row offsets relative to the
// graph's own colInd); one count launch covers all of them.  A single graph
// is a set of one.  The host fills the first block of fields, the setup
// kernel the last three.
struct GraphDesc {
    // host-filled
    const void *rowPtr;      // n+1 offsets of the set's offset width
    const uint32_t *colInd;  // ids in [0, n), every row strictly ascending
    uint64_t *ws;            // n+1 wedge prefix (workspace slice)
    uint32_t *bitmap;        // ceil(C(a,2)/32) words (workspace slice), or null
    uint64_t bm_words;       // a*a/32: words of the graph's top-a bitmap
    uint64_t row_base;       // first bitmap row of this graph in the set's row list
    uint64_t blk_base;       // first prefix-scan block of this graph
    uint64_t bm_clear_base;  // first bitmap word of this graph in the set's clear list
    uint64_t w_begin;        // wedge range to count, relative to the graph
    uint64_t w_end;
    uint32_t n;              // vertices
    uint32_t spread;         // wedges per lane (s)
    uint32_t a;              // bitmap length (top-a ranks), multiple of 32
    uint32_t thr;            // bitmap threshold max(n,a) - a (a = 0: n)
    uint32_t bm_rows;        // min(n, a)
    uint32_t mode;           // kModeTiles, kModeSmall or kModeInvalid
    // device-filled by the setup kernel (the row count: host-filled)
    uint64_t wbase;          // first counted wedge (graph-local index)
    uint64_t wcount;         // wedges counted (the row count: edges)
    uint64_t tile_base;      // first tile of this graph
};
static_assert(sizeof(GraphDesc) == 128, "GraphDesc layout");

// meta[] slots written by the setup kernel
// (kMetaNext..kMetaNext+7: per-XCD work counters of the counting kernel).
// The split count: kMetaTopWedges and kMetaListWedges, the wedges of its row
// and its slab kernel; kMetaInEdges, the top rows' in-edges; kMetaAllEdges, every
// grouped in-edge.
enum : int {
    kMetaTiles = 0,
    kMetaWedges = 1,
    kMetaTopWedges = 3,
    kMetaInEdges = 4,
    kMetaListWedges = 6,
    kMetaAllEdges = 7,
    kMetaNext = 8,
    // split count: what its dense part took of the top rows' totals
    kMetaDenseTopWedges = 8,
    kMetaDenseTopEdges = 9,
    kMetaSlots = 16
};

// Sums and tile counters that every block adds to.  Atomics to one 128-byte
// line take 12.1 ns each, one after another, wherever in the line and from
// however many blocks; to 64 lines 0.3 ns.  With one line for all, the row
// kernel's 18,432 tile grabs on R-MAT-20 took 0.22 ms of its 0.45 and its
// 8,192 waves' counts another 0.1.  So they are spread over lines by the block's
// number and summed when they are read (k_publish), and a block takes its tiles
// from its line's counter, which holds every kTileLines-th tile.
constexpr uint32_t kLineWords = 16;                 // 8-byte words of a line
constexpr uint32_t kSumLines = 64, kTileLines = 16;
constexpr uint32_t kLineRows = kSumLines, kLineSlabs = kLineRows + kTileLines;  // first tile counters of the two kernels
constexpr uint32_t kLines = kLineSlabs + kTileLines;
constexpr uint32_t kLineHits = 0, kLineWedges = 1;  // a sum line's words
// Where they start behind meta and the counts of G graphs, in words.
__host__ __device__ constexpr uint32_t lines_at(uint32_t G) {
    return (kMetaSlots + G + kLineWords - 1) / kLineWords * kLineWords;
}

// Split count of one graph (wtc_split.hip).  The in-edges are grouped by key
// in counting-sort levels: by part of 1 << part_shift keys, at most
// kSplitPartsMax parts, then by key.  With up to kSplitPartsMax <<
// kSplitFinalMax keys (R-MAT-24: 389,000) a part is at most 1 <<
// kSplitFinalMax keys and the second level groups by key; beyond that (up to
// kSplitPartsMax << kSplitPartMax keys), parts are first grouped by sub-part
// of kSplitSub keys (at most kSplitFan2 a part).  kSplitBlock: threads per
// transposition block; a tile of the row kernel is kSplitTileMinWork to
// kSplitTile units of work, an in-edge being one and a row kSplitRowCost.
constexpr uint32_t kSplitPartMax = 15;
constexpr uint32_t kSplitPartsMax = 256;
constexpr uint32_t kSplitFinalMin = 8, kSplitFinalMax = 11;
constexpr uint32_t kSplitSubShift = 8;
constexpr uint32_t kSplitSub = 1u << kSplitSubShift;
constexpr uint32_t kSplitFan2 = 1u << (kSplitPartMax - kSplitSubShift);
static_assert(kSplitPartMax <= 16 && kSplitSubShift <= 8, "A keys fit 16 bits, B keys 8");
// Records per block of the second and final levels: kSplitChunkMax, or as
// few as kSplitChunkMin for small graphs, so that the levels fill the GPU.
constexpr uint32_t kSplitChunkMax = 65536, kSplitChunkMin = 8192;
constexpr int kSplitBlock = 1024;
constexpr uint32_t kSplitTile = 1024, kSplitTileMinWork = 128;
constexpr uint32_t kSplitRowCost = 32;
// Keys per block of the key-offset scan (four per thread).
constexpr uint32_t kKeyChunk = 4 * kSplitBlock;
// Slabs of the list rows (middle vertex below thr): slab s holds the rows
// whose adjacency starts in colInd[s*kSlabSpan, (s+1)*kSlabSpan).  The slab
// kernel hashes colInd[s*kSlabSpan, +kSlabWin) into LDS, one bucket of
// four slots per position, which covers every such row of out-degree
// <= kSlabRowMax (longer rows are searched in HBM).
constexpr uint32_t kSlabSpan = 2048;
constexpr uint32_t kSlabRowMax = 1024;
constexpr uint32_t kSlabWin = kSlabSpan + kSlabRowMax;
constexpr uint32_t kSetIdsEnd = 0x7fffffffu;  // the LDS sets of ids (wtc_set.h) hold ids below this, but for the wide ones
constexpr uint32_t kSlabLong = 72;  // list tails are streamed by eight lanes where they hold this many ids on average
constexpr uint32_t kSlabTile = 1024, kSlabTileMin = 128, kSlabCost = 48;  // a tile's work; a slab's share of it

// Workspace and device-filled state of a split count.  The top rows are the
// ranks [thr, n) of the graph's GraphDesc; OffT arrays use the set's offset
// width.  Every in-edge (v, j) (j a position of adj+(v) other than its last)
// is grouped by a key: w - thr for w = colInd[j] >= thr (a top row), else
// rows + the slab of w.  Records (key, pair, slab_aux) go through the
// levels A -> ie or A -> B -> ie: A bucketed by part, B by sub-part, ie by
// key (the pairs, and a list record's slab_aux), in the arrays of the level
// before the last: B's when there is no B.  A record's position names its
// part (in A) or sub-part (in B), so A keeps the key's low part_shift bits
// and B its low 8.  A top record's pair is its tail's first packed chunk and
// number of chunks; a list record's is (j, hi), its tail [j + 1, hi) of colInd.
struct SplitDesc {
    uint64_t *ws_full;    // n+1: the full wedge prefix
    uint64_t *ie_pre;     // n+1: prefix of the in-edges of each row (its first positions)
    uint32_t *tile_v;     // first-level tiles: the vertex each starts in
    uint64_t *part_base;  // parts: first record slot of each part
    uint64_t *part_cnt;   // parts: records of each part so far
    uint32_t *c2base;     // parts+1: first second-level block of each part
    uint32_t *hist2;      // c2cap x kSplitFan2: second-level counts, then column prefixes
    uint64_t *sub_base;   // subs: first record of each sub-part
    uint32_t *c3base;     // final buckets+1: first final-level block of each part or sub-part
    uint32_t *hist3;      // c3cap << final_shift: final-level counts, then column prefixes
    uint32_t *sub_tot;    // subs: records of each sub-part
    uint32_t *list_bid;   // parts: the first list vertex w whose key lies in each part (0 up to the first list part)
    uint64_t *part_tot;   // parts: record slots of each part (>= its records)
    uint64_t *tally;      // 1: wedges of the top rows' in-edges
    uint64_t *key_part;   // key blocks: in-edges of each block of kKeyChunk keys, then their prefix
    uint32_t *key_tot;    // keys: in-edges of each key
    uint16_t *rec_id;     // cap: A keys within their part
    void *rec;            // cap pairs of OffT: A pairs
    uint32_t *rec_aux;    // cap: A slab_aux words (list records)
    uint8_t *rec_id2;     // cap: B keys within their sub-part
    void *rec2;           // cap pairs of OffT: B pairs
    uint32_t *rec_aux2;   // cap: B slab_aux words
    void *rp_in;          // keys+1 OffT: first in-edge of each key
    void *ie;             // the records' pairs grouped by key: rec2 (two levels) or rec (three)
    uint32_t *ie_aux;     // the list records' slab_aux words, beside ie
    void *packed;         // 3 cap / 4 chunks of 16 bytes, the packed top ids: over the pairs (and slab words) that ie is not in
    uint64_t cap;         // records each array holds (>= the in-edges)
    uint32_t rows;        // top rows: n - thr
    uint32_t keys;        // rows + slabs
    uint32_t parts;       // parts of 1 << part_shift keys (<= kSplitPartsMax)
    uint32_t part_shift;  // log2 of a part's keys
    uint32_t final_shift;  // log2 of the keys of a final-level bucket: part_shift, or kSplitSubShift with three levels
    uint32_t subs;        // sub-parts (three levels)
    uint32_t slabs;       // slabs of the list rows: ceil(m / kSlabSpan)
    uint32_t chunk;       // records per block of the second and final levels
    uint32_t far_ids;     // ids per far chunk of the packed top ids
    // device-filled by the range kernel
    uint64_t w_lo, w_hi;  // the counted wedges of the full order, clamped to [0, W]
    uint64_t cut_j[2];    // in-edges whose tail the range cuts, and what it leaves of
    uint64_t cut_lo[2];   // them: positions [cut_lo, cut_hi) of colInd
    uint64_t cut_hi[2];
    uint32_t v_lo, v_hi;  // vertices holding w_lo and w_hi - 1 (v_lo > v_hi: none)
    uint32_t clip;        // 1 unless [w_lo, w_hi) is the whole order
    uint32_t cuts;        // cut tails: up to two
    uint32_t cut_top;     // those of top rows
    uint32_t pad_;
};

// Where adj+(w) of a list row lies in its slab's window: bits 0-12 its start
// rowPtr[w] - slab*kSlabSpan, bits 13-25 its length (kSlabAuxLong: longer
// than kSlabRowMax, searched in HBM).
constexpr uint32_t kSlabAuxLong = 0x1fffu;
static_assert(kSlabSpan <= 8192 && kSlabRowMax < kSlabAuxLong, "slab_aux fields");
static_assert(sizeof(SplitDesc) % 8 == 0, "SplitDesc alignment");

// The dense part of a split count (wtc_dense.hip).  Class q holds the
// vertices whose wedges among the last kDenseCore0 << q ranks are counted as
// a product of bit matrices.
constexpr uint32_t kDenseCore0 = 512;
constexpr uint32_t kDenseClasses = 6;
// A class's rows hold at least one id per this many columns.  At 64 the rows
// between cost as much as they save (R-MAT-20 1.31 ms either way, R-MAT-22
// 4.12 against 4.21, R-MAT-24 20.4 against 20.6).
constexpr uint32_t kDenseSparsest = 32;
// What the other kernels take for an in-edge and a wedge, in multiply-adds of
// the product (3.1e15 a second on R-MAT-24): 24 ps for the transposition and
// the row kernel's start of a tail, 0.34 ps for a probed id.  Twice or half
// as much moves R-MAT-20 to R-MAT-26 by less than 1% (half: R-MAT-22 6%).
constexpr float kDenseEdgeCost = 75000.0f, kDenseWedgeCost = 1050.0f;
// sums[]: the dense in-edges whose middle vertex is a top row, their wedges,
// and all dense in-edges.
enum : uint32_t { kDenseTopEdges = 0, kDenseTopWedges = 1, kDenseEdges = 2, kDenseSums = 3 };

struct DenseDesc {
    void *R;                             // core x core bits: the rows of the last `core` ranks
    void *B;                             // the listed rows' bits, class by class
    uint2 *list;                         // (vertex, ids in its class's columns) per class
    uint32_t *cnt;                       // kDenseClasses: listed vertices
    uint64_t *sums;                      // kDenseSums
    uint64_t list_off[kDenseClasses];    // first list entry of each class
    uint32_t classes;                    // classes in use (0: no dense part)
    uint32_t core;                       // columns of the largest class
    float edge, wedge;                   // cost of an in-edge and a wedge elsewhere, in multiply-adds here
};
static_assert(sizeof(DenseDesc) % 8 == 0, "DenseDesc alignment");

}  // namespace wtc
