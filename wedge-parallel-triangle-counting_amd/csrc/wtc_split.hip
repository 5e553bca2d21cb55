// wtc_split.hip -- the split count of one graph (counting kernel choice
// kKernelSplit).  Every wedge (v, w, u) of a degree-oriented CSR belongs to
// one in-edge v -> w: w = colInd[j] at a position j of adj+(v) that is not
// the row's last, and u runs over the row's tail colInd[j+1 .. e).  The
// in-edge closes |tail ∩ adj+(w)| triangles.  The in-edges are grouped by
// their middle vertex w with a counting sort built per count, and counted in
// two kernels chosen by w:
//
//  * w among the top-a ranks (w >= thr): the wedges whose probe the
//    reference answers from its top-a bitmap (tc.cu:262-272).  One key per
//    row.  A block of the row kernel holds adj+(w) as a bitmap of a bits in
//    LDS, and its waves stream the tails of w's in-edges through it from a
//    packed copy of colInd (a row's ids from its top one down, 16 to 21 bits
//    each, six to eight per 16-byte load).  Each probe is one LDS read, and
//    the top-a bitmap never exists in HBM: one row of it at a time in LDS
//    instead of a*a/8 bytes.
//  * w below thr: the sorted-list probes of tc.cu:273-286.  One key per slab
//    of colInd (kSlabSpan positions; a row belongs to the slab its adjacency
//    starts in).  A block of the slab kernel hashes the rows of the slab its
//    in-edges name into LDS, and its waves stream the tails of the slab's
//    in-edges, looking each id up in adj+(w)'s hash set.
//
// A wedge range [w_begin, w_end) of the full order (the reference's wedge
// numbering, tc.cu:203-212) holds the in-edges of the vertices between its
// ends, with the tails of the two end vertices clipped.
//
// Where a row has many ids among the last ranks, its wedges there are counted
// as a product of bit matrices instead (wtc_dense.hip): those in-edges are at
// the row's end, and the rest of this file sees rows without them.
//
// Pipeline on one stream: k_split_partials, k_scan_partials and k_split_scan
// (the full wedge prefix); k_split_range; k_dense_class, k_scan_partials and
// k_split_inscan (the prefix of the in-edges left); k_dense_rows and
// k_dense_mm; the transposition, a counting sort by key: k_split_parthist
// and k_split_partbase (part sizes), k_split_l1 (records bucketed by part),
// k_split_bases; with many keys k_split_level_count, k_split_levelcols2,
// k_split_bases and k_split_level_scatter to sub-parts; then
// k_split_level_count, k_split_levelcols3, k_split_keysum, k_scan_partials,
// k_split_keyscan and k_split_level_scatter by key; k_split_pack (the
// packed ids, over the last level's input); k_split_rows (top rows);
// k_split_slabs (list rows); k_publish (the sums to the host).
#include <type_traits>
#include <utility>

#include "wtc_dev.h"
#include "wtc_kernels.h"
#include "wtc_launch.h"
#include "wtc_set.h"

namespace wtc {

namespace {

template <typename OffT>
struct TailPair {
    OffT lo, hi;  // a top record: the tail's first packed chunk, and its chunks (pack_count);
                  // a list record: (j, hi), the tail [j + 1, hi) of colInd
};

// Wedges before row i of a vertex of out-degree d in its row-major order
// (row r holds d - 1 - r wedges).
__device__ __forceinline__ uint64_t row_base(uint64_t i, uint64_t d) { return i * (d - 1) - binom2_d(i); }

// The packed copy of the top ids (k_split_pack).  A row is held from its top
// id down, so that the tail of each of its in-edges is a prefix of it: ids as
// x = n - u, first those with x <= kPackNear in 16-bit fields (near chunks),
// then the rest in wider ones (far chunks).
constexpr uint32_t kPackNear = 65528, kPackNearIds = 8;
constexpr uint32_t kPackAlign = 16;  // rows of this many ids start on a 128-byte line

// Chunk slots before those of the row that starts at position p: three for
// four ids.  A row's chunks start at its first slot, on a 128-byte line in
// rows of kPackAlign ids or more: of its d - 1 tail ids there are at most (d -
// 1) / 6 + 2 chunks and not more than d - 1, so with the alignment's 7 they
// fit.
template <typename T>
__device__ __forceinline__ T pack_slot(T p) {
    return p - (p >> 2);
}
template <typename OffT>
__device__ __forceinline__ OffT pack_row(OffT rb, OffT re) {
    const OffT c = pack_slot(rb);
    return re - rb >= kPackAlign ? (c + 7) & ~(OffT)7 : c;
}

// A tail's near and far chunks in one word (at most 8,191 and 349,526).
__device__ __forceinline__ uint32_t pack_count(uint32_t near, uint32_t far) { return near | (far << 13); }

// x / q for the far chunks' ids, 6 or 7 (block-uniform).
__device__ __forceinline__ uint32_t pack_div(uint32_t x, uint32_t q) { return q == 7 ? x / 7 : x / 6; }

}  // namespace

// --------------------------------------------------------------- prefixes

// Block b: vertices [b*kScanChunk, (b+1)*kScanChunk): the sum of the full
// order's wedges.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void k_split_partials(const GraphDesc *__restrict__ desc,
                                                           uint64_t *__restrict__ part_full) {
    __shared__ uint64_t s_f[kWavesPerBlock];
    const GraphDesc &D = desc[0];
    const OffT *__restrict__ rowPtr = static_cast<const OffT *>(D.rowPtr);
    const uint32_t n = D.n;
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk;
    uint64_t af = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        const uint64_t v = base + (uint64_t)k * kBlock + threadIdx.x;
        if (v < n) af += binom2_d((uint64_t)(rowPtr[v + 1] - rowPtr[v]));
    }
    af = wave_sum(af);
    if ((threadIdx.x & (kWave - 1)) == 0) s_f[threadIdx.x >> 6] = af;
    __syncthreads();
    if (threadIdx.x == 0) part_full[blockIdx.x] = s_f[0] + s_f[1] + s_f[2] + s_f[3];
}

// ws_full from the scanned block partials (n + 1 values: the last is the sum).
template <typename OffT>
__global__ __launch_bounds__(kBlock) void k_split_scan(const GraphDesc *__restrict__ desc,
                                                       const SplitDesc *__restrict__ sd,
                                                       const uint64_t *__restrict__ part_full) {
    __shared__ uint64_t s_tot[kScanRounds][kWavesPerBlock];
    const GraphDesc &D = desc[0];
    const gptr<OffT> rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
    uint64_t *__restrict__ wf = sd->ws_full;
    const uint32_t n = D.n;
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk;
    uint64_t x[kScanItems];
#pragma unroll
    for (int r = 0; r < kScanRounds; r++) {
        OffT p[5];
#pragma unroll
        for (int z = 0; z <= 4; z++) {
            const uint64_t v = base + chunk_at(r, z);
            p[z] = rowPtr[v < n ? v : n];
        }
#pragma unroll
        for (int z = 0; z < 4; z++) x[4 * r + z] = binom2_d((uint64_t)(p[z + 1] - p[z]));
    }
    const uint64_t sum = chunk_scan(x, part_full[blockIdx.x], s_tot);
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        const uint64_t v = base + chunk_at(i / 4, i % 4);
        if (v <= n) wf[v] = x[i];
    }
    if (base + kScanChunk == n && threadIdx.x == 0) wf[n] = sum;
}

// ie_pre: its counts of in-edges (k_dense_class) become their prefix.
__global__ __launch_bounds__(kBlock) void k_split_inscan(const GraphDesc *__restrict__ desc,
                                                         const SplitDesc *__restrict__ sd,
                                                         const uint64_t *__restrict__ part_in) {
    __shared__ uint64_t s_tot[kScanRounds][kWavesPerBlock];
    uint64_t *__restrict__ wi = sd->ie_pre;
    const uint32_t n = desc[0].n;
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk;
    uint64_t x[kScanItems];
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        const uint64_t v = base + chunk_at(i / 4, i % 4);
        x[i] = v < n ? wi[v] : 0;
    }
    const uint64_t sum = chunk_scan(x, part_in[blockIdx.x], s_tot);
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        const uint64_t v = base + chunk_at(i / 4, i % 4);
        if (v <= n) wi[v] = x[i];
    }
    if (base + kScanChunk == n && threadIdx.x == 0) wi[n] = sum;
}

// Thread 0: the counted range of the full order, its end vertices, and the
// in-edges whose tails the range cuts (row i0 of v_lo holding wedge w_lo: its
// tail starts w_lo - base(i0) ids in; likewise the one of wedge w_hi - 1).  Thread q < parts:
// list_bid[q], the first list vertex w (below thr) whose key rows +
// rowPtr[w] / kSlabSpan lies in part q or later (keys grow with w), and the
// part's counters zeroed.
template <typename OffT>
__global__ __launch_bounds__(kSplitPartsMax) void k_split_range(const GraphDesc *__restrict__ desc,
                                                                SplitDesc *__restrict__ sd) {
    const GraphDesc &D = desc[0];
    SplitDesc &S = sd[0];
    const OffT *__restrict__ rowPtr = static_cast<const OffT *>(D.rowPtr);
    const uint32_t q = threadIdx.x;
    if (q < S.parts) {
        const uint64_t first = S.rows >> S.part_shift;  // the part of the first list key
        uint32_t bid = 0;
        if (q > first) {
            const uint64_t at = (((uint64_t)q << S.part_shift) - S.rows) * kSlabSpan;  // colInd position
            uint32_t lo = 0, hi = D.thr;  // the first w in [0, thr] with rowPtr[w] >= at (thr: none below)
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo) >> 1);
                if ((uint64_t)rowPtr[mid] < at) lo = mid + 1;
                else hi = mid;
            }
            bid = lo;
        }
        S.list_bid[q] = bid;
        S.part_tot[q] = 0;
        S.part_cnt[q] = 0;
    }
    if (threadIdx.x != 0) return;
    const uint32_t n = D.n;
    const uint64_t *wf = S.ws_full;
    const uint64_t W = wf[n];
    const uint64_t lo = D.w_begin < W ? D.w_begin : W, hi = D.w_end < W ? D.w_end : W;
    S.w_lo = lo;
    S.w_hi = hi;
    S.cuts = 0;
    S.cut_top = 0;
    S.tally[0] = 0;
    if (lo == 0 && hi == W) {  // the whole order: nothing clipped
        S.clip = 0;
        S.v_lo = 0;
        S.v_hi = n - 1;
        return;
    }
    S.clip = 1;
    if (lo >= hi) {  // nothing to count
        S.v_lo = 1;
        S.v_hi = 0;
        return;
    }
    const uint32_t v[2] = {rightmost_le(wf, 0u, n - 1, lo), rightmost_le(wf, 0u, n - 1, hi - 1)};
    S.v_lo = v[0];
    S.v_hi = v[1];
    // the in-edges that hold the range's first and last wedge, and the
    // positions [b, e) of their tails that the range leaves
    uint64_t j[2], b[2], e[2], end[2];
    for (int z = 0; z < 2; z++) {
        const uint64_t rb = (uint64_t)rowPtr[v[z]], d = (uint64_t)rowPtr[(uint64_t)v[z] + 1] - rb;
        const uint64_t off = (z ? hi - 1 : lo) - wf[v[z]];
        uint64_t s = 0, t = d - 1;  // the last i in [0, d - 2] with row_base(i) <= off
        while (t - s > 1) {
            const uint64_t mid = s + ((t - s) >> 1);
            if (row_base(mid, d) <= off) s = mid;
            else t = mid;
        }
        j[z] = rb + s;
        end[z] = rb + d;
        b[z] = j[z] + 1 + (z ? 0 : off - row_base(s, d));
        e[z] = z ? j[z] + 1 + (off + 1 - row_base(s, d)) : end[z];
    }
    if (j[0] == j[1]) e[0] = e[1];
    for (int z = 0; z < 2; z++) {
        if ((z && j[0] == j[1]) || (b[z] == j[z] + 1 && e[z] == end[z])) continue;
        const bool top = to_global(D.colInd)[j[z]] >= D.thr;
        S.cut_j[S.cuts] = j[z];
        S.cut_lo[S.cuts] = b[z];
        S.cut_hi[S.cuts] = e[z];
        S.cuts++;
        S.cut_top += top;
        if (top) S.tally[0] += e[z] - b[z];
    }
}

// ------------------------------------------------------------ transposition

// Whether the tail [j+1, e) of in-edge j of an end vertex of the counted
// range (row start rb, full-order base ws) lies wholly in the range: the tail
// ids of row i = j - rb are the wedges [base, base + L) of the full order
// (tc.cu:203-212 numbering).  At most one tail is cut at each end of the
// range; the row kernel counts those by themselves.
template <typename OffT>
__device__ __forceinline__ bool whole_tail(OffT j, OffT e, OffT rb, uint64_t ws, uint64_t w_lo, uint64_t w_hi) {
    const uint64_t bse = ws + row_base((uint64_t)(j - rb), (uint64_t)(e - rb));
    return bse >= w_lo && bse + (uint64_t)(e - j - 1) <= w_hi;
}

// Records staged in LDS per tile of a scatter: 4096 with 4-byte offsets,
// 2048 with 8-byte ones (32 KB of pairs either way).
template <typename OffT>
struct LevelTile {
    static constexpr uint32_t kT = sizeof(OffT) == 4 ? 4096 : 2048;
    static_assert(kT >= kSplitTileMin, "tile_v holds a vertex per tile");
};

// First-level part sizes, as an upper bound: every position of the counted
// vertices' rows in its id's part (the in-edges are all of them but each
// row's last or its dense ones, and fewer where the range clips a row).  Positions in order
// run through a row's ascending ids, so neighbouring lanes mostly share a
// part: one LDS atomic per run of equal parts instead of one per id, which
// with few parts all fell on the same counters (R-MAT-20: 112 us).  A list
// vertex's part comes from list_bid (no rowPtr read).  Also finds the vertex
// that each tile of k_split_l1 starts in.
template <typename OffT>
__global__ __launch_bounds__(kSplitBlock) void k_split_parthist(const GraphDesc *__restrict__ desc,
                                                                const SplitDesc *__restrict__ sd) {
    __shared__ uint32_t s_cnt[kSplitPartsMax];
    __shared__ uint32_t s_bid[kSplitPartsMax];
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const OffT *__restrict__ rowPtr = static_cast<const OffT *>(D.rowPtr);
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const uint32_t thr = D.thr, parts = S.parts, shift = S.part_shift;
    if (S.v_lo > S.v_hi) return;  // nothing counted
    for (uint32_t i = threadIdx.x; i < parts; i += kSplitBlock) {
        s_cnt[i] = 0u;
        s_bid[i] = S.list_bid[i];
    }
    __syncthreads();
    auto part_of = [&](uint32_t id) -> uint32_t {
        if (id >= thr) return (id - thr) >> shift;
        uint32_t lo = 0, hi = parts;  // s_bid[lo] <= id < s_bid[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_bid[mid] <= id) lo = mid;
            else hi = mid;
        }
        return lo;
    };
    // the vertex that each first-level tile starts in
    {
        const cptr<uint64_t> iep = to_const(static_cast<const uint64_t *>(S.ie_pre));
        const uint64_t K0 = iep[S.v_lo], K1 = iep[(uint64_t)S.v_hi + 1];
        const uint64_t tiles = (K1 - K0 + LevelTile<OffT>::kT - 1) / LevelTile<OffT>::kT;
        for (uint64_t t = blockIdx.x * (uint64_t)kSplitBlock + threadIdx.x; t < tiles; t += gridDim.x * (uint64_t)kSplitBlock)
            S.tile_v[t] = rightmost_le(to_global(static_cast<const uint64_t *>(S.ie_pre)), S.v_lo, S.v_hi,
                                       K0 + t * LevelTile<OffT>::kT);
    }
    const uint64_t p0 = rowPtr[S.v_lo], p1 = rowPtr[(uint64_t)S.v_hi + 1];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    constexpr uint32_t kIn = 8;  // loads in flight per thread
    constexpr uint64_t kStep = (uint64_t)kIn * kSplitBlock;
    for (uint64_t base = p0 + blockIdx.x * kStep; base < p1; base += gridDim.x * kStep) {
        uint32_t id[kIn];
#pragma unroll
        for (uint32_t z = 0; z < kIn; z++) {
            const uint64_t q = base + z * kSplitBlock + threadIdx.x;
            id[z] = q < p1 ? colInd[q] : 0u;
        }
#pragma unroll
        for (uint32_t z = 0; z < kIn; z++) {
            const uint64_t q = base + z * kSplitBlock + threadIdx.x;
            const uint32_t part = q < p1 ? part_of(id[z]) : kSentinel;
            const uint32_t next = (uint32_t)__shfl_down((int)part, 1, kWave);
            const bool last = lane == kWave - 1 || next != part;
            const uint64_t ends = __ballot(last);
            if (last && part != kSentinel) {
                const uint64_t below = ends & ((1ull << lane) - 1);  // run ends before this lane
                const uint32_t first = below ? 64u - (uint32_t)__builtin_clzll(below) : 0u;
                atomicAdd(&s_cnt[part], lane + 1 - first);
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < parts; i += kSplitBlock)
        if (s_cnt[i]) atomicAdd(reinterpret_cast<unsigned long long *>(&S.part_tot[i]), (unsigned long long)s_cnt[i]);
}

// Exclusive scan over the kSplitBlock threads of a block; the block's sum
// into total.  s_w holds a word per wave.
__device__ __forceinline__ uint64_t split_block_scan(uint64_t x, uint64_t *s_w, uint64_t &total) {
    constexpr int kWaves = kSplitBlock / kWave;
    const uint64_t inc = wave_incl_scan(x);
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x >> 6;
    if (lane == kWave - 1) s_w[wv] = inc;
    __syncthreads();
    uint64_t off = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        const uint64_t t = s_w[w];
        off += w < (int)wv ? t : 0;
        all += t;
    }
    __syncthreads();
    total = all;
    return off + inc - x;
}

// One block, thread per part: part_base as the prefix of the part sizes.
__global__ __launch_bounds__(kBlock) void k_split_partbase(const SplitDesc *__restrict__ sd) {
    __shared__ uint64_t s_tot[kWavesPerBlock];
    static_assert(kSplitPartsMax <= (uint32_t)kBlock, "a part per thread");
    const SplitDesc &S = sd[0];
    const uint32_t q = threadIdx.x, parts = S.parts;
    uint64_t tt;
    const uint64_t et = block_excl_scan(q < parts ? S.part_tot[q] : 0, s_tot, tt);
    if (q < parts) S.part_base[q] = et;
}

// Exclusive prefix of the kN counts in s_cnt into s_off by a block of
// kSplitBlock threads (s_w: a word per wave); s_cnt is final and s_off and s_w
// free on entry, s_off is whole after the next barrier.
template <uint32_t kN>
__device__ __forceinline__ void block_prefix(const uint32_t *s_cnt, uint32_t *s_off, uint32_t *s_w) {
    constexpr uint32_t kPer = kN > (uint32_t)kSplitBlock ? kN / kSplitBlock : 1;
    constexpr uint32_t kWaves = kN / kPer / kWave;  // those that hold counts
    static_assert(kN % (kPer * kWave) == 0 && kWaves * kWave <= (uint32_t)kSplitBlock, "whole waves of counts");
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x >> 6;
    uint32_t v[kPer], sum = 0, incl = 0;
    if (wv < kWaves) {
#pragma unroll
        for (uint32_t z = 0; z < kPer; z++) {
            v[z] = s_cnt[threadIdx.x * kPer + z];
            sum += v[z];
        }
        incl = sum;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o, kWave);
            incl += (int)lane >= o ? y : 0u;
        }
        if (lane == kWave - 1) s_w[wv] = incl;
    }
    __syncthreads();
    if (wv < kWaves) {
        uint32_t run = incl - sum;
        for (uint32_t w = 0; w < wv; w++) run += s_w[w];
#pragma unroll
        for (uint32_t z = 0; z < kPer; z++) {
            s_off[threadIdx.x * kPer + z] = run;
            run += v[z];
        }
    }
}

// First level of the transposition.  The counted vertices' in-edges in
// order, [K0, K1) of the in-edge prefix ie_pre, are cut into tiles of kT
// that the blocks take in turn, so every block has the same work however the
// in-edges fall on the vertices, and the tiles in flight are neighbours: a
// part's records, and in the end a row's in-edges, stay nearly in the order
// of their vertices, which the row kernel's reads of the tails need (with a
// contiguous share of the tiles per block it took 19.2 instead of 16.4 ms on
// R-MAT-24).  Per tile:
//  1. the vertices that own its in-edges, read kSplitBlock at a time, mark
//     their first slot and leave their row's position and end there; a
//     running maximum over the marks tells each in-edge its vertex's slot;
//  2. every in-edge loads its id (consecutive positions, so coalesced),
//     is dropped where the counted range does not hold its whole tail, and
//     gets its key -- w - thr for a top row w, else rows +
//     rowPtr[w] / kSlabSpan -- and the part key >> part_shift;
//  3. the tile is ranked per part (LDS atomics), takes its slots of every
//     part with one global atomic per part, and leaves sorted by part
//     through LDS, a part's records as consecutive lanes of one store.
// Bound by the chain of loads and barriers of a tile, so held to 64 registers
// for two blocks a CU (with one, 96 registers: R-MAT-24 1.92 against 1.52 ms,
// R-MAT-26 10.4 against 8.4), then by the records' 10 bytes written.  R-MAT-20:
// part sizes and records in 0.12 ms against 0.36 with vertex chunks counted and
// dealt to waves, whose lanes stored straight to 32,768-key parts; R-MAT-22
// 0.53 against 0.90; R-MAT-24 1.9 against 2.7, and its parts are small enough
// to leave out a level.
template <typename OffT>
__global__ __launch_bounds__(kSplitBlock, 8) void k_split_l1(const GraphDesc *__restrict__ desc,
                                                          const SplitDesc *__restrict__ sd) {
    constexpr uint32_t kT = LevelTile<OffT>::kT, kPer = kT / kSplitBlock;
    constexpr uint32_t kWaves = kSplitBlock / kWave;
    // step 1's slots and step 3's staged pairs share their memory
    union SlotOrPair {
        struct {
            OffT rb, e;     // the row's bounds
            uint32_t near;  // its near ids (set where a far in-edge is in the tile)
        } v;
        TailPair<OffT> t;
    };
    __shared__ SlotOrPair s_x[kT];
    __shared__ uint64_t s_front;  // in-edges of the tile's first row before the tile
    __shared__ unsigned long long s_tally;
    __shared__ uint32_t s_open;  // the last row's far in-edges reach the tile's end
    __shared__ uint16_t s_mark[kT];
    __shared__ uint16_t s_key[kT];
    __shared__ uint8_t s_part[kT];
    __shared__ uint32_t s_cnt[kSplitPartsMax], s_off[kSplitPartsMax];
    __shared__ uint64_t s_base[kSplitPartsMax];
    __shared__ uint32_t s_w[kWaves];
    static_assert(kSplitPartsMax <= 256 && kT <= 65536, "8-bit parts, 16-bit slots");
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const OffT *__restrict__ rowPtr = static_cast<const OffT *>(D.rowPtr);
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const uint64_t *__restrict__ iep = S.ie_pre;
    uint16_t *__restrict__ rec_id = S.rec_id;
    TailPair<OffT> *__restrict__ rec = static_cast<TailPair<OffT> *>(S.rec);
    uint32_t *__restrict__ rec_aux = S.rec_aux;
    const uint32_t thr = D.thr, rows = S.rows, parts = S.parts, shift = S.part_shift;
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    const bool clip = S.clip != 0;
    const uint32_t v_lo = S.v_lo, v_hi = S.v_hi;
    if (v_lo > v_hi) return;  // nothing counted
    const uint64_t w_lo = S.w_lo, w_hi = S.w_hi;
    // the end vertices' rows, whose tails the range may clip
    const OffT rl0 = uni(rowPtr[v_lo]), rl1 = uni(rowPtr[(uint64_t)v_lo + 1]);
    const OffT rh0 = uni(rowPtr[v_hi]), rh1 = uni(rowPtr[(uint64_t)v_hi + 1]);
    const uint64_t K0 = uni64(iep[v_lo]), K1 = uni64(iep[(uint64_t)v_hi + 1]);
    const uint64_t tiles = (K1 - K0 + kT - 1) / kT;
    const uint32_t list_part = rows >> shift;  // the first part with list keys
    // the top ids below far_end are far
    const uint32_t far_ids = S.far_ids, far_end = uni32(D.n > kPackNear ? D.n - kPackNear : 0u);
    const uint32_t far_rows = far_end > thr ? far_end - thr : 0;
    uint64_t tops = 0;  // wedges of the top in-edges
    if (threadIdx.x == 0) s_tally = 0;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        uint64_t vb = uni32(S.tile_v[tile]);
        const uint64_t t0 = K0 + tile * kT, t1 = t0 + kT < K1 ? t0 + kT : K1;
        const uint32_t nt = (uint32_t)(t1 - t0);
        __syncthreads();  // the previous tile is written out
        for (uint32_t i = threadIdx.x; i < kT / 2; i += kSplitBlock) reinterpret_cast<uint32_t *>(s_mark)[i] = 0u;
        if (threadIdx.x < kSplitPartsMax) s_cnt[threadIdx.x] = 0u;
        if (threadIdx.x == 0) s_open = 0;
        __syncthreads();
        auto owner = [&](uint32_t at, OffT rb, OffT re) {  // of in-edge slot `at` and on
            s_mark[at] = (uint16_t)at;
            s_x[at].v.rb = rb;
            s_x[at].v.e = re;
            s_x[at].v.near = 0;
        };
        for (uint32_t win = 1;; win++) {  // windows of kSplitBlock vertices from vb, up to the one holding t1 - 1
            const uint64_t v = vb + threadIdx.x, vn = vb + kSplitBlock;
            const uint64_t next = vn > v_hi ? t1 : uni64(iep[vn]);
            if (v <= v_hi) {
                const uint64_t a = iep[v], z = iep[v + 1];
                const OffT rb = rowPtr[v], re = rowPtr[v + 1];
                if (z > a && z > t0 && a < t1) {
                    const uint32_t at = a > t0 ? (uint32_t)(a - t0) : 0u;
                    owner(at, rb, re);
                    if (at == 0) s_front = t0 - a;
                }
            }
            if (next >= t1) break;  // block-uniform
            vb = vn;
            if (win == kRowWindows) {  // block-uniform: the owners of the slots left
                const gptr<uint64_t> iepG = to_global(iep);
#pragma unroll 1
                for (uint32_t i = threadIdx.x; i < nt; i += kSplitBlock) {
                    if (t0 + i < next) continue;
                    const uint32_t r = rightmost_le(iepG, (uint32_t)vb, v_hi, t0 + i);
                    if (iepG[r] == t0 + i) owner(i, rowPtr[r], rowPtr[(uint64_t)r + 1]);
                }
                break;
            }
        }
        __syncthreads();
        // running maximum of the marks: kPer consecutive slots a thread
        {
            uint32_t x[kPer], mx = 0;
#pragma unroll
            for (uint32_t z = 0; z < kPer; z++) {
                const uint32_t y = s_mark[threadIdx.x * kPer + z];
                mx = y > mx ? y : mx;
                x[z] = mx;
            }
            uint32_t run = mx;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)run, o, kWave);
                run = (int)lane >= o && y > run ? y : run;
            }
            if (lane == kWave - 1) s_w[wv] = run;
            uint32_t before = (uint32_t)__shfl_up((int)run, 1, kWave);
            before = lane ? before : 0u;
            __syncthreads();
            for (uint32_t w = 0; w < wv; w++) before = s_w[w] > before ? s_w[w] : before;
#pragma unroll
            for (uint32_t z = 0; z < kPer; z++) s_mark[threadIdx.x * kPer + z] = (uint16_t)(x[z] > before ? x[z] : before);
        }
        __syncthreads();
        const OffT front = (OffT)uni64(s_front);
        auto position = [&](uint32_t i) -> OffT {  // of in-edge slot i in colInd
            const uint32_t p = s_mark[i];
            return s_x[p].v.rb + (OffT)(i - p) + (p ? 0 : front);
        };
        uint32_t id[kPer], nid[kPer];
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t i = threadIdx.x + u * kSplitBlock;
            id[u] = nid[u] = 0;
            if (i < nt) {
                const OffT j = position(i);
                id[u] = colInd[j];
                nid[u] = colInd[j + 1];  // an in-edge is not its row's last
            }
        }
        OffT rp[kPer], rp1[kPer];
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t i = threadIdx.x + u * kSplitBlock;
            rp[u] = rp1[u] = 0;
            if (i < nt && id[u] < thr) {
                rp[u] = rowPtr[id[u]];
                rp1[u] = rowPtr[(uint64_t)id[u] + 1];
            }
        }
        uint32_t key[kPer], aux[kPer];
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            key[u] = id[u] >= thr ? id[u] - thr : rows + (uint32_t)((uint64_t)rp[u] / kSlabSpan);
            const uint64_t len = (uint64_t)(rp1[u] - rp[u]);
            aux[u] = (uint32_t)((uint64_t)rp[u] % kSlabSpan) | ((len <= kSlabRowMax ? (uint32_t)len : kSlabAuxLong) << 13);
        }
        // a row's near ids are those after its last far one: where two
        // neighbours show it; of a row whose far in-edges reach the tile's
        // end, by a search
        if (far_rows) {  // block-uniform
#pragma unroll
            for (uint32_t u = 0; u < kPer; u++) {
                const uint32_t i = threadIdx.x + u * kSplitBlock;
                if (i >= nt || key[u] >= far_rows) continue;
                if (nid[u] >= far_end) s_x[s_mark[i]].v.near = (uint32_t)(s_x[s_mark[i]].v.e - position(i) - 1);
                else if (i == nt - 1) s_open = 1;
            }
            __syncthreads();
            if (s_open) {  // block-uniform
                if (wv == 0) {
                    const OffT re = s_x[s_mark[nt - 1]].v.e, at = position(nt - 1);
                    const uint32_t last = wave_rightmost_le((uint32_t)(re - at - 1), (uint64_t)far_end - 1,
                                                            [&](uint32_t x) { return (uint64_t)colInd[at + x]; });
                    if (lane == 0) s_x[s_mark[nt - 1]].v.near = (uint32_t)(re - at - 1 - last);
                }
                __syncthreads();
            }
        }
        uint32_t cut = 0;  // bit u: in-edge u is not wholly in the range
        if (clip) {
#pragma unroll 1
            for (uint32_t u = 0; u < kPer; u++) {
                const uint32_t i = threadIdx.x + u * kSplitBlock;
                if (i >= nt) continue;
                const OffT j = position(i), e = s_x[s_mark[i]].v.e;
                const bool in = j >= rl0 && j < rl1   ? whole_tail<OffT>(j, e, rl0, S.ws_full[v_lo], w_lo, w_hi)
                                : j >= rh0 && j < rh1 ? whole_tail<OffT>(j, e, rh0, S.ws_full[v_hi], w_lo, w_hi)
                                                      : true;
                cut |= in ? 0u : 1u << u;
            }
        }
        uint32_t rank[kPer];
        TailPair<OffT> t[kPer];
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t i = threadIdx.x + u * kSplitBlock;
            if (i >= nt || (cut >> u & 1u)) {
                key[u] = kSentinel;
                continue;
            }
            const uint32_t p = s_mark[i];
            const OffT j = position(i), e = s_x[p].v.e;
            const uint32_t tail = (uint32_t)(e - j - 1);
            if (key[u] < rows) {
                tops += tail;
                const uint32_t near = key[u] < far_rows ? s_x[p].v.near : tail;
                t[u].lo = pack_row<OffT>(s_x[p].v.rb, e);
                t[u].hi = pack_count((near + kPackNearIds - 1) / kPackNearIds, pack_div(tail - near + far_ids - 1, far_ids));
            } else {
                t[u] = TailPair<OffT>{j, e};
            }
            rank[u] = atomicAdd(&s_cnt[key[u] >> shift], 1u);
        }
        __syncthreads();  // s_x's rows are read, the counts are done
        uint64_t slot = 0;
        if (threadIdx.x < parts) {
            const uint32_t c = s_cnt[threadIdx.x];
            if (c)
                slot = S.part_base[threadIdx.x] +
                       atomicAdd(reinterpret_cast<unsigned long long *>(&S.part_cnt[threadIdx.x]), (unsigned long long)c);
        }
        if (wv == kWaves - 1) {  // another wave than the atomics'
            constexpr uint32_t kQ = kSplitPartsMax / kWave;
            uint32_t v[kQ], sum = 0;
#pragma unroll
            for (uint32_t z = 0; z < kQ; z++) {
                v[z] = s_cnt[lane * kQ + z];
                sum += v[z];
            }
            uint32_t run = sum;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)run, o, kWave);
                if ((int)lane >= o) run += y;
            }
            run -= sum;
#pragma unroll
            for (uint32_t z = 0; z < kQ; z++) {
                s_off[lane * kQ + z] = run;
                run += v[z];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < kPer; u++) {
            if (key[u] == kSentinel) continue;
            const uint32_t q = key[u] >> shift, at = s_off[q] + rank[u];
            rank[u] = at;
            s_x[at].t = t[u];
            s_key[at] = (uint16_t)(key[u] & ((1u << shift) - 1));
            s_part[at] = (uint8_t)q;
        }
        if (threadIdx.x < parts) s_base[threadIdx.x] = slot;
        __syncthreads();
        const uint32_t kept = s_off[kSplitPartsMax - 1] + s_cnt[kSplitPartsMax - 1];
        for (uint32_t i = threadIdx.x; i < kept; i += kSplitBlock) {
            const uint32_t q = s_part[i];
            const uint64_t p = s_base[q] + (i - s_off[q]);
            rec_id[p] = s_key[i];
            rec[p] = s_x[i].t;
        }
        const uint32_t lists = s_off[list_part];  // sorted by part: the list keys are at the end
        if (lists < kept) {  // block-uniform
            __syncthreads();
            uint32_t *s_aux = reinterpret_cast<uint32_t *>(s_x);
#pragma unroll
            for (uint32_t u = 0; u < kPer; u++)
                if (key[u] != kSentinel) s_aux[rank[u]] = aux[u];
            __syncthreads();
            for (uint32_t i = lists + threadIdx.x; i < kept; i += kSplitBlock) {
                const uint32_t q = s_part[i];
                if ((q << shift) + s_key[i] >= rows) rec_aux[s_base[q] + (i - s_off[q])] = s_aux[i];
            }
        }
    }
    tops = wave_sum(tops);
    __syncthreads();  // s_tally is zeroed, also without a tile
    if (lane == 0 && tops) atomicAdd(&s_tally, (unsigned long long)tops);
    __syncthreads();
    if (threadIdx.x == 0 && s_tally) atomicAdd(reinterpret_cast<unsigned long long *>(S.tally), s_tally);
}

// Later levels.  With up to kSplitPartsMax << kSplitFinalMax keys, a part
// has at most 1 << kSplitFinalMax keys and the final level groups its A
// records by key into ie.  With more, level 2 first groups each part's A
// records by sub-part of kSplitSub keys into B and the final level groups
// each sub-part's B records by key.
// A level's input bucket b holds the records [base[b], base[b] + cnt[b]) and
// is split into blocks of S.chunk records (its blocks start at cbase[b]); an
// output bucket is one of the kF sub-parts of a part, or one of the keys of
// the bucket.  k_split_level_count counts a block's records per output
// bucket into hist[c][0..kF); k_split_level_scatter (hist then holding, per
// output bucket, the records of the input bucket's earlier blocks) places
// each record at the next slot of its output bucket.  Blocks stride over the
// level's blocks.
constexpr int kLevelRecords = 4;  // records per thread per step, loads issued together
// Most blocks a level launches (they stride over its blocks of records).
constexpr uint32_t kLevelGridMax = 2048;

// The last b in [0, nb) with cbase[b] <= c (cbase[0] = 0 <= c).
__device__ __forceinline__ uint32_t bucket_of_block(const uint32_t *cbase, uint32_t nb, uint32_t c) {
    uint32_t lo = 0, hi = nb;  // cbase[lo] <= c < cbase[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (cbase[mid] <= c) lo = mid;
        else hi = mid;
    }
    return lo;
}

// What a level reads and writes.  KeyIn: 16-bit keys within a part (A) or
// 8-bit ones within a sub-part (B); kFinal: grouped by key, else by
// sub-part; kF output buckets (level 2: at most kSplitFan2).
template <typename KeyIn, bool kFinal, uint32_t kF>
struct SplitLevel {
    static constexpr bool kFromA = sizeof(KeyIn) == 2;
    const SplitDesc &S;
    __device__ __forceinline__ explicit SplitLevel(const SplitDesc &s) : S(s) {}
    __device__ __forceinline__ uint32_t buckets() const { return kFromA ? S.parts : S.subs; }
    __device__ __forceinline__ const uint64_t *base() const { return kFromA ? S.part_base : S.sub_base; }
    __device__ __forceinline__ uint64_t count(uint32_t b) const { return kFromA ? S.part_cnt[b] : S.sub_tot[b]; }
    __device__ __forceinline__ const uint32_t *cbase() const { return kFinal ? S.c3base : S.c2base; }
    __device__ __forceinline__ uint32_t *hist() const { return kFinal ? S.hist3 : S.hist2; }
    __device__ __forceinline__ const KeyIn *keys() const {
        return reinterpret_cast<const KeyIn *>(kFromA ? (const void *)S.rec_id : (const void *)S.rec_id2);
    }
    __device__ __forceinline__ const void *pairs() const { return kFromA ? S.rec : S.rec2; }
    __device__ __forceinline__ const uint32_t *aux() const { return kFromA ? S.rec_aux : S.rec_aux2; }
    // keys of an input bucket
    __device__ __forceinline__ uint32_t unit_shift() const { return kFromA ? S.part_shift : kSplitSubShift; }
    __device__ __forceinline__ uint32_t bucket(uint32_t key) const { return kFinal ? key : key >> kSplitSubShift; }
    // output buckets of an input bucket: kF of them in hist, `fan` in the tables
    __device__ __forceinline__ uint32_t fan() const { return kFinal ? kF : 1u << (S.part_shift - kSplitSubShift); }
};

template <typename KeyIn, bool kFinal, uint32_t kF>
__global__ __launch_bounds__(kSplitBlock) void k_split_level_count(const SplitDesc *__restrict__ sd) {
    __shared__ uint32_t s_cnt[kF];
    const SplitLevel<KeyIn, kFinal, kF> L(sd[0]);
    const uint32_t nb = L.buckets(), chunk = L.S.chunk;
    const uint64_t *__restrict__ base_in = L.base();
    const uint32_t *__restrict__ cbase = L.cbase();
    const KeyIn *__restrict__ key_in = L.keys();
    const uint32_t nblk = cbase[nb];
    for (uint32_t c = blockIdx.x; c < nblk; c += gridDim.x) {
        const uint32_t b = bucket_of_block(cbase, nb, c);
        const uint64_t k0 = base_in[b] + (uint64_t)(c - cbase[b]) * chunk;
        const uint64_t kq = base_in[b] + L.count(b), k1 = k0 + chunk < kq ? k0 + chunk : kq;
        __syncthreads();  // the previous block's LDS reads are done
        for (uint32_t i = threadIdx.x; i < kF; i += kSplitBlock) s_cnt[i] = 0u;
        __syncthreads();
        constexpr int kU = kLevelRecords;
        for (uint64_t kb = k0 + threadIdx.x; kb < k1; kb += (uint64_t)kU * kSplitBlock) {
            uint32_t key[kU];
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const uint64_t k = kb + (uint64_t)u * kSplitBlock;
                key[u] = k < k1 ? key_in[k] : kSentinel;
            }
#pragma unroll
            for (int u = 0; u < kU; u++)
                if (key[u] != kSentinel) atomicAdd(&s_cnt[L.bucket(key[u])], 1u);
        }
        __syncthreads();
        uint32_t *__restrict__ h = L.hist() + (uint64_t)c * kF;
        for (uint32_t i = threadIdx.x; i < kF; i += kSplitBlock) h[i] = s_cnt[i];
    }
}

// Records of a scatter's tile: twice LevelTile's (one block a CU by LDS) where
// a bucket gets four or fewer of a tile.  Writes of less than 64 bytes pass L2
// one by one, some 54 a nanosecond, and bound the kernel: R-MAT-24 (2,048
// buckets) 2.02 -> 1.74 ms with tiles of 8,192, R-MAT-22 (1,024) 0.42 -> 0.35,
// R-MAT-20 (512) 0.068 either way.
template <typename OffT, uint32_t kF>
struct ScatterTile {
    static constexpr bool kTwo = kF < 1024;  // two blocks a CU
    static constexpr uint32_t kT = LevelTile<OffT>::kT * (kTwo ? 1 : 2);
};

// The scatter of a level.  hist[c] holds, per output bucket, the input
// bucket's records in blocks before c.  The block takes its records in tiles
// of kT: each tile is ranked per output bucket (LDS atomics), staged in LDS
// sorted by output bucket, and written out in that order, so that the
// records of one output bucket in a tile -- kT / kF of them on average --
// leave as consecutive lanes of one store to consecutive addresses.  The
// list records' slab words go through the same LDS after the pairs, in
// buckets that hold list keys only.
template <typename OffT, typename KeyIn, bool kFinal, uint32_t kF>
__global__ __launch_bounds__(kSplitBlock, (ScatterTile<OffT, kF>::kTwo ? 8 : 4)) void k_split_level_scatter(
    const SplitDesc *__restrict__ sd) {
    constexpr uint32_t kT = ScatterTile<OffT, kF>::kT;
    constexpr uint32_t kPerThread = kT / kSplitBlock;
    __shared__ uint64_t s_base[kF];  // next output slot of each output bucket
    __shared__ uint32_t s_tcnt[kF];  // the tile's records per output bucket
    __shared__ uint32_t s_toff[kF];  // their exclusive prefix: each bucket's first staged slot
    __shared__ uint32_t s_w[kSplitBlock / kWave];
    __shared__ uint16_t st_key[kT];
    __shared__ TailPair<OffT> st_rec[kT];
    const SplitLevel<KeyIn, kFinal, kF> L(sd[0]);
    const SplitDesc &S = L.S;
    const uint32_t rows = S.rows, keys = S.keys, nb = L.buckets(), chunk = S.chunk, fan = L.fan();
    const uint64_t *__restrict__ base_in = L.base();
    const uint32_t *__restrict__ cbase = L.cbase();
    const uint32_t *__restrict__ hist = L.hist();
    const KeyIn *__restrict__ key_in = L.keys();
    const TailPair<OffT> *__restrict__ rec_in = static_cast<const TailPair<OffT> *>(L.pairs());
    const uint32_t *__restrict__ aux_in = L.aux();
    uint8_t *__restrict__ key_out = S.rec_id2;  // level 2 only
    TailPair<OffT> *__restrict__ rec_out = static_cast<TailPair<OffT> *>(kFinal ? S.ie : S.rec2);
    uint32_t *__restrict__ aux_out = kFinal ? S.ie_aux : S.rec_aux2;
    const OffT *__restrict__ rp_in = static_cast<const OffT *>(S.rp_in);
    const uint32_t nblk = cbase[nb];
    for (uint32_t c = blockIdx.x; c < nblk; c += gridDim.x) {
        const uint32_t b = bucket_of_block(cbase, nb, c);
        const uint64_t k0 = base_in[b] + (uint64_t)(c - cbase[b]) * chunk;
        const uint64_t kq = base_in[b] + L.count(b), k1 = k0 + chunk < kq ? k0 + chunk : kq;
        const uint32_t first_key = b << L.unit_shift();
        const bool lists = (uint64_t)first_key + (1u << L.unit_shift()) > rows;  // block-uniform
        const uint32_t *__restrict__ h = hist + (uint64_t)c * kF;
        __syncthreads();  // the previous block's LDS reads are done
        for (uint32_t i = threadIdx.x; i < kF; i += kSplitBlock) {
            // first slot of output bucket i: a sub-part's first record, or a key's first in-edge
            uint64_t ob = 0;
            if (kFinal) ob = first_key + i < keys ? (uint64_t)rp_in[first_key + i] : 0;
            else if (i < fan) ob = S.sub_base[b * fan + i];
            s_base[i] = ob + h[i];
        }
        for (uint64_t t0 = k0; t0 < k1; t0 += kT) {  // block-uniform
            for (uint32_t i = threadIdx.x; i < kF; i += kSplitBlock) s_tcnt[i] = 0u;
            __syncthreads();
            uint32_t key[kPerThread], rank[kPerThread], aux[kPerThread];
            TailPair<OffT> t[kPerThread];
#pragma unroll
            for (uint32_t u = 0; u < kPerThread; u++) {
                const uint64_t k = t0 + threadIdx.x + (uint64_t)u * kSplitBlock;
                key[u] = k < k1 ? key_in[k] : kSentinel;
                aux[u] = 0u;
                if (key[u] != kSentinel) {
                    t[u] = rec_in[k];
                    if (lists && first_key + key[u] >= rows) aux[u] = aux_in[k];  // a list record
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kPerThread; u++)
                if (key[u] != kSentinel) rank[u] = atomicAdd(&s_tcnt[L.bucket(key[u])], 1u);
            __syncthreads();
            block_prefix<kF>(s_tcnt, s_toff, s_w);
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < kPerThread; u++) {
                if (key[u] == kSentinel) continue;
                const uint32_t at = s_toff[L.bucket(key[u])] + rank[u];
                rank[u] = at;
                st_key[at] = (uint16_t)key[u];
                st_rec[at] = t[u];
            }
            __syncthreads();
            const uint32_t nt = (uint32_t)(k1 - t0 < kT ? k1 - t0 : kT);
#pragma unroll
            for (uint32_t u = 0; u < kPerThread; u++) {
                const uint32_t i = threadIdx.x + u * kSplitBlock;
                if (i >= nt) continue;
                const uint32_t k = st_key[i], q = L.bucket(k);  // the key within the input bucket
                const uint64_t p = s_base[q] + (i - s_toff[q]);
                if (!kFinal) key_out[p] = (uint8_t)(k & (kSplitSub - 1));
                rec_out[p] = st_rec[i];
            }
            __syncthreads();
            if (lists) {
                uint32_t *st_aux = reinterpret_cast<uint32_t *>(st_rec);
#pragma unroll
                for (uint32_t u = 0; u < kPerThread; u++)
                    if (key[u] != kSentinel) st_aux[rank[u]] = aux[u];
                __syncthreads();
#pragma unroll
                for (uint32_t u = 0; u < kPerThread; u++) {
                    const uint32_t i = threadIdx.x + u * kSplitBlock;
                    if (i >= nt) continue;
                    const uint32_t k = st_key[i], q = L.bucket(k);
                    if (first_key + k >= rows) aux_out[s_base[q] + (i - s_toff[q])] = st_aux[i];
                }
                __syncthreads();
            }
            for (uint32_t i = threadIdx.x; i < kF; i += kSplitBlock) s_base[i] += s_tcnt[i];
        }
    }
}

// Thread per key o of the final level: the column prefix of hist3 over its
// input bucket's blocks (hist3[c][i] becomes the key's records in the
// bucket's earlier blocks) and the key's total into key_tot.
__global__ __launch_bounds__(kBlock) void k_split_levelcols3(const SplitDesc *__restrict__ sd) {
    const SplitDesc &S = sd[0];
    const uint32_t o = blockIdx.x * kBlock + threadIdx.x;
    if (o >= S.keys) return;
    const uint32_t sh = S.final_shift, b = o >> sh, i = o & ((1u << sh) - 1);
    const uint32_t *__restrict__ cbase = S.c3base;
    uint32_t *__restrict__ hist = S.hist3;
    uint32_t s = 0;
    const uint32_t c1 = cbase[b + 1];
    for (uint32_t c = cbase[b]; c < c1; c += 8) {  // eight loads in flight
        uint32_t x[8];
#pragma unroll
        for (uint32_t z = 0; z < 8; z++) x[z] = c + z < c1 ? hist[((uint64_t)(c + z) << sh) + i] : 0u;
#pragma unroll
        for (uint32_t z = 0; z < 8; z++) {
            if (c + z < c1) hist[((uint64_t)(c + z) << sh) + i] = s;
            s += x[z];
        }
    }
    S.key_tot[o] = s;
}

// The second level's column prefixes, one block per part: the part's blocks
// are cut into kSplitBlock / kSplitFan2 segments whose column sums are taken
// in parallel first (a part spans hundreds of blocks).
__global__ __launch_bounds__(kSplitBlock) void k_split_levelcols2(const SplitDesc *__restrict__ sd) {
    constexpr uint32_t kF = kSplitFan2, kSeg = kSplitBlock / kF;
    __shared__ uint32_t s_sum[kSeg][kF];
    const SplitDesc &S = sd[0];
    const uint32_t b = blockIdx.x, i = threadIdx.x % kF, sg = threadIdx.x / kF;
    const uint32_t fan = 1u << (S.part_shift - kSplitSubShift);
    const uint32_t cb0 = S.c2base[b], nb = S.c2base[b + 1] - cb0;
    const uint32_t per = (nb + kSeg - 1) / kSeg;
    const uint32_t s0 = cb0 + (sg * per < nb ? sg * per : nb), s1 = cb0 + ((sg + 1) * per < nb ? (sg + 1) * per : nb);
    uint32_t *__restrict__ hist = S.hist2;
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t c = s0; c < s1; c++) sum += hist[(uint64_t)c * kF + i];
    s_sum[sg][i] = sum;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (uint32_t z = 0; z < kSeg; z++) {
        const uint32_t x = s_sum[z][i];
        pre += z < sg ? x : 0u;
        tot += x;
    }
#pragma unroll 8
    for (uint32_t c = s0; c < s1; c++) {
        const uint32_t x = hist[(uint64_t)c * kF + i];
        hist[(uint64_t)c * kF + i] = pre;
        pre += x;
    }
    if (sg == 0 && i < fan) S.sub_tot[b * fan + i] = tot;
}

// One block: the blocks of a level's input buckets, c2base or c3base as the
// prefix of ceil(count / chunk); with the sub-parts also sub_base, the
// prefix of their totals (in key order).
template <bool kSubs>
__global__ __launch_bounds__(kSplitBlock) void k_split_bases(const SplitDesc *__restrict__ sd) {
    constexpr int kWaves = kSplitBlock / kWave;
    __shared__ uint64_t s_r[kWaves], s_b[kWaves];
    const SplitDesc &S = sd[0];
    const uint32_t nb = kSubs ? S.subs : S.parts, chunk = S.chunk;
    uint32_t *__restrict__ cbase = kSubs || S.part_shift == S.final_shift ? S.c3base : S.c2base;
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x >> 6;
    uint64_t cr = 0, cb = 0;
    for (uint32_t base = 0; base < nb; base += kSplitBlock) {
        const uint32_t i = base + threadIdx.x;
        const uint64_t x = i < nb ? (kSubs ? (uint64_t)S.sub_tot[i] : S.part_cnt[i]) : 0;
        const uint64_t y = (x + chunk - 1) / chunk;
        const uint64_t ix = wave_incl_scan(x), iy = wave_incl_scan(y);
        if (lane == kWave - 1) {
            s_r[wv] = ix;
            s_b[wv] = iy;
        }
        __syncthreads();
        uint64_t ox = 0, oy = 0, ax = 0, ay = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            ox += w < (int)wv ? s_r[w] : 0;
            oy += w < (int)wv ? s_b[w] : 0;
            ax += s_r[w];
            ay += s_b[w];
        }
        __syncthreads();
        if (i < nb) {
            if (kSubs) S.sub_base[i] = cr + ox + ix - x;
            cbase[i] = (uint32_t)(cb + oy + iy - y);
        }
        cr += ax;
        cb += ay;
    }
    if (threadIdx.x == 0) cbase[nb] = (uint32_t)cb;
}

// Block b: the in-edges of keys [b*kKeyChunk, (b+1)*kKeyChunk) into
// key_part[b].
__global__ __launch_bounds__(kSplitBlock) void k_split_keysum(const SplitDesc *__restrict__ sd) {
    __shared__ uint64_t s_w[kSplitBlock / kWave];
    const SplitDesc &S = sd[0];
    const uint64_t i0 = (uint64_t)blockIdx.x * kKeyChunk + 4ull * threadIdx.x;
    uint64_t x = 0;
#pragma unroll
    for (uint32_t z = 0; z < 4; z++)
        if (i0 + z < S.keys) x += S.key_tot[i0 + z];
    x = wave_sum(x);
    if ((threadIdx.x & (kWave - 1)) == 0) s_w[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        for (int w = 0; w < kSplitBlock / kWave; w++) t += s_w[w];
        S.key_part[blockIdx.x] = t;
    }
}

// Block b (key_part then holding the exclusive prefix of the key blocks):
// rp_in of its keys; the block of key `rows` puts the top rows' in-edges
// into meta, the last block rp_in[keys] and the rest of meta (the wedges of
// the two kernels, what the dense part took, the counted wedges and all
// in-edges).
template <typename OffT>
__global__ __launch_bounds__(kSplitBlock) void k_split_keyscan(const SplitDesc *__restrict__ sd,
                                                               const DenseDesc *__restrict__ dd,
                                                               uint64_t *__restrict__ meta) {
    __shared__ uint64_t s_w[kSplitBlock / kWave];
    const SplitDesc &S = sd[0];
    const uint64_t *__restrict__ dense = dd->sums;  // the dense in-edges and wedges are in the totals
    const uint32_t keys = S.keys, rows = S.rows;
    OffT *__restrict__ rp = static_cast<OffT *>(S.rp_in);
    const uint64_t i0 = (uint64_t)blockIdx.x * kKeyChunk + 4ull * threadIdx.x;
    uint32_t v[4];
    uint64_t x = 0;
#pragma unroll
    for (uint32_t z = 0; z < 4; z++) {
        v[z] = i0 + z < keys ? S.key_tot[i0 + z] : 0u;
        x += v[z];
    }
    uint64_t tot;
    uint64_t at = S.key_part[blockIdx.x] + split_block_scan(x, s_w, tot);
#pragma unroll
    for (uint32_t z = 0; z < 4; z++) {
        if (i0 + z < keys) rp[i0 + z] = (OffT)at;
        if (i0 + z == rows) meta[kMetaInEdges] = at + dense[kDenseTopEdges] + S.cut_top;
        at += v[z];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        const uint64_t all = S.key_part[blockIdx.x] + tot;
        rp[keys] = (OffT)all;
        if (rows >= keys) meta[kMetaInEdges] = all + dense[kDenseTopEdges] + S.cut_top;
        meta[kMetaTopWedges] = S.tally[0] + dense[kDenseTopWedges];
        meta[kMetaDenseTopWedges] = dense[kDenseTopWedges];
        meta[kMetaDenseTopEdges] = dense[kDenseTopEdges];
        meta[kMetaListWedges] = S.w_hi - S.w_lo - S.tally[0] - dense[kDenseTopWedges];
        meta[kMetaWedges] = S.w_hi - S.w_lo;
        meta[kMetaAllEdges] = all + dense[kDenseEdges] + S.cuts;
    }
}

// ------------------------------------------------------------- top-a part

// The top rows' tails as packed ids.  A top in-edge v -> w (w >= thr) has a
// tail of ids above w, which is a prefix of row v from the top; x = n - u of
// each is below rows (the a-bit row must fit a block's LDS, so rows <= 2^21).
// Each counted row's tail ids (all but its lowest) are packed as 16-byte
// chunks: kPackNearIds near ids to a chunk, then P far ones in fields of the
// fewest bits B that the graph's rows allow, and the end of a row's last near
// and last far chunk with 0.  So the row kernel streams 2 or 16/P bytes per
// tail id instead of 4, long rows by whole lines, and every field of a tail's
// chunks can be looked up in the bitmap of adj+(w) with nothing masked off: a
// chunk's ids past the tail are at most w, adj+(w) holds ids above w only,
// and no id has x = 0.
// The row kernel is bound by the 128-byte lines that it misses L2 for (every
// one of them: 7.0 TB/s on R-MAT-24).  With rows in colInd's order, 7 ids a
// chunk cut at fixed positions and the ends masked, a tail of R-MAT-24 touched
// 3.3 lines and a lookup took 10.4 vector instructions; now 2.7 and 6.7.  Row
// kernel 10.3 -> 8.4 ms there, 59.9 -> 48.2 on R-MAT-26; packing 0.39 -> 0.73
// and 1.6 -> 2.6 (R-MAT-24 0.64 with eight waves a SIMD).
// Layouts of the far chunks (PackLayout<L>):
//   0: P = 6, B = 21, rows <= 2^19, field (x >> 5) << 7 | (x & 31): bits
//      [5, 21) are the LDS byte address of x's bitmap word and bits [0, 5)
//      its bit, so that the row kernel takes both with one extract;
//   1: P = 6, B = 21, rows <= 2^21, field x;
//   2: P = 7, B = 18, rows <= 2^18, field x;
//   3: near chunks only, rows <= kPackNear (P = 8, B = 16: the near fields).
template <int L>
struct PackLayout;
template <>
struct PackLayout<0> {
    static constexpr int P = 6, B = 21;
    static constexpr bool kAddr = true;
};
template <>
struct PackLayout<1> {
    static constexpr int P = 6, B = 21;
    static constexpr bool kAddr = false;
};
template <>
struct PackLayout<2> {
    static constexpr int P = 7, B = 18;
    static constexpr bool kAddr = false;
};
template <>
struct PackLayout<3> {
    static constexpr int P = 8, B = 16;
    static constexpr bool kAddr = false;
};
constexpr uint32_t kPackRowsMax = 1u << 21;
constexpr uint32_t kPackTile = 8192, kPackTileMin = 2048;  // slots a block packs at a time
constexpr uint32_t kPackGrid = 2048;  // blocks of the packing kernel (eight a CU)

// The layout of a graph with `rows` top rows (rows <= kPackRowsMax).
__host__ __device__ __forceinline__ int pack_layout(uint32_t rows) {
    return rows <= kPackNear ? 3 : rows <= (1u << 18) ? 2 : rows <= (1u << 19) ? 0 : 1;
}

// Field i of a chunk, shifted down so that its bits start at bit 0 (bits
// above B hold the next field's; the readers extract what they need).
template <int B, int i>
__device__ __forceinline__ uint32_t chunk_field(u32x4 d) {
    constexpr int bit = B * i, k = bit / 32, sh = bit % 32;
    if constexpr (sh + B <= 32) {
        return d[k] >> sh;
    } else {
        return __builtin_amdgcn_alignbit(d[k + 1], d[k], sh);
    }
}

template <int B, int... I>
__device__ __forceinline__ void chunk_fields(u32x4 d, uint32_t *f, std::integer_sequence<int, I...>) {
    ((f[I] = chunk_field<B, I>(d)), ...);
}

// The chunk of the cnt (1 to P) ids that end at position end of colInd, from
// the last one down.
template <int L>
__device__ __forceinline__ u32x4 pack_chunk(gptr<uint32_t> colInd, uint64_t end, uint32_t cnt, uint32_t n,
                                            uint32_t thr) {
    using PL = PackLayout<L>;
    constexpr int P = PL::P, B = PL::B;
    typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));
    uint32_t id[8];
    if (end >= 8) {
        const u32x4u x = *reinterpret_cast<gptr<u32x4u>>(colInd + (end - 4));
        const u32x4u y = *reinterpret_cast<gptr<u32x4u>>(colInd + (end - 8));
#pragma unroll
        for (int z = 0; z < 8; z++) id[z] = z < 4 ? x[3 - z] : y[7 - z];
    } else {
#pragma unroll
        for (int z = 0; z < 8; z++) id[z] = (uint32_t)z < cnt ? colInd[end - 1 - z] : 0u;
    }
    uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int z = 0; z < P; z++) {
        const uint32_t x = (uint32_t)z < cnt && id[z] > thr ? n - id[z] : 0u;  // below rows
        const uint32_t f = PL::kAddr ? ((x >> 5) << 7) | (x & 31u) : x;
        const int bit = B * z, k = bit / 32, sh = bit % 32;
        d[k] |= f << sh;
        if (sh + B > 32) d[k + 1] |= f >> (32 - sh);
    }
    return u32x4{d[0], d[1], d[2], d[3]};
}

// Packs the counted rows into S.packed (the memory of the final level's
// input pairs and slab words).  Blocks take tiles of chunk slots in
// turn, and the rows with slots in the tile kBlock at a time: a thread finds
// its row's near ids by a binary search and with them its chunks in the tile,
// whose prefix over the block deals them out; a thread finds a chunk's row in
// the prefix, loads the ids by two 16-byte loads of any alignment and packs
// them.  Chunks of ids up to thr only are left unwritten: no tail holds them.
template <typename OffT>
__global__ __launch_bounds__(kBlock, 8) void k_split_pack(const GraphDesc *__restrict__ desc,
                                                       const SplitDesc *__restrict__ sd) {
    __shared__ OffT s_re[kBlock], s_at[kBlock];  // a row's end; slot of its chunk 0 less the prefix
    __shared__ uint32_t s_tail[kBlock], s_near[kBlock], s_pre[kBlock], s_skip[kBlock];
    __shared__ uint32_t s_w[kWavesPerBlock];
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const gptr<OffT> rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
    const gptr<uint32_t> colInd = to_global(D.colInd);
    u32x4 *__restrict__ dst = static_cast<u32x4 *>(S.packed);
    const uint32_t v_lo = S.v_lo, v_hi = S.v_hi, n = D.n, thr = D.thr, P = S.far_ids;
    if (v_lo > v_hi) return;  // nothing counted
    const uint32_t near_end = n > kPackNear ? n - kPackNear : 0;  // ids from here on are near
    const int layout = pack_layout(S.rows);
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x >> 6;
    const uint64_t p1 = rowPtr[(uint64_t)v_hi + 1];
    const uint64_t c0 = pack_slot((uint64_t)rowPtr[v_lo]), c1 = pack_slot(p1);
    // two tiles a block, of kPackTileMin to kPackTile slots (R-MAT-20 43 us; with
    // 8,192 slots each, for which there are fewer tiles than blocks, 79)
    uint64_t slots = (c1 - c0) / (2ull * gridDim.x);
    slots = slots < kPackTileMin ? kPackTileMin : slots > kPackTile ? kPackTile : slots;
    const uint64_t tiles = (c1 - c0 + slots - 1) / slots;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint64_t s0 = c0 + tile * slots, s1 = s0 + slots < c1 ? s0 + slots : c1;
        uint64_t vb = v_lo + wave_rightmost_le(v_hi - v_lo, s0, [&](uint32_t x) { return pack_slot((uint64_t)rowPtr[(uint64_t)v_lo + x]); });
        uint32_t win = 0;
        uint64_t pos = 0;  // the first position of a window by positions, or 0
        for (;;) {  // windows of kBlock vertices from vb
            uint64_t v = vb + threadIdx.x, vn = vb + kBlock;
            const bool by_pos = pos != 0;  // block-uniform
            if (by_pos) {  // the rows that start at one of kBlock positions
                const uint64_t q = pos + threadIdx.x;
                v = (uint64_t)v_hi + 1;
                if (q < p1) {
                    const uint32_t r = rightmost_le(rowPtr, (uint32_t)vb, v_hi, q);
                    if ((uint64_t)rowPtr[r] == q) v = r;
                }
                pos += kBlock;
                // the row after those that start before pos
                vn = pos >= p1 ? (uint64_t)v_hi + 1
                               : vb + 1 + wave_rightmost_le((uint32_t)(v_hi - vb), pos - 1, [&](uint32_t r) { return (uint64_t)rowPtr[vb + r]; });
                pos = 0;
            }
            const uint64_t next = rowPtr[vn <= v_hi ? vn : (uint64_t)v_hi + 1];
            const bool more = vn <= v_hi && pack_slot(next) < s1;
            uint32_t cnt = 0, near = 0, tail = 0, skip = 0;
            OffT re = 0, c = 0;
            if (v <= v_hi) {
                const OffT rb = rowPtr[v];
                re = rowPtr[v + 1];
                c = pack_row<OffT>(rb, re);
                if (re - rb >= 2 && c < s1 && pack_slot(re) > s0 && colInd[re - 1] > thr) {
                    tail = (uint32_t)(re - rb - 1);
                    OffT lo = rb + 1, hi = re;  // the first near one of the tail ids (without far ones: any)
                    while (layout != 3 && lo < hi) {
                        const OffT mid = lo + ((hi - lo) >> 1);
                        if (colInd[mid] < near_end) lo = mid + 1;
                        else hi = mid;
                    }
                    near = (uint32_t)(re - lo);
                    const uint32_t far = layout == 3 ? 0u : pack_div(tail - near + P - 1, P);
                    const uint64_t z = (uint64_t)c + (near + kPackNearIds - 1) / kPackNearIds + far;
                    skip = c < s0 ? (uint32_t)(s0 - c) : 0u;
                    const uint64_t e = z < s1 ? z : s1;
                    cnt = e > c + skip ? (uint32_t)(e - c - skip) : 0u;
                }
            }
            uint32_t incl = cnt;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)incl, o, kWave);
                incl += (int)lane >= o ? y : 0u;
            }
            if (lane == kWave - 1) s_w[wv] = incl;
            __syncthreads();  // also: the previous window is packed
            uint32_t before = 0, total = 0;
#pragma unroll
            for (uint32_t w = 0; w < (uint32_t)kWavesPerBlock; w++) {
                before += w < wv ? s_w[w] : 0u;
                total += s_w[w];
            }
            s_pre[threadIdx.x] = before + incl - cnt;
            s_skip[threadIdx.x] = skip;
            s_near[threadIdx.x] = near;
            s_tail[threadIdx.x] = tail;
            s_re[threadIdx.x] = re;
            s_at[threadIdx.x] = c;
            __syncthreads();
            for (uint32_t t = threadIdx.x; t < total; t += kBlock) {
                uint32_t r = 0;  // the last row with s_pre[r] <= t
#pragma unroll
                for (uint32_t o = kBlock / 2; o > 0; o >>= 1) r += s_pre[r + o] <= t ? o : 0u;
                const uint32_t q = t - s_pre[r] + s_skip[r], near_r = s_near[r], tail_r = s_tail[r];
                const uint32_t qn = (near_r + kPackNearIds - 1) / kPackNearIds;
                const bool is_near = q < qn;
                const uint32_t first = is_near ? kPackNearIds * q : near_r + P * (q - qn);
                const uint32_t left = (is_near ? near_r : tail_r) - first;
                const uint64_t end = (uint64_t)s_re[r] - first;
                if (colInd[end - 1] <= thr) continue;
                const uint64_t at = (uint64_t)s_at[r] + q;
                if (is_near) dst[at] = pack_chunk<3>(colInd, end, left < kPackNearIds ? left : kPackNearIds, n, thr);
                else if (layout == 2) dst[at] = pack_chunk<2>(colInd, end, left < P ? left : P, n, thr);
                else if (layout == 0) dst[at] = pack_chunk<0>(colInd, end, left < P ? left : P, n, thr);
                else dst[at] = pack_chunk<1>(colInd, end, left < P ? left : P, n, thr);
            }
            if (!more) break;  // block-uniform
            vb = vn;
            if (by_pos || ++win % kRowWindows == 0) {  // few positions in as many windows more: by these
                const uint64_t far = vn + kRowWindows * kBlock;
                if (far <= v_hi && uni64(rowPtr[far] - next) < 2 * kBlock) pos = uni64(next);
            }
            __syncthreads();  // s_w is read
        }
        __syncthreads();
    }
}

// Lanes per in-edge tail in the row kernel (a wave takes kWave / kSplitLanes
// in-edges per step), a 16-byte chunk per lane: eight take a line at a time
// (four: R-MAT-19 to 22 0 to 2% less, a quarter of R-MAT-21's wedges 2% and
// R-MAT-26 1% more).
constexpr int kSplitLanes = 8;

// The hits of the P packed ids of a chunk.  Every field names a bit of the
// row bitmap (word and bit straight from the fields: a field's bit offset is
// its low 5 bits), and those outside the tail name bits that are not set.  An
// address field's bits [5, 21) are the byte offset of its word in the bitmap.
template <int L>
__device__ __forceinline__ uint32_t rows_chunk_hits(const uint32_t *s_bits, u32x4 ch) {
    using PL = PackLayout<L>;
    constexpr int P = PL::P, B = PL::B;
    uint32_t f[P];
    chunk_fields<B>(ch, f, std::make_integer_sequence<int, P>{});
    uint32_t wrd[P];
#pragma unroll
    for (int z = 0; z < P; z++) {
        const uint32_t addr = PL::kAddr ? __builtin_amdgcn_ubfe(f[z], 5u, 16u) : (f[z] >> 3) & (((1u << (B - 5)) - 1) << 2);
        wrd[z] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(s_bits) + addr);
    }
    uint32_t h = 0;
#pragma unroll
    for (int z = 0; z < P; z++) h += __builtin_amdgcn_ubfe(wrd[z], f[z], 1u);
    return h;
}

// The hits of a tail's `chunks` chunks from `at` on (each lane's own first
// one), kLanes lanes to a tail, this one's number sl.
template <int L, int kLanes>
__device__ __forceinline__ uint32_t rows_tail_hits(const uint32_t *s_bits, gptr<u32x4> at, uint32_t chunks, uint32_t sl) {
    if (chunks <= sl) return 0;
    uint32_t left = (chunks - sl + kLanes - 1) / kLanes, h = 0;  // the lane's chunks
    u32x4 a = at[0], b;
    for (;;) {  // two chunks a turn, each loaded before the one before is counted
        if (left > 1) b = at[kLanes];
        h += rows_chunk_hits<L>(s_bits, a);
        if (left <= 1) break;
        if (left > 2) a = at[2 * kLanes];
        h += rows_chunk_hits<L>(s_bits, b);
        if (left <= 2) break;
        left -= 2;
        at += 2 * kLanes;
    }
    return h;
}

// Persistent blocks take tiles of the rows' work from one counter, or short
// ones from sixteen.  The work
// of a row is kSplitRowCost for its bitmap and one unit per in-edge, so a
// tile is up to `tile` in-edges of few rows, or fewer in-edges where rows
// have few each: tiles of in-edges alone left blocks with hundreds of such
// rows to the end, one chain of loads and barriers after another (a quarter
// of R-MAT-21's wedges: 1.75 ms).
// Per row of a tile the block puts adj+(w) into an LDS bitmap as bits n -
// u, its waves take the row's in-edges in the tile (kLanes lanes each),
// and each tail is streamed through the bitmap from the packed ids
// (k_split_pack) by 16-byte chunks of 6 to 8 ids, the next
// chunk loaded before this one is counted, and the next in-edges' bounds
// before these are streamed.  A row's ids are loaded while the row before is
// streamed; its bits go in as the other row's go out, all by exclusive or,
// so a row takes two barriers.  With 4-byte offsets held to 64 registers (it
// takes 65 by itself), for eight waves a SIMD.
template <typename OffT, int kWaves, int kLanes, int kLayout>
__global__ __launch_bounds__(kWave * kWaves, (sizeof(OffT) == 4 ? 8 : 7)) void k_split_rows(const GraphDesc *__restrict__ desc,
                                                               const SplitDesc *__restrict__ sd,
                                                               uint64_t *__restrict__ lines) {
    // dynamic LDS only: the row bitmap, then the tile slot
    extern __shared__ uint32_t s_bits[];
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const gptr<OffT> rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const gptr<u32x4> packed = to_global(static_cast<const u32x4 *>(S.packed));
    const gptr<OffT> rp_in = to_global(static_cast<const OffT *>(S.rp_in));
    const gptr<OffT> ieG = to_global(static_cast<const OffT *>(S.ie));
    const uint32_t n = D.n, thr = D.thr, rows = S.rows;
    constexpr uint32_t kThreads = kWave * kWaves;
    constexpr uint32_t kPer = kWave / kLanes;  // in-edges a wave takes per step
    constexpr uint32_t kHold = 2;              // ids of a row a thread keeps
    const uint32_t words = (rows + 31) >> 5;
    uint64_t &s_tile = *reinterpret_cast<uint64_t *>(s_bits + ((words + 1) & ~1u));
    for (uint32_t i = threadIdx.x; i < words; i += kThreads) s_bits[i] = 0;
    const uint64_t K = uni((uint64_t)rp_in[rows]), work = K + (uint64_t)kSplitRowCost * rows;
    // about eight tiles a block, of kSplitTileMinWork to kSplitTile
    uint64_t tile = work / (8ull * gridDim.x);
    tile = tile < kSplitTileMinWork ? kSplitTileMinWork : tile > kSplitTile ? kSplitTile : tile;
    // short tiles come from sixteen counters (with one, R-MAT-20 0.45 ms instead
    // of 0.26); full ones, 20 ns apart at the least, from one, which keeps those
    // in flight closest (R-MAT-24 8.3 ms, two counters 8.6, eight 8.9)
    const uint32_t of = tile < kSplitTile ? kTileLines : 1u;
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    const uint32_t sub = lane / kLanes, sl = lane % kLanes;
    uint64_t hits = 0;
    // the tails that the ends of a range cut: searched by one block
    if (blockIdx.x == 0) {
        for (uint32_t z = 0; z < S.cuts; z++) {
            const uint32_t w = colInd[S.cut_j[z]];
            const OffT wb = rowPtr[w], we = rowPtr[(uint64_t)w + 1];
            for (uint64_t q = S.cut_lo[z] + threadIdx.x; q < S.cut_hi[z]; q += kThreads) {
                const uint32_t u = colInd[q];
                OffT lb = wb, n_ = we - wb;
                while (n_ > 0) {
                    const OffT half = n_ >> 1;
                    const bool less = colInd[lb + half] < u;
                    lb = less ? lb + half + 1 : lb;
                    n_ = less ? n_ - half - 1 : half;
                }
                hits += lb < we && colInd[lb] == u ? 1u : 0u;
            }
        }
    }
    // the row in the bitmap: the pl ids of adj+ from colInd[pb] on, its first
    // ones in held[] (ids by their number in the row: a position past a row's
    // end may pass 2^32)
    OffT pb = 0;
    uint32_t pl = 0;
    uint32_t held[kHold] = {0, 0};
    auto flip = [&](uint32_t u) { atomicXor(&s_bits[(n - u) >> 5], 1u << ((n - u) & 31u)); };
    if (threadIdx.x == 0) s_tile = line_tile(lines, kLineRows, of);
    __syncthreads();
    uint64_t t = uni64(s_tile);
    while (t * tile < work) {  // block-uniform
        const uint64_t t0 = t * tile, t1 = t0 + tile < work ? t0 + tile : work;
        __syncthreads();  // s_tile is read
        if (threadIdx.x == 0) s_tile = line_tile(lines, kLineRows, of);  // the next tile, read at this one's end
        // row r's work is [rp_in[r] + r*kSplitRowCost, rp_in[r + 1] + (r + 1)*kSplitRowCost)
        const uint32_t r0 = wave_rightmost_le(rows - 1, t0, [&](uint32_t r) {
            return (uint64_t)rp_in[r] + (uint64_t)kSplitRowCost * r;
        });
        // lane l: in-edge and adjacency bounds of row r0 + l (a tile has fewer than 63 rows)
        static_assert(kSplitTile / kSplitRowCost + 2 < kWave, "a tile's rows fit a wave");
        const uint32_t rl = r0 + lane < rows ? r0 + lane : rows;
        const OffT my_in = rp_in[rl], my_adj = rowPtr[(uint64_t)thr + rl];
        // the tile's in-edges [ka, kz) and adjacency, al ids from ab on, of row r0 + x
        auto row_bounds = [&](uint32_t x, uint64_t &ka, uint64_t &kz, OffT &ab, uint32_t &al) {
            const uint64_t b = readlane_u64((uint64_t)my_in, x), e = readlane_u64((uint64_t)my_in, x + 1);
            const uint64_t c = (uint64_t)kSplitRowCost * (r0 + x + 1);
            ka = t0 > b + c ? t0 - c : b;
            kz = t1 < e + c ? (t1 > b + c ? t1 - c : b) : e;
            ab = (OffT)readlane_u64((uint64_t)my_adj, x);
            al = (uint32_t)((OffT)readlane_u64((uint64_t)my_adj, x + 1) - ab);
        };
        // the next row from x on with in-edges in the tile, or kSentinel
        auto next_row = [&](uint32_t x) -> uint32_t {
            for (; r0 + x < rows; x++) {
                uint64_t ka, kz;
                OffT b;
                uint32_t l;
                row_bounds(x, ka, kz, b, l);
                if ((uint64_t)readlane_u64((uint64_t)my_in, x) + (uint64_t)kSplitRowCost * (r0 + x) >= t1) break;
                if (ka < kz) return x;
            }
            return kSentinel;
        };
        uint32_t x = next_row(0);
        uint64_t k = 0, kend = 0;
        OffT ab = 0;
        uint32_t al = 0, ids[kHold] = {0, 0};
        if (x != kSentinel) {
            row_bounds(x, k, kend, ab, al);
#pragma unroll
            for (uint32_t z = 0; z < kHold; z++) {
                const uint32_t i = threadIdx.x + z * kThreads;
                if (i < al) ids[z] = colInd[ab + (OffT)i];
            }
        }
        while (x != kSentinel) {  // block-uniform
            // this row's bits in, the row before's out
#pragma unroll
            for (uint32_t z = 0; z < kHold; z++) {
                if (threadIdx.x + z * kThreads < pl) flip(held[z]);
                if (threadIdx.x + z * kThreads < al) flip(ids[z]);
                held[z] = ids[z];
            }
            for (uint32_t i = threadIdx.x + kHold * kThreads; i < pl; i += kThreads) flip(colInd[pb + (OffT)i]);
            for (uint32_t i = threadIdx.x + kHold * kThreads; i < al; i += kThreads) flip(colInd[ab + (OffT)i]);
            pb = ab;
            pl = al;
            const uint64_t ck = k, ckend = kend;
            const bool far = rows - (r0 + x) > kPackNear;  // the row's tails have far ids
            __syncthreads();
            // the next row's ids, on their way while this row is streamed
            x = next_row(x + 1);
            if (x != kSentinel) {
                row_bounds(x, k, kend, ab, al);
#pragma unroll
                for (uint32_t z = 0; z < kHold; z++) {
                    const uint32_t i = threadIdx.x + z * kThreads;
                    if (i < al) ids[z] = colInd[ab + (OffT)i];
                }
            }
            uint32_t h = 0;
            uint64_t x0 = ck + (uint64_t)wv * kPer;
            OffT lo = 0, hi = 0;  // a tail's first chunk, its chunks
            if (x0 + sub < ckend) {
                lo = ieG[2 * (x0 + sub)];
                hi = ieG[2 * (x0 + sub) + 1];
            }
            while (x0 < ckend) {
                // the bounds of the step after this one
                x0 += (uint64_t)kWaves * kPer;
                OffT nlo = 0, nhi = 0;
                if (x0 + sub < ckend) {
                    nlo = ieG[2 * (x0 + sub)];
                    nhi = ieG[2 * (x0 + sub) + 1];
                }
                const gptr<u32x4> at = packed + lo + sl;
                const uint32_t near = (uint32_t)hi & 8191u;
                h += rows_tail_hits<3, kLanes>(s_bits, at, near, sl);
                if (kLayout != 3 && far) h += rows_tail_hits<kLayout, kLanes>(s_bits, at + near, (uint32_t)hi >> 13, sl);
                lo = nlo;
                hi = nhi;
            }
            hits += h;
            __syncthreads();
        }
        __syncthreads();  // the next tile is there, also after a tile without in-edges
        t = uni64(s_tile);
    }
    hits = wave_sum(hits);
    if (lane == 0 && hits) line_add(lines, kLineHits, hits);
}

// ---------------------------------------------------------------- list part

// Persistent blocks take tiles of the slabs' work from sixteen counters: a slab's
// work is kSlabCost for its rows and one unit per in-edge, in tiles of at most
// kSlabTile, as in the row kernel (with tiles of in-edges alone, those over
// the many slabs with few in-edges took 0.45 ms on R-MAT-20 however few the
// list rows were; half or twice as large tiles cost R-MAT-24 12% and 22%).
// A tile's in-edges of one slab form a segment.  Per segment, the block hashes
// into LDS every row of the slab the segment's in-edges name that is not there
// yet (the table is kept while the next segment stays in the slab; a wave per
// row clears its buckets and inserts its ids): the row starting at window
// position st with len entries owns the buckets [st, st + len) of kSetWays
// slots each, so a quarter of its slots are filled; an id whose bucket is full
// marks it and goes to the next.  Then the segment's in-edges are dealt to the
// waves, 4 or 8 lanes each, the next step's first ids and the bounds of the
// one after on their way while this one's tails are streamed and looked up
// (set_hits; by a binary search in HBM for a row longer than kSlabRowMax).
// No one unit is full (R-MAT-26: vector instructions 54%, lines from beyond
// L2 60%, LDS 37%): bound by the chain of a segment at the 24 waves a CU that
// the tables leave.  Against a hash by 32-bit multiplications, full buckets
// not marked (a wave met a full one in 7 of 10 lookups, now one in 5) and
// loads not ahead of the tables: R-MAT-26 36.2 -> 27.8 ms, R-MAT-24 2.61 ->
// 2.08, R-MAT-22 0.43 -> 0.37.  Eight lanes where tails are long: R-MAT-26
// (~90 ids) 27.8 against 30.1 with four, R-MAT-24 (49 ids) 2.16 against 2.06.
// Where a is short for the graph, most list wedges name long rows and the
// searches' chains of loads are the time (R-MAT-26 at a = 65,536: four ids a
// lane side by side 218 ms, one after the other 308).
// Same alignment and slack needs as the row kernel.
template <typename OffT, int kWaves, bool kWide>
__global__ __launch_bounds__(kWave * kWaves) void k_split_slabs(const GraphDesc *__restrict__ desc,
                                                                const SplitDesc *__restrict__ sd,
                                                                const uint64_t *__restrict__ meta,
                                                                uint64_t *__restrict__ lines) {
    constexpr uint32_t kRefWords = kSlabSpan / 32;
    __shared__ __align__(16) uint32_t s_tab[kSlabWin * kSetWays];
    __shared__ uint32_t s_ref[kRefWords];  // rows (by start position) hashed so far
    __shared__ uint32_t s_new[kSlabTile];  // slab_aux words of the rows a segment adds
    __shared__ uint32_t s_nnew;
    __shared__ uint64_t s_tile;
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const OffT *__restrict__ rowPtr = static_cast<const OffT *>(D.rowPtr);
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const cptr<OffT> rp_in = to_const(static_cast<const OffT *>(S.rp_in));
    const gptr<OffT> ieG = to_global(static_cast<const OffT *>(S.ie));
    const gptr<uint32_t> auxG = to_global(static_cast<const uint32_t *>(S.ie_aux));
    const uint32_t rows = S.rows, keys = S.keys;
    const uint64_t L0 = (uint64_t)rp_in[rows], L1 = (uint64_t)rp_in[keys];
    constexpr uint32_t kThreads = kWave * kWaves;
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    // lanes to a tail: a turn of four takes 16 ids, of eight 32
    const uint32_t lanes = uni64(meta[kMetaListWedges]) > (uint64_t)kSlabLong * (L1 - L0) ? 8u : 4u;
    const uint32_t per = kWave / lanes, deal = kWaves * per, step = 4 * lanes, sub = lane / lanes, sl = lane % lanes;
    uint32_t cur = kSentinel;  // slab in s_tab (block-uniform)
    uint64_t hits = 0;
    const uint64_t work = L1 - L0 + (uint64_t)kSlabCost * (keys - rows);
    // about four tiles a block: their chains are long (R-MAT-20 63 us, with eight 79)
    uint64_t tile = work / (4ull * gridDim.x);
    tile = tile < kSlabTileMin ? kSlabTileMin : tile > kSlabTile ? kSlabTile : tile;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_tile = line_tile(lines, kLineSlabs, kTileLines);
        __syncthreads();
        const uint64_t t0 = uni64(s_tile) * tile;
        if (t0 >= work || L0 == L1) break;  // block-uniform
        const uint64_t t1 = t0 + tile < work ? t0 + tile : work;
        // slab y's work is [rp_in[rows + y] - L0 + y*kSlabCost, rp_in[rows + y + 1] - L0 + (y + 1)*kSlabCost)
        const uint32_t y0 = wave_rightmost_le(keys - rows - 1, t0, [&](uint32_t y) {
            return (uint64_t)rp_in[rows + y] - L0 + (uint64_t)kSlabCost * y;
        });
        for (uint32_t key = rows + y0; key < keys; key++) {
            const uint64_t c = (uint64_t)kSlabCost * (key - rows + 1);  // in-edges after this much of the work
            const uint64_t kb = (uint64_t)rp_in[key] - L0, ke = (uint64_t)rp_in[key + 1] - L0;
            if (kb + c - kSlabCost >= t1) break;  // block-uniform
            const uint64_t k = L0 + (t0 > kb + c ? t0 - c : kb);
            const uint64_t kend = L0 + (t1 < ke + c ? (t1 > kb + c ? t1 - c : kb) : ke);
            if (k >= kend) continue;
            const uint32_t slab = key - rows;
            const uint64_t wb = (uint64_t)slab * kSlabSpan;  // window start in colInd
            // the segment's in-edges are dealt to the waves, `lanes` lanes each;
            // the first two steps' and the first tails' first ids are on their
            // way while the table is built
            struct Edge {
                OffT j, hi;
                uint32_t aux;
                // the tail from the aligned position at or before it: its
                // first position and what is from there to its end (positions
                // by what is left: one past the tail may pass 2^32)
                __device__ __forceinline__ OffT base() const { return (j + 1) & ~(OffT)3; }
                __device__ __forceinline__ uint32_t span() const { return (uint32_t)(hi - base()); }
                __device__ __forceinline__ bool hashed() const { return (aux >> 13) != 0 && (aux >> 13) != kSlabAuxLong; }
            };
            auto edge = [&](uint64_t x) -> Edge {
                Edge e{0, 0, 0u};
                if (x < kend) {
                    e.j = ieG[2 * x];
                    e.hi = ieG[2 * x + 1];
                    e.aux = auxG[x];
                }
                return e;
            };
            auto head = [&](const Edge &e) -> u32x4 {
                u32x4 r = {0u, 0u, 0u, 0u};
                if (e.hashed() && 4 * sl < e.span()) r = *reinterpret_cast<gptr<u32x4>>(colInd + e.base() + 4 * sl);
                return r;
            };
            uint64_t x0 = k + (uint64_t)wv * per + sub;
            Edge ed = edge(x0), en = edge(x0 + deal);
            u32x4 ids = head(ed);
            // the rows this segment names that the table lacks
            __syncthreads();  // the previous segment's lookups are done
            if (slab != cur)
                for (uint32_t i = threadIdx.x; i < kRefWords; i += kThreads) s_ref[i] = 0u;
            if (threadIdx.x == 0) s_nnew = 0u;
            cur = slab;
            __syncthreads();
            for (uint64_t x = k + threadIdx.x; x < kend; x += kThreads) {
                const uint32_t aux = auxG[x], st = aux & kSlabAuxLong, len = aux >> 13;
                if (len == kSlabAuxLong || len == 0) continue;  // searched in HBM, or empty
                const uint32_t bit = 1u << (st & 31u);
                if ((atomicOr(&s_ref[st >> 5], bit) & bit) == 0u) s_new[atomicAdd(&s_nnew, 1u)] = aux;
            }
            __syncthreads();
            // a wave per new row: its buckets cleared, then its ids inserted
            // (one wave's LDS operations stay in order), the next row's first
            // ids loaded before
            const uint32_t nnew = s_nnew;
            {
                uint32_t aux = wv < nnew ? s_new[wv] : 0u;
                uint32_t u = lane < aux >> 13 ? colInd[wb + (aux & kSlabAuxLong) + lane] : 0u;
                for (uint32_t r = wv; r < nnew; r += kWaves) {
                    const uint32_t naux = r + kWaves < nnew ? s_new[r + kWaves] : 0u;
                    const uint32_t nu = lane < naux >> 13 ? colInd[wb + (naux & kSlabAuxLong) + lane] : 0u;
                    const uint32_t st = aux & kSlabAuxLong, len = aux >> 13;
                    for (uint32_t i = lane; i < len; i += kWave)
                        reinterpret_cast<uint4 *>(s_tab)[st + i] = make_uint4(kSetFree<kWide>, kSetFree<kWide>, kSetFree<kWide>, kSetFree<kWide>);
                    for (uint32_t i = lane; i < len; i += kWave) {
                        if (i >= kWave) u = colInd[wb + st + i];
                        set_insert<kWide>(s_tab, st, len, u);
                    }
                    aux = naux;
                    u = nu;
                }
            }
            __syncthreads();
            uint32_t h = 0;
            for (; x0 - sub < kend; x0 += deal) {
                const Edge e2 = edge(x0 + 2 * deal);
                const u32x4 nids = head(en);
                const uint32_t st = ed.aux & kSlabAuxLong, len = ed.aux >> 13;
                const bool some = 4 * sl < ed.span();  // this lane's share of the tail
                uint32_t left = some ? ed.span() - 4 * sl : 0u;
                const uint32_t skip = sl == 0 ? (uint32_t)(ed.j + 1 - ed.base()) : 0u;  // ids before the tail
                gptr<uint32_t> p = colInd + ed.base() + 4 * sl;
                if (ed.hashed() && some) {
                    u32x4 a = ids;
                    if (skip) {  // 0 is in no row
                        a[0] = 0u;
                        a[1] = skip > 1 ? 0u : a[1];
                        a[2] = skip > 2 ? 0u : a[2];
                    }
                    for (;;) {
                        u32x4 b = a;
                        if (left > step) b = *reinterpret_cast<gptr<u32x4>>(p + step);
                        const uint32_t u[4] = {a[0], a[1], a[2], a[3]};
                        h += set_hits<kWide>(s_tab, u, left, st, len);
                        if (left <= step) break;
                        left -= step;
                        p += step;
                        a = b;
                    }
                } else if (len == kSlabAuxLong) {  // a long row: adj+(w) searched in HBM
                    const uint32_t w = colInd[ed.j];
                    OffT gb = rowPtr[w];
                    const OffT ge = rowPtr[(uint64_t)w + 1];
                    for (uint32_t before = skip; left; before = 0) {  // four ids' halvings side by side
                        const u32x4 a = *reinterpret_cast<gptr<u32x4>>(p);
                        OffT at[4] = {gb, gb, gb, gb};  // the last id <= a[z], or the range's first
                        for (OffT n_ = ge - gb; n_ > 1;) {
                            const OffT half = n_ >> 1;
                            uint32_t v[4];
#pragma unroll
                            for (int z = 0; z < 4; z++) v[z] = colInd[at[z] + half];
#pragma unroll
                            for (int z = 0; z < 4; z++) at[z] = v[z] <= a[z] ? at[z] + half : at[z];
                            n_ -= half;
                        }
#pragma unroll
                        for (uint32_t z = 0; z < 4; z++)
                            h += z >= before && z < left && colInd[at[z]] == a[z] ? 1u : 0u;
                        gb = at[3];  // the lane's next id is larger
                        left = left > step ? left - step : 0u;
                        p += step;
                    }
                }
                ed = en;
                en = e2;
                ids = nids;
            }
            hits += h;
        }
    }
    hits = wave_sum(hits);
    if (lane == 0 && hits) line_add(lines, kLineHits, hits);
}

// ---------------------------------------------------------------- launches

hipError_t launch_split_prefix(const GraphDesc *desc, const SplitDesc *sd, int ob, uint32_t nblocks,
                               uint64_t *partials, hipStream_t st) {
    if (nblocks == 0) return hipSuccess;
    hipError_t e = WTC_LAUNCH_OFF(ob, k_split_partials, dim3(nblocks), dim3(kBlock), 0, st, desc, partials);
    if (e != hipSuccess) return e;
    if ((e = launch_scan_partials(partials, nblocks, st)) != hipSuccess) return e;
    return WTC_LAUNCH_OFF(ob, k_split_scan, dim3(nblocks), dim3(kBlock), 0, st, desc, sd, (const uint64_t *)partials);
}

hipError_t launch_split_inscan(const GraphDesc *desc, const SplitDesc *sd, uint32_t nblocks, uint64_t *part_in,
                               hipStream_t st) {
    hipError_t e = launch_scan_partials(part_in, nblocks, st);
    if (e != hipSuccess) return e;
    k_split_inscan<<<dim3(nblocks), dim3(kBlock), 0, st>>>(desc, sd, part_in);
    return hipGetLastError();
}

// 8-byte row offsets that all fit 32 bits, copied to 4 bytes.
__global__ __launch_bounds__(kBlock) void k_split_narrow_offsets(const uint64_t *__restrict__ src,
                                                                uint32_t *__restrict__ dst, uint64_t count) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = (uint32_t)src[i];
}

hipError_t launch_split_narrow_offsets(const uint64_t *src, uint32_t *dst, uint64_t count, hipStream_t st) {
    if (count == 0) return hipSuccess;
    const uint64_t blocks = (count + kBlock - 1) / kBlock;
    k_split_narrow_offsets<<<dim3((uint32_t)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, st>>>(src, dst, count);
    return hipGetLastError();
}

hipError_t launch_split_range(const GraphDesc *desc, SplitDesc *sd, int ob, hipStream_t st) {
    return WTC_LAUNCH_OFF(ob, k_split_range, dim3(1), dim3(kSplitPartsMax), 0, st, desc, sd);
}

namespace {

template <typename KeyIn, bool kFinal, uint32_t kF>
hipError_t launch_level_count(const SplitDesc *sd, uint32_t grid, hipStream_t st) {
    k_split_level_count<KeyIn, kFinal, kF><<<dim3(grid), dim3(kSplitBlock), 0, st>>>(sd);
    return hipGetLastError();
}

template <typename OffT, typename KeyIn, bool kFinal, uint32_t kF>
hipError_t launch_level_scatter(const SplitDesc *sd, uint32_t grid, hipStream_t st) {
    k_split_level_scatter<OffT, KeyIn, kFinal, kF><<<dim3(grid), dim3(kSplitBlock), 0, st>>>(sd);
    return hipGetLastError();
}

// The final level's count or scatter: from B, or from A by a part's keys.
template <typename OffT>
hipError_t launch_final(bool scatter, bool from_b, uint32_t shift, const SplitDesc *sd, uint32_t grid, hipStream_t st) {
    if (from_b)
        return scatter ? launch_level_scatter<OffT, uint8_t, true, kSplitSub>(sd, grid, st)
                       : launch_level_count<uint8_t, true, kSplitSub>(sd, grid, st);
    switch (shift) {
        case 8:
            return scatter ? launch_level_scatter<OffT, uint16_t, true, 256>(sd, grid, st)
                           : launch_level_count<uint16_t, true, 256>(sd, grid, st);
        case 9:
            return scatter ? launch_level_scatter<OffT, uint16_t, true, 512>(sd, grid, st)
                           : launch_level_count<uint16_t, true, 512>(sd, grid, st);
        case 10:
            return scatter ? launch_level_scatter<OffT, uint16_t, true, 1024>(sd, grid, st)
                           : launch_level_count<uint16_t, true, 1024>(sd, grid, st);
        case 11:
            return scatter ? launch_level_scatter<OffT, uint16_t, true, 2048>(sd, grid, st)
                           : launch_level_count<uint16_t, true, 2048>(sd, grid, st);
        default: return hipErrorInvalidValue;
    }
}

template <typename OffT>
hipError_t transpose(const GraphDesc *desc, const SplitDesc *sd, const DenseDesc *dd, const SplitGrids &g,
                     uint64_t *key_part, uint64_t *meta, hipStream_t st) {
    const dim3 blk(kSplitBlock);
    const uint32_t g2 = g.c2cap < kLevelGridMax ? g.c2cap : kLevelGridMax;
    const uint32_t g3 = g.c3cap < kLevelGridMax ? g.c3cap : kLevelGridMax;
    const bool three = g.part_shift != g.final_shift;
    hipError_t e;
    k_split_parthist<OffT><<<dim3(g.chunks), blk, 0, st>>>(desc, sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_split_partbase<<<dim3(1), dim3(kBlock), 0, st>>>(sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_split_l1<OffT><<<dim3(g.chunks), blk, 0, st>>>(desc, sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_split_bases<false><<<dim3(1), blk, 0, st>>>(sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (three) {
        if ((e = launch_level_count<uint16_t, false, kSplitFan2>(sd, g2, st)) != hipSuccess) return e;
        k_split_levelcols2<<<dim3(g.parts), blk, 0, st>>>(sd);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        k_split_bases<true><<<dim3(1), blk, 0, st>>>(sd);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = launch_level_scatter<OffT, uint16_t, false, kSplitFan2>(sd, g2, st)) != hipSuccess) return e;
    }
    if ((e = launch_final<OffT>(false, three, g.final_shift, sd, g3, st)) != hipSuccess) return e;
    k_split_levelcols3<<<dim3((g.keys + kBlock - 1) / kBlock), dim3(kBlock), 0, st>>>(sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const dim3 gkb((g.keys + kKeyChunk - 1) / kKeyChunk);
    k_split_keysum<<<gkb, blk, 0, st>>>(sd);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = launch_scan_partials(key_part, gkb.x, st)) != hipSuccess) return e;
    k_split_keyscan<OffT><<<gkb, blk, 0, st>>>(sd, dd, meta);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = launch_final<OffT>(true, three, g.final_shift, sd, g3, st)) != hipSuccess) return e;
    // the packed top ids, over the final level's input pairs
    k_split_pack<OffT><<<dim3(kPackGrid), dim3(kBlock), 0, st>>>(desc, sd);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_split_transpose(const GraphDesc *desc, const SplitDesc *sd, const DenseDesc *dd, int ob,
                                  const SplitGrids &g, uint64_t *key_part, uint64_t *meta, hipStream_t st) {
    if (g.keys == 0 || g.chunks == 0 || g.c3cap == 0 || g.parts == 0 || g.parts > kSplitPartsMax)
        return hipErrorInvalidValue;
    return ob == 8 ? transpose<uint64_t>(desc, sd, dd, g, key_part, meta, st)
                   : transpose<uint32_t>(desc, sd, dd, g, key_part, meta, st);
}

uint32_t split_far_ids(uint32_t rows) { return pack_layout(rows) == 2 ? PackLayout<2>::P : PackLayout<0>::P; }

size_t split_rows_lds(uint32_t rows) { return (size_t)(((rows + 31) / 32 + 1) & ~1u) * sizeof(uint32_t) + sizeof(uint64_t); }

template <int W, int L>
static const void *split_rows_fn(int ob) {
    return ob == 8 ? reinterpret_cast<const void *>(&k_split_rows<uint64_t, W, kSplitLanes, L>)
                   : reinterpret_cast<const void *>(&k_split_rows<uint32_t, W, kSplitLanes, L>);
}

template <int L>
static const void *split_rows_kernel_l(int ob, int wpb) {
    switch (wpb) {
        case 4: return split_rows_fn<4, L>(ob);
        case 16: return split_rows_fn<16, L>(ob);
        default: return split_rows_fn<8, L>(ob);
    }
}

// The row kernel for a graph of `rows` top rows (the packing's layout).
static const void *split_rows_kernel(int ob, int wpb, uint32_t rows) {
    switch (pack_layout(rows)) {
        case 0: return split_rows_kernel_l<0>(ob, wpb);
        case 1: return split_rows_kernel_l<1>(ob, wpb);
        case 2: return split_rows_kernel_l<2>(ob, wpb);
        default: return split_rows_kernel_l<3>(ob, wpb);
    }
}

bool valid_split_waves(int wpb) { return wpb == 4 || wpb == 8 || wpb == 16; }

hipError_t split_rows_grid(int ob, uint32_t rows, int wpb, int num_cus, uint32_t *grid) {
    if (!valid_split_waves(wpb)) return hipErrorInvalidValue;
    const void *fn = split_rows_kernel(ob, wpb, rows);
    const size_t shm = split_rows_lds(rows);
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return e;
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, wpb * kWave, shm);
    if (e != hipSuccess) return e;
    if (per_cu < 1) return hipErrorInvalidConfiguration;  // the row bitmap does not fit LDS
    *grid = (uint32_t)per_cu * (uint32_t)(num_cus > 0 ? num_cus : 1);
    return hipSuccess;
}

hipError_t launch_split_rows(const GraphDesc *desc, const SplitDesc *sd, int ob, uint32_t rows, int wpb,
                             uint64_t *lines, uint32_t grid, hipStream_t st) {
    if (rows == 0) return hipSuccess;
    if (!valid_split_waves(wpb) || grid == 0 || rows > kPackRowsMax) return hipErrorInvalidValue;
    const void *fn = split_rows_kernel(ob, wpb, rows);
    void *args[] = {&desc, &sd, &lines};
    return hipLaunchKernel(fn, dim3(grid), dim3(wpb * kWave), args, split_rows_lds(rows), st);
}

// The slab kernel's block (three to a CU by their LDS).
constexpr int kSlabWaves = 8;

template <bool kWide>
static const void *split_slabs_fn(int ob) {
    return ob == 8 ? reinterpret_cast<const void *>(&k_split_slabs<uint64_t, kSlabWaves, kWide>)
                   : reinterpret_cast<const void *>(&k_split_slabs<uint32_t, kSlabWaves, kWide>);
}

// The slab kernel for a graph of n vertices (its sets of ids).
static const void *split_slabs_kernel(int ob, uint32_t n) {
    return n > kSetIdsEnd ? split_slabs_fn<true>(ob) : split_slabs_fn<false>(ob);
}

hipError_t split_slabs_grid(int ob, uint32_t n, int num_cus, uint32_t *grid) {
    int per_cu = 0;
    hipError_t e =
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, split_slabs_kernel(ob, n), kSlabWaves * kWave, 0);
    if (e != hipSuccess) return e;
    if (per_cu < 1) return hipErrorInvalidConfiguration;
    *grid = (uint32_t)per_cu * (uint32_t)(num_cus > 0 ? num_cus : 1);
    return hipSuccess;
}

hipError_t launch_split_slabs(const GraphDesc *desc, const SplitDesc *sd, int ob, uint32_t n, const uint64_t *meta,
                              uint64_t *lines, uint32_t grid, hipStream_t st) {
    if (grid == 0) return hipErrorInvalidValue;
    void *args[] = {&desc, &sd, &meta, &lines};
    return hipLaunchKernel(split_slabs_kernel(ob, n), dim3(grid), dim3(kSlabWaves * kWave), args, 0, st);
}

}  // namespace wtc
