// wtc_rows.hip -- the row count (counting kernel choice kKernelRows): whole
// graphs, alone or in sets, counted edge by edge against hashed rows.
//
// Every edge v -> w closes |adj+(v) ∩ adj+(w)| triangles: the ids of adj+(w)
// are above w, so this is the intersection of w's row with the tail of v's
// row after w, which the wedge-parallel kernels check wedge by wedge
// (tc.cu:203-287).  A block takes a tile of kRowsTile consecutive positions
// of colInd (edges), hashes the rows of v that they lie in into LDS, streams
// adj+(w) for each of its edges with 16-byte loads, and looks every id up in
// v's set: one 16-byte LDS read an id.  These are the arrow wedges v -> w -> u
// (counted on R-MAT, Erdos-Renyi and Barabasi-Albert graphs 1.2 to 4 times as
// many as the wedges (w, u) of v), with no wedge prefix, no tile search per
// wedge, no bitmap and no chain of dependent probes: three launches a count
// (descriptors and zeroes, the count, the results), whatever the number of
// graphs.
//
// Nothing bounds the arrow wedges by the wedges: where many vertices of few
// neighbours hang on a dense core there are ten to sixty times as many.  So an
// edge whose adj+(w) is long beside what is left of v's row (kRowsLong,
// kRowsFew) is done the other way round: the rest of v's row is searched in
// adj+(w).  What is streamed is then at most kRowsLong ids an edge and kRowsFew
// a wedge.  1,000 vertices all joined with 10^7 of two neighbours among them:
// 7.6 ms streamed, 0.77 so, 0.84 by the staged kernel; 400 with 2 * 10^6: 0.49,
// 0.18 and 0.34; R-MAT-16 102 -> 96 us, R-MAT-18 0.52 -> 0.48 ms.
//
// Measured against the staged kernel on its tuned shape (whole call): R-MAT-12
// 28 us instead of 146, R-MAT-16 95 instead of 323, R-MAT-18 0.48 ms instead
// of 0.88, Erdos-Renyi n = 10^6 of degree 16 0.21 ms instead of 0.58, 256
// Erdos-Renyi and Barabasi-Albert graphs 1.23 ms instead of 2.69.  From 2^27
// wedges on skewed graphs the split count is faster (R-MAT-18: 0.33 against
// 0.48 ms, R-MAT-19: 0.47 against 1.7).  Bound by a tile's chain of loads and
// barriers at the 24 waves a CU that its registers leave, on skewed graphs by
// a lookup's vector instructions as well.
#include "wtc_dev.h"
#include "wtc_kernels.h"
#include "wtc_launch.h"
#include "wtc_set.h"

namespace wtc {

namespace {

// Four ids at any element (4-byte) alignment.
typedef uint32_t u32x4_e __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRowsThreads = 512;
static_assert(kRowsThreads == (int)kRowsTile, "a position per thread");
constexpr uint32_t kRowsWaves = kRowsThreads / kWave;
// Buckets of four slots per position: one bucket in 6,000 is left by an id
// that finds it full.
constexpr uint32_t kRowsSpread = 2;
// The table has that many for the tile and a last row of as many positions; a
// longer last row gets what is left.
constexpr uint32_t kRowsBuckets = kRowsSpread * 2 * kRowsTile;
// Longest row (from its first position in the tile) hashed, two ids a bucket
// at most; what is longer is searched in memory.  (With 512, two graphs of
// 1,000 vertices all joined took 1.91 ms, the staged kernel 1.65; so 0.30.)
constexpr uint32_t kRowsRowMax = 2048;
static_assert(4 * (kRowsBuckets - kRowsSpread * (kRowsTile - 1)) > kRowsRowMax, "the longest row hashed leaves slots free");
// An edge's adj+(w) of kRowsLong ids or more is not streamed where it has
// kRowsFew times the ids of the rest of v's row or more: those are searched in
// it.  (kRowsFew 8: R-MAT-18 0.54 ms, 16 and 32 0.48 and 0.49, R-MAT-16 97 and
// 99 us; kRowsLong 128 or 256: within 1%, R-MAT-17 3% more.)
constexpr uint32_t kRowsLong = 64, kRowsFew = 16;

}  // namespace

// The descriptors from the host's pinned memory, the counts and the wedge
// total zeroed: a kernel, not copies, since two of those cost more than the
// rest of a small graph's count.
__global__ __launch_bounds__(kBlock) void k_rows_init(const uint64_t *__restrict__ host_desc, GraphDesc *__restrict__ desc,
                                                      uint32_t G, uint64_t *__restrict__ meta,
                                                      unsigned long long *__restrict__ counts,
                                                      uint64_t *__restrict__ lines) {
    static_assert(sizeof(GraphDesc) % 8 == 0, "copied by words");
    const uint64_t step = (uint64_t)gridDim.x * kBlock, at = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (host_desc)
        for (uint64_t i = at; i < (uint64_t)G * (sizeof(GraphDesc) / 8); i += step)
            reinterpret_cast<uint64_t *>(desc)[i] = host_desc[i];
    for (uint64_t i = at; i < G; i += step) counts[i] = 0ull;
    if (at < kMetaSlots) meta[at] = 0ull;
    for (uint64_t i = at; i < kLines * kLineWords; i += step) lines[i] = 0ull;
}

// Groups of `group` consecutive tiles of the set (D.tile_base: a graph's first
// tile; D.wcount: its edges) dealt to the blocks in turn.  Per tile:
//  1. the rows of the tile set their first position's bit and leave their end
//     there (the first row of a group is found by a 64-way search, later ones
//     from the tile before), while the table of sets is cleared;
//  2. every position finds its row as the last bit at or before it, its id w
//     goes into the set of its row v (a row of len positions owns kRowsSpread *
//     len buckets of four slots, one 16-byte LDS read each), the last row's ids
//     past the tile too, and its edge into a list;
//  3. the edges with an adj+(w) that may meet v's row are listed by the
//     length of adj+(w) and streamed by 2, 4 or 8 lanes each, four ids a lane a
//     step, so that a long one takes many steps and little of them is empty
//     (with up to 32 lanes: R-MAT-16 117 against 112 us, the serving mix 2.77
//     against 2.65 ms); the next step's ids load while this one's are looked
//     up.  The edges to be searched go to the last waves first, which have the
//     least to stream (R-MAT-12 27.8 us, dealt from the first wave on 28.7).
// The next tile's rows, ids and bounds of adj+(w) load while a tile is
// streamed.  Three barriers a tile (with a running maximum over marks, a clear
// of the table by the rows' extent and lists packed by a prefix, seven:
// Erdos-Renyi graph 260 against 250 us, the batch 1.34 against 1.28 ms).
// (Six waves a SIMD, three blocks a CU, take 80 registers and the lookups two
// at a time; with five 0.30 instead of 0.26 ms on the Erdos-Renyi graph, and
// with eight, spilling, 0.35.)
template <typename OffT>
__global__ __launch_bounds__(kRowsThreads, 6) void k_rows(const GraphDesc *__restrict__ desc, uint32_t G, uint64_t tiles,
                                                       uint32_t group, uint32_t tile_edges,
                                                       unsigned long long *__restrict__ counts,
                                                       uint64_t *__restrict__ lines) {
    constexpr uint32_t kT = kRowsTile;
    // adj+(w) of up to 8, of up to 32 ids, and more; the rest of v's row to be
    // searched in it; edges of a row not hashed
    constexpr uint32_t kStreams = 3, kSearch = kStreams, kUnhashed = kStreams + 1, kLists = kStreams + 2;
    __shared__ __align__(16) uint32_t s_tab[kRowsBuckets * 4];
    __shared__ OffT s_ws[kT];        // start of adj+(w)
    __shared__ uint32_t s_wl[kT];    // its length
    __shared__ uint16_t s_end[kT];   // at a row's first position: its end, from the tile's start (at most 2^16 - 1)
    __shared__ uint16_t s_mark[kT];  // a position's row, as the row's first position
    __shared__ uint16_t s_list[kLists][kT];  // the edges to stream
    // rows' first positions as bits, and the lists' edges, of this tile and (zeroed) the next
    __shared__ unsigned long long s_first[2][kT / 64];
    constexpr uint32_t kCounts = 8, kRare = 4;  // list c's count at c, the rare lists' at kRare and on
    __shared__ __align__(16) uint32_t s_n[2][kCounts];
    __shared__ uint64_t s_sum[kRowsWaves];
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    uint32_t cur_g = kSentinel, buf = 0;
    uint64_t hits = 0, wedges = 0;
    if (threadIdx.x < kT / 64) s_first[1][threadIdx.x] = 0ull;
    if (threadIdx.x < kCounts) s_n[1][threadIdx.x] = 0u;
    // x summed over the block (thread 0)
    auto block_sum = [&](uint64_t x) -> uint64_t {
        const uint64_t t = wave_sum(x);
        __syncthreads();
        if (lane == 0) s_sum[wv] = t;
        __syncthreads();
        uint64_t all = 0;
        if (threadIdx.x == 0)
            for (uint32_t w = 0; w < kRowsWaves; w++) all += s_sum[w];
        return all;
    };
    // the block's hits of graph cur_g into its count
    auto flush = [&]() {
        const uint64_t all = block_sum(hits);
        if (threadIdx.x == 0 && all) {
            if (G == 1) line_add(lines, kLineHits, all);
            else atomicAdd(&counts[cur_g], (unsigned long long)all);
        }
        hits = 0;
    };
    // the current tile: its graph's arrays, positions [p0, p0 + nt) of m
    gptr<OffT> rowPtr = nullptr;
    gptr<uint32_t> colInd = nullptr;
    uint32_t n = 1;
    uint64_t p0 = 0, m = 0, g_end = 0;
    uint64_t vb = 0;  // a row at or before the tile's first, within kRowsThreads rows of it but for empty rows
    // this thread's row vb + threadIdx.x of the tile, and its position's id and adj+ bounds
    OffT ra = 0, rz = 0, ws = 0, we = 0;
    uint32_t id = 0;
    auto load = [&](uint64_t q0, uint64_t r0) {
        const uint64_t v = r0 + threadIdx.x;
        ra = rz = ws = we = 0;
        id = 0;
        if (v < n) {
            ra = rowPtr[v];
            rz = rowPtr[v + 1];
        }
        if (q0 + threadIdx.x < m) {
            id = colInd[q0 + threadIdx.x];
            ws = rowPtr[id];
            we = rowPtr[(uint64_t)id + 1];
        }
    };
    for (uint64_t t0 = (uint64_t)blockIdx.x * group; t0 < tiles; t0 += (uint64_t)gridDim.x * group) {
        bool fresh = true;
        const uint64_t t1 = t0 + group < tiles ? t0 + group : tiles;
        for (uint64_t tile = t0; tile < t1; tile++) {
            if (fresh || tile >= g_end) {  // block-uniform: a group's or a graph's first tile
                uint32_t g = 0;
                if (G > 1) {  // the last graph whose first tile is at or before this one
                    uint32_t lo = 0, hi = G - 1;
                    while (lo < hi) {
                        const uint32_t mid = (lo + hi + 1) >> 1;
                        if (desc[mid].tile_base <= tile) lo = mid;
                        else hi = mid - 1;
                    }
                    g = lo;
                }
                if (g != cur_g) {
                    if (cur_g != kSentinel) flush();
                    cur_g = g;
                    const GraphDesc &D = desc[g];
                    rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
                    colInd = to_global(D.colInd);
                    n = D.n;
                    m = D.wcount;
                    g_end = D.tile_base + (m + tile_edges - 1) / tile_edges;
                }
                p0 = (tile - desc[g].tile_base) * tile_edges;
                vb = wave_rightmost_le(n - 1, p0, [&](uint32_t r) { return (uint64_t)rowPtr[r]; });
                load(p0, vb);
                fresh = false;
            }
            const uint32_t nt = m - p0 < tile_edges ? (uint32_t)(m - p0) : tile_edges;
            buf ^= 1;
            __syncthreads();  // the previous tile's lookups are done
#pragma unroll
            for (uint32_t i = threadIdx.x; i < kRowsBuckets; i += kRowsThreads)
                reinterpret_cast<uint4 *>(s_tab)[i] = make_uint4(kSetFree<false>, kSetFree<false>, kSetFree<false>, kSetFree<false>);
            if (threadIdx.x < kT / 64) s_first[buf ^ 1][threadIdx.x] = 0ull;
            if (threadIdx.x < kCounts) s_n[buf ^ 1][threadIdx.x] = 0u;
            // windows of rows up to the one holding the tile's last position, or
            // kRowWindows of them and the rows of the positions left
            for (uint32_t win = 1;; win++) {
                const uint64_t a = ra, z = rz;
                if (z > a && z > p0 && a < p0 + nt) {
                    const uint32_t at = a > p0 ? (uint32_t)(a - p0) : 0u;
                    atomicOr(&s_first[buf][at >> 6], 1ull << (at & 63u));
                    s_end[at] = z - p0 < 0xffffull ? (uint16_t)(z - p0) : (uint16_t)0xffffu;
                    if (a >= p0) wedges += binom2_d(z - a);
                }
                if (win > kRowWindows) break;
                const uint64_t vn = vb + kRowsThreads;
                if (vn >= n) break;  // block-uniform
                const uint64_t next = rowPtr[vn];
                if (next >= p0 + nt) break;  // block-uniform
                ra = rz = 0;
                if (win < kRowWindows) {
                    vb = vn;
                    if (vb + threadIdx.x < n) {
                        ra = rowPtr[vb + threadIdx.x];
                        rz = rowPtr[vb + threadIdx.x + 1];
                    }
                } else {  // block-uniform
                    const uint64_t q = p0 + threadIdx.x;
                    if (threadIdx.x < nt && q >= next) {
                        const uint32_t r = rightmost_le(rowPtr, (uint32_t)vn, n - 1, q);
                        ra = rowPtr[r];
                        rz = (uint64_t)ra == q ? rowPtr[(uint64_t)r + 1] : ra;
                    }
                    vb = vn + wave_rightmost_le((uint32_t)(n - 1 - vn), p0 + nt - 1,
                                                [&](uint32_t r) { return (uint64_t)rowPtr[vn + r]; });
                }
            }
            __syncthreads();
            // a position's row: the last first position at or before it (one
            // is at 0)
            auto row_at = [&](uint32_t i) -> uint32_t {
                uint32_t w = i >> 6;
                unsigned long long x = s_first[buf][w] & (~0ull >> (63u - (i & 63u)));
                while (x == 0) x = s_first[buf][--w];
                return 64u * w + 63u - (uint32_t)__builtin_clzll(x);
            };
            // positions hashed: the tile's rows, the last one to its end, or
            // without it if it is too long (only the last row can be: a row
            // that ends in the tile has at most kT positions there)
            static_assert(kRowsRowMax >= kT, "a row ending in the tile is hashed");
            // a row's region of the table: its first bucket, its buckets above 16 bits
            auto region = [&](uint32_t st, uint32_t end) -> uint32_t {
                constexpr uint32_t kEnd = kRowsBuckets / kRowsSpread;
                return kRowsSpread * (st | ((end < kEnd ? end : kEnd) - st) << 16);
            };
            const uint32_t st_last = uni32(row_at(nt - 1)), end_last = uni32(s_end[st_last]);
            const bool long_last = end_last - st_last > kRowsRowMax;
            const uint32_t bl = long_last ? st_last : end_last;
            const uint32_t me = threadIdx.x;
            if (me < nt) {
                const uint32_t st = row_at(me), end = s_end[st];
                s_mark[me] = (uint16_t)st;
                const uint32_t len = (uint32_t)(we - ws);  // < n
                if (len != 0 && me + 1 != end) {  // else nothing to stream, or nothing after w in v's row
                    s_ws[me] = ws;
                    s_wl[me] = len;
                    uint32_t c = len <= 8 ? 0u : len <= 32 ? 1u : 2u;
                    if (len >= kRowsLong) c = len >= kRowsFew * (end - me - 1) ? kSearch : c;
                    c = long_last && st == st_last ? kUnhashed : c;
                    s_list[c][atomicAdd(&s_n[buf][c + (c >= kStreams ? kRare - kStreams : 0u)], 1u)] = (uint16_t)me;
                }
                if (me < bl) {
                    const uint32_t r = region(st, end);
                    set_insert(s_tab, r & 0xffffu, r >> 16, id);
                }
            }
            for (uint32_t i = nt + threadIdx.x; i < bl; i += kRowsThreads) {
                const uint32_t r = region(st_last, end_last);
                set_insert(s_tab, r & 0xffffu, r >> 16, colInd[p0 + i]);
            }
            __syncthreads();
            const uint64_t cp0 = p0;
            p0 += tile_edges;
            if (tile + 1 < t1 && tile + 1 < g_end) load(p0, vb);
            uint32_t h = 0;
            for (uint32_t c = 0; c < kStreams; c++) {  // list c: 2 << c lanes an edge, four ids each a step
                const uint32_t lanes = 2u << c, o = 4 * (lane & (lanes - 1)), end = uni32(s_n[buf][c]);
                uint32_t x = threadIdx.x >> (c + 1);
                // the step ahead: ids of row st at `at` of the wl from ws
                uint32_t at = 0, wl = 0, set = 0;  // set: v's region, its length above 16 bits
                OffT from = 0;
                u32x4 q = {0u, 0u, 0u, 0u};
                auto edge = [&]() {
                    const uint32_t i = s_list[c][x];
                    from = s_ws[i];
                    wl = s_wl[i];
                    const uint32_t st = s_mark[i];
                    set = region(st, s_end[st]);
                    at = o;
                };
                auto ids = [&]() { q = *reinterpret_cast<gptr<u32x4_e>>(colInd + from + (at < wl ? at : 0u)); };
                if (x < end) {
                    edge();
                    ids();
                }
                while (x < end) {
                    const u32x4 cq = q;
                    const uint32_t left = at < wl ? wl - at : 0u, cfirst = set & 0xffffu, clen = set >> 16;
                    at += 4 * lanes;
                    if (at - o >= wl) {  // the edge is done
                        x += kRowsThreads >> (c + 1);
                        if (x < end) edge();
                    }
                    if (x < end) ids();
                    const uint32_t lo[2] = {cq[0], cq[1]}, hi[2] = {cq[2], cq[3]};
                    h += set_hits(s_tab, lo, left, cfirst, clen);
                    __builtin_amdgcn_sched_barrier(0);
                    h += set_hits(s_tab, hi, left > 2 ? left - 2 : 0u, cfirst, clen);
                }
            }
            // four lanes an edge, two ids each a step, their halvings side by side
            const uint2 rare = *reinterpret_cast<const uint2 *>(&s_n[buf][kRare]);
            const uint32_t few = uni32(rare.x), rest = uni32(rare.y);
            if (few) {
                for (uint32_t x = (kRowsThreads - 1 - threadIdx.x) >> 2; x < few; x += kRowsThreads >> 2) {
                    const uint32_t i = s_list[kSearch][x], wl = s_wl[i], end = s_end[s_mark[i]];
                    const OffT from = s_ws[i];
                    for (uint32_t q = i + 1 + (lane & 3u); q < end; q += 8) {
                        const uint32_t y0 = colInd[cp0 + q], y1 = q + 4 < end ? colInd[cp0 + q + 4] : y0;
                        OffT at0 = from, at1 = from;  // the last id <= y, or the first id
                        for (uint32_t k = wl; k > 1;) {
                            const uint32_t half = k >> 1;
                            const uint32_t v0 = colInd[at0 + half], v1 = colInd[at1 + half];
                            at0 = v0 <= y0 ? at0 + half : at0;
                            at1 = v1 <= y1 ? at1 + half : at1;
                            k -= half;
                        }
                        h += colInd[at0] == y0 ? 1u : 0u;
                        h += q + 4 < end && colInd[at1] == y1 ? 1u : 0u;
                    }
                }
            }
            uint64_t end = 0;
            if (rest) {  // block-uniform: the last row is not hashed
                const uint32_t r = wave_rightmost_le(n - 1, cp0 + st_last, [&](uint32_t y) { return (uint64_t)rowPtr[y]; });
                end = rowPtr[(uint64_t)r + 1];
            }
            for (uint32_t x = wv; x < rest; x += kRowsWaves) {  // adj+(w) and v's row after w: the shorter in the longer
                const uint32_t i = s_list[kUnhashed][x];
                const uint64_t w0 = s_ws[i], v0 = cp0 + i + 1, wl = s_wl[i], vl = end - v0;
                const uint64_t from = wl < vl ? w0 : v0, in = wl < vl ? v0 : w0;
                const uint64_t ids = wl < vl ? wl : vl, top = in + (wl < vl ? vl : wl);
                for (uint64_t at = lane; at < ids; at += kWave) {
                    const uint32_t y = colInd[from + at];
                    uint64_t lo = in, hi = top;
                    while (lo < hi) {
                        const uint64_t mid = lo + ((hi - lo) >> 1);
                        if (colInd[mid] < y) lo = mid + 1;
                        else hi = mid;
                    }
                    h += lo < top && colInd[lo] == y ? 1u : 0u;
                }
            }
            hits += h;
        }
    }
    if (cur_g != kSentinel) flush();  // block-uniform
    wedges = block_sum(wedges);
    if (threadIdx.x == 0 && wedges) line_add(lines, kLineWedges, wedges);
}

// ---------------------------------------------------------------- launches

hipError_t rows_grid(int ob, int num_cus, uint32_t *grid) {
    int per_cu = 0;
    const hipError_t e = ob == 8 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_rows<uint64_t>, kRowsThreads, 0)
                                 : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_rows<uint32_t>, kRowsThreads, 0);
    if (e != hipSuccess) return e;
    *grid = (uint32_t)(per_cu < 1 ? 1 : per_cu) * (uint32_t)(num_cus > 0 ? num_cus : 1);
    return hipSuccess;
}

// Half tiles where they fit one turn of the grid: R-MAT-12 36 against 40 us,
// R-MAT-13 40 against 43; quarter tiles cost R-MAT-13 6 us, and R-MAT-16 in
// three even turns of 395 edges takes 117 us against 109.
uint32_t rows_tile_edges(uint64_t edges, uint32_t grid) { return edges <= 256ull * grid ? kRowsTileMin : kRowsTile; }

hipError_t launch_rows(const uint64_t *host_desc, GraphDesc *desc, uint32_t G, int ob, uint64_t tiles, uint32_t tile_edges,
                       uint64_t *meta, unsigned long long *counts, uint64_t *lines, uint32_t grid,
                       hipStream_t st) {
    if (G == 0 || grid == 0) return hipErrorInvalidValue;
    const uint64_t ib = ((uint64_t)G * (sizeof(GraphDesc) / 8) + kBlock - 1) / kBlock;
    k_rows_init<<<dim3((uint32_t)(ib < 256 ? ib : 256)), dim3(kBlock), 0, st>>>(host_desc, desc, G, meta, counts, lines);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || tiles == 0) return e;
    // up to four tiles in a row, with several turns for every block
    uint64_t group = tiles / (4ull * grid);
    group = group < 1 ? 1 : group > 4 ? 4 : group;
    const uint64_t groups = (tiles + group - 1) / group;
    return WTC_LAUNCH_OFF(ob, k_rows, dim3(groups < grid ? (uint32_t)groups : grid), dim3(kRowsThreads), 0, st, desc, G,
                          tiles, (uint32_t)group, tile_edges, counts, lines);
}

}  // namespace wtc
