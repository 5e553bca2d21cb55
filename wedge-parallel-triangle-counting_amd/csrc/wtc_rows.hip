// wtc_rows.hip -- the row count (counting kernel choice kKernelRows): whole
// graphs, alone or in sets, counted edge by edge against hashed rows.
//
// Every edge v -> w closes |adj+(v) ∩ adj+(w)| triangles: the ids of adj+(w)
// are above w, so this is the intersection of w's row with the tail of v's
// row after w, which the wedge-parallel kernels check wedge by wedge
// (tc.cu:203-287).  A block takes a tile of kRowsTile consecutive positions
// of colInd (edges), hashes the rows of v that they lie in into LDS, streams
// adj+(w) for each of its edges with 16-byte loads, and looks every id up in
// v's set: one 16-byte LDS read an id.  It checks the arrow wedges v -> w -> u
// (1.2 to 4 times as many as the wedges (w, u) of v, more on skewed graphs),
// but needs no wedge prefix, no tile search per wedge, no bitmap and no chain
// of dependent probes: two launches a count, whatever the number of graphs.
//
// Measured against the staged kernel on its tuned shape (whole call): R-MAT-12
// 41 us instead of 146, R-MAT-16 123 instead of 329, R-MAT-18 0.60 ms instead
// of 0.88, Erdos-Renyi n = 10^6 of degree 16 0.26 ms instead of 0.58, 256
// Erdos-Renyi and Barabasi-Albert graphs 1.37 ms instead of 2.83.  Past 2^28
// wedges on skewed graphs the split count is faster (R-MAT-19: 0.93 against
// 1.9 ms).  On flat graphs a tile's chain of loads and barriers bounds it
// (24 waves a CU wait 70% of their cycles), on skewed ones the 20 vector
// instructions of a lookup.
#include "wtc_dev.h"
#include "wtc_kernels.h"
#include "wtc_launch.h"

namespace wtc {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Four ids at any element (4-byte) alignment.
typedef uint32_t u32x4_e __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRowsThreads = 512;
static_assert(kRowsThreads == (int)kRowsTile, "a position per thread");
constexpr uint32_t kRowsWaves = kRowsThreads / kWave;
// Longest row (from its first position in the tile) hashed; the ids of a
// longer one are searched in memory.
constexpr uint32_t kRowsRowMax = 512;
// Buckets of four slots per position: with two, one bucket in 600 is full (a
// lookup that misses in a full one goes on to the next, and some lane of a
// wave's four lookups would in most steps with one).
constexpr uint32_t kRowsSpread = 2;
constexpr uint32_t kRowsBuckets = kRowsSpread * (kRowsTile + kRowsRowMax);

// Bucket of id u in a region of len buckets (len < 2^12): twelve bits of u in
// reverse, so that neighbouring ids fall far apart, all in instructions of
// full rate (a 32-bit multiply takes four times as long).
__device__ __forceinline__ uint32_t rows_bucket(uint32_t u, uint32_t len) {
    return __umul24(__builtin_bitreverse32(u ^ (u >> 11)) >> 20, len) >> 12;
}

}  // namespace

// The descriptors from the host's pinned memory, the counts and the wedge
// total zeroed: a kernel, not copies, since two of those cost more than the
// rest of a small graph's count.
__global__ __launch_bounds__(kBlock) void k_rows_init(const uint64_t *__restrict__ host_desc, GraphDesc *__restrict__ desc,
                                                      uint32_t G, uint64_t *__restrict__ meta,
                                                      unsigned long long *__restrict__ counts) {
    static_assert(sizeof(GraphDesc) % 8 == 0, "copied by words");
    const uint64_t step = (uint64_t)gridDim.x * kBlock, at = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (host_desc)
        for (uint64_t i = at; i < (uint64_t)G * (sizeof(GraphDesc) / 8); i += step)
            reinterpret_cast<uint64_t *>(desc)[i] = host_desc[i];
    for (uint64_t i = at; i < G; i += step) counts[i] = 0ull;
    if (at < kMetaSlots) meta[at] = 0ull;
}

// Groups of `group` consecutive tiles of the set (D.tile_base: a graph's first
// tile; D.wcount: its edges) dealt to the blocks in turn.  Per tile:
//  1. the rows of the tile mark their first position and leave their end
//     there, and a running maximum gives every position its row (the first
//     row of a group is found by a 64-way search, later ones from the tile
//     before);
//  2. every position's id w goes into the set of its row v (a row of len
//     positions owns kRowsSpread * len buckets of four slots, one 16-byte LDS
//     read each), the last row's ids past the tile too;
//  3. the edges with an adj+(w) that may meet v's row are listed by the
//     length of adj+(w) and streamed by 2 to 32 lanes each, four ids a lane:
//     up to 64 ids in one step, longer ones 128 at a time; the next step's
//     ids load while this one's are looked up.
// The next tile's rows, ids and bounds of adj+(w) load while a tile is
// streamed.
// (Six waves a SIMD, three blocks a CU, take 80 registers and the lookups two
// at a time; with five 0.30 instead of 0.26 ms on the Erdos-Renyi graph, and
// with eight, spilling, 0.35.)
template <typename OffT>
__global__ __launch_bounds__(kRowsThreads, 6) void k_rows(const GraphDesc *__restrict__ desc, uint32_t G, uint64_t tiles,
                                                       uint32_t group, uint64_t *__restrict__ meta,
                                                       unsigned long long *__restrict__ counts) {
    constexpr uint32_t kT = kRowsTile;
    constexpr uint32_t kLists = 6;  // adj+(w) of up to 8, 16, 32, 64 ids, and more; edges of a row not hashed
    __shared__ __align__(16) uint32_t s_tab[kRowsBuckets * 4];
    __shared__ OffT s_ws[kT];        // start of adj+(w)
    __shared__ uint32_t s_wl[kT];    // its length
    __shared__ uint16_t s_end[kT];   // at a row's first position: its end, from the tile's start (at most 2^16 - 1)
    __shared__ uint16_t s_mark[kT];  // a position's row, as the row's first position
    __shared__ uint16_t s_list[kT];  // the edges to stream, list by list
    __shared__ uint32_t s_n[kLists];
    __shared__ uint32_t s_w[kRowsWaves];
    __shared__ uint64_t s_sum[kRowsWaves];
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    const u32x4 *const tab4 = reinterpret_cast<const u32x4 *>(s_tab);
    uint32_t cur_g = kSentinel;
    uint64_t hits = 0, wedges = 0;
    // the block's hits of graph cur_g into its count
    auto flush = [&]() {
        const uint64_t t = wave_sum(hits);
        if (lane == 0) s_sum[wv] = t;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t all = 0;
            for (uint32_t w = 0; w < kRowsWaves; w++) all += s_sum[w];
            if (all) atomicAdd(&counts[cur_g], (unsigned long long)all);
        }
        __syncthreads();
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
                    g_end = D.tile_base + (m + kT - 1) / kT;
                }
                p0 = (tile - desc[g].tile_base) * kT;
                vb = wave_rightmost_le(n - 1, p0, [&](uint32_t r) { return (uint64_t)rowPtr[r]; });
                load(p0, vb);
                fresh = false;
            }
            const uint32_t nt = m - p0 < kT ? (uint32_t)(m - p0) : kT;
            __syncthreads();  // the previous tile's lookups are done
            s_mark[threadIdx.x] = 0;
            if (threadIdx.x < kLists) s_n[threadIdx.x] = 0u;
            __syncthreads();
            for (;;) {  // windows of rows up to the one holding the tile's last position
                const uint64_t a = ra, z = rz;
                if (z > a && z > p0 && a < p0 + nt) {
                    const uint32_t at = a > p0 ? (uint32_t)(a - p0) : 0u;
                    s_mark[at] = (uint16_t)at;
                    s_end[at] = z - p0 < 0xffffull ? (uint16_t)(z - p0) : (uint16_t)0xffffu;
                    if (a >= p0) wedges += binom2_d(z - a);
                }
                const uint64_t vn = vb + kRowsThreads;
                if (vn >= n || (uint64_t)rowPtr[vn] >= p0 + nt) break;  // block-uniform
                vb = vn;
                ra = rz = 0;
                if (vb + threadIdx.x < n) {
                    ra = rowPtr[vb + threadIdx.x];
                    rz = rowPtr[vb + threadIdx.x + 1];
                }
            }
            __syncthreads();
            {  // running maximum of the marks
                uint32_t run = s_mark[threadIdx.x];
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const uint32_t y = (uint32_t)__shfl_up((int)run, o, kWave);
                    run = (int)lane >= o && y > run ? y : run;
                }
                if (lane == kWave - 1) s_w[wv] = run;
                __syncthreads();
                for (uint32_t w = 0; w < wv; w++) run = s_w[w] > run ? s_w[w] : run;
                s_mark[threadIdx.x] = (uint16_t)run;
            }
            __syncthreads();
            // positions hashed: the tile's rows, the last one to its end, or
            // without it if it is too long (only the last row can be: a row
            // that ends in the tile has at most kT positions there)
            static_assert(kRowsRowMax >= kT, "a row ending in the tile is hashed");
            const uint32_t st_last = s_mark[nt - 1], end_last = s_end[st_last];
            const bool long_last = end_last - st_last > kRowsRowMax;
            const uint32_t bl = long_last ? st_last : end_last;
            for (uint32_t i = threadIdx.x; i < kRowsSpread * bl; i += kRowsThreads)
                reinterpret_cast<uint4 *>(s_tab)[i] = make_uint4(kSentinel, kSentinel, kSentinel, kSentinel);
            // this position's edge: its list and place there
            const uint32_t me = threadIdx.x;
            uint32_t my_list = kSentinel, my_rank = 0;
            const uint32_t my_st = s_mark[me];
            if (me < nt) {
                const uint64_t len = (uint64_t)(we - ws);
                if (len != 0 && me + 1 != s_end[my_st]) {  // else nothing to stream, or nothing after w in v's row
                    s_ws[me] = ws;
                    s_wl[me] = (uint32_t)len;  // < n
                    my_list = len <= 8 ? 0u : len <= 16 ? 1u : len <= 32 ? 2u : len <= 64 ? 3u : 4u;
                    if (long_last && my_st == st_last) my_list = 5u;
                    my_rank = atomicAdd(&s_n[my_list], 1u);
                }
            }
            __syncthreads();
            auto insert = [&](uint32_t st, uint32_t u) {
                const uint32_t first = kRowsSpread * st, len = kRowsSpread * (s_end[st] - st);
                uint32_t bk = first + rows_bucket(u, len);
                for (bool done = false; !done;) {
                    for (uint32_t z = 0; z < 4 && !done; z++)
                        done = atomicCAS(&s_tab[bk * 4 + z], kSentinel, u) == kSentinel;
                    bk = bk + 1 == first + len ? first : bk + 1;
                }
            };
            uint32_t off[kLists + 1];
            off[0] = 0;
#pragma unroll
            for (uint32_t c = 0; c < kLists; c++) off[c + 1] = off[c] + uni32(s_n[c]);
            if (me < nt && me < bl) insert(my_st, id);
            if (my_list != kSentinel) {
                uint32_t o = off[0];
#pragma unroll
                for (uint32_t c = 1; c < kLists; c++) o = my_list == c ? off[c] : o;
                s_list[o + my_rank] = (uint16_t)me;
            }
            for (uint32_t i = nt + threadIdx.x; i < bl; i += kRowsThreads) insert(st_last, colInd[p0 + i]);
            __syncthreads();
            const uint64_t cp0 = p0;
            p0 += kT;
            if (tile + 1 < t1 && tile + 1 < g_end) load(p0, vb);
            uint32_t h = 0;
            uint32_t begin = 0;
            for (uint32_t c = 0; c < 5; c++) {  // list c: 2 << c lanes an edge, four ids each a step
                const uint32_t lanes = 2u << c, o = 4 * (lane & (lanes - 1)), end = begin + uni32(s_n[c]);
                uint32_t x = begin + (threadIdx.x >> (c + 1));
                begin = end;
                // the step ahead: ids of row st at `at` of the wl from ws
                uint32_t at = 0, wl = 0, st = 0;
                OffT from = 0;
                u32x4 q = {0u, 0u, 0u, 0u};
                auto edge = [&]() {
                    const uint32_t i = s_list[x];
                    from = s_ws[i];
                    wl = s_wl[i];
                    st = s_mark[i];
                    at = o;
                };
                auto ids = [&]() { q = *reinterpret_cast<gptr<u32x4_e>>(colInd + from + (at < wl ? at : 0u)); };
                if (x < end) {
                    edge();
                    ids();
                }
                while (x < end) {
                    const u32x4 cq = q;
                    const uint32_t left = at < wl ? wl - at : 0u, cst = st;
                    at += 4 * lanes;
                    if (at - o >= wl) {  // the edge is done
                        x += kRowsThreads >> (c + 1);
                        if (x < end) edge();
                    }
                    if (x < end) ids();
                    const uint32_t first = kRowsSpread * cst, len = kRowsSpread * (s_end[cst] - cst);
                    uint32_t full = 0;
#pragma unroll
                    for (uint32_t z0 = 0; z0 < 4; z0 += 2) {
                        u32x4 t[2];
#pragma unroll
                        for (uint32_t z = 0; z < 2; z++) t[z] = tab4[first + rows_bucket(cq[z0 + z], len)];
#pragma unroll
                        for (uint32_t z = 0; z < 2; z++) {
                            const uint32_t y = cq[z0 + z];
                            const bool f = (t[z][0] == y) | (t[z][1] == y) | (t[z][2] == y) | (t[z][3] == y);
                            const bool in = z0 + z < left;
                            h += (in & f) ? 1u : 0u;
                            full |= (in & !f & (t[z][3] != kSentinel)) ? 1u << (z0 + z) : 0u;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    while (full) {  // a full bucket: on to the next
                        const uint32_t z = (uint32_t)__builtin_ctz(full);
                        full &= full - 1;
                        const uint32_t y = z == 0 ? cq[0] : z == 1 ? cq[1] : z == 2 ? cq[2] : cq[3];
                        uint32_t b2 = first + rows_bucket(y, len);
                        for (;;) {
                            b2 = b2 + 1 == first + len ? first : b2 + 1;
                            const u32x4 w2 = tab4[b2];
                            const bool f2 = (w2[0] == y) | (w2[1] == y) | (w2[2] == y) | (w2[3] == y);
                            h += f2 ? 1u : 0u;
                            if (f2 | (w2[3] == kSentinel)) break;
                        }
                    }
                }
            }
            const uint32_t n5 = uni32(s_n[5]);
            uint64_t end = 0;
            if (n5) {  // block-uniform: the last row is not hashed
                const uint32_t r = wave_rightmost_le(n - 1, cp0 + st_last, [&](uint32_t y) { return (uint64_t)rowPtr[y]; });
                end = rowPtr[(uint64_t)r + 1];
            }
            for (uint32_t x = begin + wv; x < begin + n5; x += kRowsWaves) {  // searched in v's row after w
                const uint32_t i = s_list[x], wl = s_wl[i];
                for (uint32_t at = lane; at < wl; at += kWave) {
                    const uint32_t y = colInd[s_ws[i] + at];
                    uint64_t lo = cp0 + i + 1, hi = end;
                    while (lo < hi) {
                        const uint64_t mid = lo + ((hi - lo) >> 1);
                        if (colInd[mid] < y) lo = mid + 1;
                        else hi = mid;
                    }
                    h += lo < end && colInd[lo] == y ? 1u : 0u;
                }
            }
            hits += h;
        }
    }
    if (cur_g != kSentinel) flush();  // block-uniform
    wedges = wave_sum(wedges);
    if (lane == 0 && wedges) atomicAdd(reinterpret_cast<unsigned long long *>(&meta[kMetaWedges]), (unsigned long long)wedges);
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

hipError_t launch_rows(const uint64_t *host_desc, GraphDesc *desc, uint32_t G, int ob, uint64_t tiles, uint64_t *meta,
                       unsigned long long *counts, uint32_t grid, hipStream_t st) {
    if (G == 0 || grid == 0) return hipErrorInvalidValue;
    const uint64_t ib = ((uint64_t)G * (sizeof(GraphDesc) / 8) + kBlock - 1) / kBlock;
    k_rows_init<<<dim3((uint32_t)(ib < 256 ? ib : 256)), dim3(kBlock), 0, st>>>(host_desc, desc, G, meta, counts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || tiles == 0) return e;
    // up to four tiles in a row, with several turns for every block
    uint64_t group = tiles / (4ull * grid);
    group = group < 1 ? 1 : group > 4 ? 4 : group;
    const uint64_t groups = (tiles + group - 1) / group;
    return WTC_LAUNCH_OFF(ob, k_rows, dim3(groups < grid ? (uint32_t)groups : grid), dim3(kRowsThreads), 0, st, desc, G,
                          tiles, (uint32_t)group, meta, counts);
}

}  // namespace wtc
