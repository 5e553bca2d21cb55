// wtc_dense.hip -- the dense part of a count: the wedges among the top ranks
// of a degree-ordered graph, counted as a product of bit matrices on the
// matrix cores.
//
// Degree order gathers the neighbours of the vertices with many wedges in
// the last ranks: the rows of R-MAT-24's top 16,384 ranks hold 7% or more of
// all columns there.  For a vertex v let cnt of its cnt ids of largest rank
// lie in the last K ranks.  Its C(cnt, 2) wedges (v; w, u) there close
//     sum over w of B[v][w] * (sum over u of B[v][u] * R[w][u])
// triangles, with B[v] the row of v and R[w] = adj+(w) as bits over the last
// K ranks: a product of the matrix of the chosen rows with R, masked by the
// rows themselves.  It checks every pair (w, u) instead of the wedges, K^2/2
// multiply-adds per row, but the matrix cores do those at 3.1e15 a second
// (R-MAT-24: 6.4e12 in 2.04 ms, 62% of the 4-bit peak), against 1 to 2.5e12
// wedges a second of the probing kernels, so a row with cnt / K of a few
// percent is counted faster this way, and its in-edges there are not grouped
// at all.  R-MAT-24: 45% of the wedges and 22% of the in-edges; the row
// kernel 16.2 -> 10.3 ms, the transposition 5.3 -> 4.2 ms, the count 24.7 ->
// 20.4 ms.  Bound by the matrix instructions and the vector instructions that
// spread the bits to operands beside them.
//
//   k_dense_class  per vertex, the class (K = kDenseCore0 << q columns) that
//                  saves most by the cost model below, or none; the chosen
//                  vertices are listed by class, and every vertex's in-edges
//                  left to the other kernels are counted
//   k_dense_rows   R and the listed rows B as bits
//   k_dense_mm     the masked product
//
// Columns are counted from the top: column c is the rank n - 1 - c, so R's
// row c has bits only at columns below c and R's first K rows and columns
// are the core of every class with at most K columns.
//
// Layout of both matrices: tiles of 32 rows by 256 columns, 1 KB each, the
// 16 bytes of lane l of a tile being the words 4*(l / 32) .. +3 (of the
// tile's 8 words a row) of row l % 32.  One 16-byte load per lane then
// brings the operand bits of four matrix instructions of 32 rows by 64
// columns, and a word is the lane's 32 values of one of them.
#include "wtc_dev.h"
#include "wtc_kernels.h"
#include "wtc_launch.h"

namespace wtc {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Byte offset within a 32-row matrix of `kb` tiles a row block of the word
// holding column c of row r (r < 32).
__device__ __forceinline__ uint32_t tile_word(uint32_t r, uint32_t c) {
    const uint32_t w = (c >> 5) & 7u;
    return ((c >> 8) * 64u + (r + 32u * (w >> 2))) * 4u + (w & 3u);
}

// Rows of the class lists are padded to this many (a wave of the product
// takes kDenseRows rows).
constexpr uint32_t kDenseRows = 128;

__device__ __forceinline__ uint32_t dense_cols(uint32_t q) { return kDenseCore0 << q; }

// First tile of class q's rows: the classes one after another, each padded
// to kDenseRows rows.
__device__ __forceinline__ uint64_t dense_base(const uint32_t *cnt, uint32_t q) {
    uint64_t t = 0;
    for (uint32_t p = 0; p < q; p++)
        t += (uint64_t)((cnt[p] + kDenseRows - 1) / kDenseRows) * (kDenseRows / 32) * (dense_cols(p) >> 8);
    return t;
}

}  // namespace

// Zeroes the counters of a split count and the nblocks sums of part_in.
__global__ __launch_bounds__(kBlock) void k_dense_init(const DenseDesc *__restrict__ dd, uint64_t *__restrict__ part_in,
                                                       uint32_t nblocks, unsigned long long *__restrict__ counts,
                                                       uint64_t *__restrict__ lines) {
    const DenseDesc &N = dd[0];
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < nblocks; i += gridDim.x * kBlock) part_in[i] = 0ull;
    if (blockIdx.x != 0) return;
    if (threadIdx.x < kDenseClasses) N.cnt[threadIdx.x] = 0u;
    if (threadIdx.x < kDenseSums) N.sums[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) counts[0] = 0ull;
    for (uint32_t i = threadIdx.x; i < kLines * kLineWords; i += kBlock) lines[i] = 0ull;
}

// A thread takes a vertex (the rows worth a class lie together at the last
// ranks, so blocks are small, to spread them).  For a vertex of the counted
// range whose tail no end of the range clips, the ids in the last K ranks are
// counted for every class by binary searches of its row, all classes'
// searches in step so that their loads overlap (one load per class tells most
// rows off first); the class kept is the one with the largest
//     edge * (cnt - 1) + wedge * C(cnt, 2) - min(K, n - v)^2 / 2,
// edge and wedge being what one in-edge and one wedge cost elsewhere, in
// multiply-adds.  A row needs cnt >= K / kDenseSparsest too: its bits then
// take no more bytes than its ids, which bounds the matrix by 4 bytes an
// edge.  part_in[], zeroed before, gets the in-edges left by prefix block.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void k_dense_class(const GraphDesc *__restrict__ desc,
                                                        const SplitDesc *__restrict__ sd,
                                                        const DenseDesc *__restrict__ dd,
                                                        uint64_t *__restrict__ part_in) {
    __shared__ uint32_t s_cnt[kDenseClasses], s_base[kDenseClasses];
    __shared__ uint64_t s_w[kWavesPerBlock][4];
    static_assert(kScanChunk % kBlock == 0, "a block's vertices are in one prefix block");
    const GraphDesc &D = desc[0];
    const SplitDesc &S = sd[0];
    const DenseDesc &N = dd[0];
    const gptr<OffT> rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const uint32_t n = D.n, thr = D.thr, nq = N.classes;
    const bool clip = S.clip != 0;
    const uint32_t v_lo = S.v_lo, v_hi = S.v_hi;
    if (threadIdx.x < kDenseClasses) s_cnt[threadIdx.x] = 0u;
    __syncthreads();
    const uint64_t blk = (uint64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const uint64_t v = blk * kBlock + threadIdx.x;
    uint32_t cls = kSentinel, num = 0, pos = 0;
    uint64_t left = 0, dense_top = 0, dense_topw = 0, dense_all = 0;
    if (v < n) {
        const OffT s = rowPtr[v], e = rowPtr[v + 1];
        const uint64_t d = (uint64_t)(e - s);
        left = d ? d - 1 : 0;
        if (d >= kDenseCore0 / kDenseSparsest && (!clip || (v > v_lo && v < v_hi))) {
            // a class takes the row if its id K / kDenseSparsest from the end
            // is in the class's columns; then cnt = e - lower_bound(n - K)
            uint32_t x[kDenseClasses];
#pragma unroll
            for (uint32_t q = 0; q < kDenseClasses; q++) {
                const uint32_t least = dense_cols(q) / kDenseSparsest;
                x[q] = q < nq && d >= least ? colInd[e - least] : 0u;
            }
            OffT lb[kDenseClasses];
            uint32_t len[kDenseClasses];
            uint32_t more = 0, fits = 0;
#pragma unroll
            for (uint32_t q = 0; q < kDenseClasses; q++) {
                const uint32_t K = dense_cols(q), least = K / kDenseSparsest;
                const bool fit = q < nq && d >= least && x[q] >= (n > K ? n - K : 0u);
                fits |= fit ? 1u << q : 0u;
                len[q] = fit ? (uint32_t)(d < K ? d : K) - least : 0u;  // [e - min(d, K), e - least)
                lb[q] = e - (OffT)(len[q] + least);
                more |= len[q];
            }
            while (more) {
#pragma unroll
                for (uint32_t q = 0; q < kDenseClasses; q++)
                    if (len[q]) x[q] = colInd[lb[q] + (len[q] >> 1)];
                more = 0;
#pragma unroll
                for (uint32_t q = 0; q < kDenseClasses; q++) {
                    const uint32_t K = dense_cols(q), first = n > K ? n - K : 0u, half = len[q] >> 1;
                    if (len[q]) {
                        const bool lt = x[q] < first;
                        lb[q] += lt ? (OffT)(half + 1) : (OffT)0;
                        len[q] = lt ? len[q] - half - 1 : half;
                    }
                    more |= len[q];
                }
            }
            float best = 0.0f;
            const float dv = (float)(n - (uint32_t)v);
#pragma unroll
            for (uint32_t q = 0; q < kDenseClasses; q++) {
                const uint32_t K = dense_cols(q), c = (uint32_t)(e - lb[q]);
                if (!(fits >> q & 1u)) continue;
                const float fk = fminf((float)K, dv), fc = (float)c;
                const float gain = N.edge * (fc - 1.0f) + N.wedge * 0.5f * fc * (fc - 1.0f) - 0.5f * fk * fk;
                if (gain > best) {
                    best = gain;
                    cls = q;
                    num = c;
                }
            }
            if (cls != kSentinel) {
                left = d - num;
                // the dense wedges' share whose middle vertex is a top row
                OffT a = e - (OffT)num, z = e;
                if (colInd[a] >= thr) z = a;
                while (a < z) {
                    const OffT mid = a + ((z - a) >> 1);
                    if (colInd[mid] < thr) a = mid + 1;
                    else z = mid;
                }
                const uint64_t t = (uint64_t)(e - a);
                dense_top = t ? t - 1 : 0;
                dense_topw = binom2_d(t);
                dense_all = (uint64_t)num - 1;
                pos = atomicAdd(&s_cnt[cls], 1u);
            }
        }
        S.ie_pre[v] = left;
    }
    __syncthreads();
    if (threadIdx.x < kDenseClasses && s_cnt[threadIdx.x])
        s_base[threadIdx.x] = atomicAdd(&N.cnt[threadIdx.x], s_cnt[threadIdx.x]);
    __syncthreads();
    if (cls != kSentinel) N.list[N.list_off[cls] + s_base[cls] + pos] = make_uint2((uint32_t)v, num);
    left = wave_sum(left);
    if (__ballot(cls != kSentinel)) {
        dense_top = wave_sum(dense_top);
        dense_topw = wave_sum(dense_topw);
        dense_all = wave_sum(dense_all);
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        uint64_t *x = s_w[threadIdx.x >> 6];
        x[0] = left;
        x[1] = dense_top;
        x[2] = dense_topw;
        x[3] = dense_all;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        uint64_t t = 0;
        for (int w = 0; w < kWavesPerBlock; w++) t += s_w[w][threadIdx.x];
        uint64_t *to = threadIdx.x == 0 ? &part_in[blk * kBlock / kScanChunk] : &N.sums[threadIdx.x - 1];
        if (t) atomicAdd(reinterpret_cast<unsigned long long *>(to), (unsigned long long)t);
    }
}

// Threads of a block of k_dense_rows.
constexpr int kRowsThreads = 512;

// The rows of classes [q0, q1) (padded rows are zero), after R's when core is
// set.  A block takes one 32-row block at a time, sets its bits in LDS and
// writes its tiles out.  R's row block rb has bits in its first rb / 8 + 1
// tiles only; R is built up to the largest class in use.  Short classes go
// in a launch of their own, with less LDS a block.
template <typename OffT>
__global__ __launch_bounds__(kRowsThreads) void k_dense_rows(const GraphDesc *__restrict__ desc,
                                                       const DenseDesc *__restrict__ dd, uint32_t q0, uint32_t q1,
                                                       bool with_core) {
    extern __shared__ __align__(16) uint32_t s_rows[];
    const GraphDesc &D = desc[0];
    const DenseDesc &N = dd[0];
    const gptr<OffT> rowPtr = to_global(static_cast<const OffT *>(D.rowPtr));
    const gptr<uint32_t> colInd = to_global(D.colInd);
    const uint32_t n = D.n, nq = N.classes;
    uint32_t cnt[kDenseClasses], top = 0, items = 0;
    for (uint32_t q = 0; q < kDenseClasses; q++) {
        cnt[q] = q < nq ? N.cnt[q] : 0u;
        if (cnt[q]) top = dense_cols(q);
    }
    const uint32_t r_items = with_core ? top / 32 : 0u;
    items = r_items;
    if (q1 > nq) q1 = nq;
    for (uint32_t q = q0; q < q1; q++) items += (cnt[q] + kDenseRows - 1) / kDenseRows * (kDenseRows / 32);
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    for (uint32_t it = blockIdx.x; it < items; it += gridDim.x) {
        uint32_t q = 0, rb = 0, tiles;
        u32x4 *dst;
        const bool core = it < r_items;
        if (core) {
            rb = r_items - 1 - it;  // the longest first
            tiles = (rb >> 3) + 1;
            dst = static_cast<u32x4 *>(N.R) + (uint64_t)rb * (N.core >> 8) * 64;
        } else {
            rb = it - r_items;
            for (q = q0; q < q1; q++) {
                const uint32_t b = (cnt[q] + kDenseRows - 1) / kDenseRows * (kDenseRows / 32);
                if (rb < b) break;
                rb -= b;
            }
            tiles = dense_cols(q) >> 8;
            dst = static_cast<u32x4 *>(N.B) + (dense_base(cnt, q) + (uint64_t)rb * tiles) * 64;
        }
        __syncthreads();  // the previous tiles are written out
        for (uint32_t i = threadIdx.x; i < tiles * 64; i += kRowsThreads)
            reinterpret_cast<uint4 *>(s_rows)[i] = make_uint4(0u, 0u, 0u, 0u);
        // this wave's rows: bounds in its first lanes, then one row at a time
        constexpr uint32_t kRows = 32 / (kRowsThreads / kWave);
        OffT b = 0, e = 0;
        if (lane < kRows) {
            const uint32_t r = rb * 32 + wv * kRows + lane;
            if (core) {
                if (r < n) {
                    b = rowPtr[n - 1 - r];
                    e = rowPtr[n - r];
                }
            } else if (r < cnt[q]) {
                const uint2 x = N.list[N.list_off[q] + r];
                e = rowPtr[x.x + 1];
                b = e - (OffT)x.y;
            }
        }
        __syncthreads();
        for (uint32_t k = 0; k < kRows; k++) {
            const OffT rb0 = (OffT)readlane_u64((uint64_t)b, k), re = (OffT)readlane_u64((uint64_t)e, k);
            // by the number of the id in the row: a position past a row's end
            // may pass 2^32
            const uint32_t len = (uint32_t)(re - rb0);
            for (uint32_t i = lane; i < len; i += 8 * kWave) {  // eight loads in flight
                uint32_t u[8];
#pragma unroll
                for (uint32_t z = 0; z < 8; z++) u[z] = i + z * kWave < len ? colInd[rb0 + (OffT)(i + z * kWave)] : kSentinel;
#pragma unroll
                for (uint32_t z = 0; z < 8; z++) {
                    if (u[z] == kSentinel) continue;
                    const uint32_t c = n - 1 - u[z];
                    atomicOr(&s_rows[tile_word(wv * kRows + k, c)], 1u << (c & 31u));
                }
            }
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < tiles * 64; i += kRowsThreads) dst[i] = reinterpret_cast<u32x4 *>(s_rows)[i];
    }
}

// The 32 values of a lane's operand, 4 bits each (e2m1: 1, 2, 4 are 0.5,
// 1.0, 2.0), from 32 bits: bit 4 i + j of x becomes value i of word j, an
// order of the summed index that both operands share.  The bits stay where
// they are as far as they can, so that the two operands' values for the same
// bit multiply to 1: 0.5 and 2.0 for j = 0, 2.0 and 0.5 for j = 2.
__device__ __forceinline__ i32x8 dense_operand_v(uint32_t x) {
    i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
    r[0] = (int)(x & 0x11111111u);
    r[1] = (int)(x & 0x22222222u);
    r[2] = (int)(x & 0x44444444u);
    r[3] = (int)((x >> 2) & 0x22222222u);
    return r;
}
__device__ __forceinline__ i32x8 dense_operand_w(uint32_t x) {
    i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
    r[0] = (int)((x << 2) & 0x44444444u);
    r[1] = (int)(x & 0x22222222u);
    r[2] = (int)((x >> 2) & 0x11111111u);
    r[3] = (int)((x >> 2) & 0x22222222u);
    return r;
}

// Units of 256 core rows w by kDenseRows rows v, classes with many columns and
// core rows far from the top (the longest sums) first, dealt to the blocks in
// turn; each of a block's four waves takes 64 of the core rows.  A wave loads
// the bits of its rows tile by tile straight from memory, the next tile while
// the current one is multiplied: operands are bits until they are in
// registers, so a tile of 256 columns costs six 16-byte loads per lane (the
// four of B shared by the waves through the CU's cache) for 32 matrix
// instructions and needs no LDS.  A unit's last tile loads the next unit's
// first one and its mask: with units from a counter, whose loads began after
// it answered, R-MAT-18 and 20, whose units are one to sixteen tiles long,
// took 52 and 109 us instead of 36 and 79.  Waves without a bit B[v][w] have nothing to do.
// Counts are exact: the sums are whole numbers up to 2^15 in 32-bit floats, a
// unit's total per lane below 2^22.
__global__ __launch_bounds__(kBlock, 2) void k_dense_mm(const DenseDesc *__restrict__ dd,
                                                        uint64_t *__restrict__ lines) {
    const DenseDesc &N = dd[0];
    const uint32_t nq = N.classes, lane = threadIdx.x & (kWave - 1), wv = uni32(threadIdx.x >> 6);
    static_assert(kWavesPerBlock == 4, "a wave per 64 of a unit's 256 core rows");
    uint32_t nv[kDenseClasses];    // row tiles
    uint64_t first[kDenseClasses];  // first tile of the rows
    uint64_t units = 0, at = 0;
#pragma unroll
    for (uint32_t q = 0; q < kDenseClasses; q++) {
        nv[q] = q < nq ? (uni32(N.cnt[q]) + kDenseRows - 1) / kDenseRows : 0u;
        first[q] = at;
        at += (uint64_t)nv[q] * (kDenseRows / 32) * (dense_cols(q) >> 8);
        units += (uint64_t)nv[q] * (dense_cols(q) >> 8);
    }
    const gptr<u32x4> R = to_global(static_cast<const u32x4 *>(N.R)) + lane;
    const gptr<u32x4> Bs = to_global(static_cast<const u32x4 *>(N.B)) + lane;
    const uint32_t r_tiles = N.core >> 8;
    // unit u's operands: this wave's core rows A, the row tile B of b_tiles
    // tiles a row block, its group wg of core rows
    auto unit = [&](uint64_t u, gptr<u32x4> &A, gptr<u32x4> &B, uint32_t &b_tiles, uint32_t &wg) {
        uint32_t vt = 0;
        uint64_t row0 = 0;
        bool found = false;
        b_tiles = 1;
        wg = 0;
#pragma unroll
        for (int q = (int)kDenseClasses - 1; q >= 0; q--) {
            const uint32_t t = dense_cols((uint32_t)q) >> 8;
            const uint64_t here = (uint64_t)nv[q] * t;
            if (!found && u < here) {
                found = true;
                b_tiles = t;
                wg = t - 1 - (uint32_t)u / nv[q];
                vt = (uint32_t)u % nv[q];
                row0 = first[q];
            }
            if (!found) u -= here;
        }
        A = R + (uint64_t)(wg * 8 + wv * 2) * r_tiles * 64;
        B = Bs + (row0 + (uint64_t)vt * (kDenseRows / 32) * b_tiles) * 64;
    };
    // the mask words of a unit: rows v = lane % 32 of four row blocks, this
    // wave's two blocks of core rows
    auto mask = [&](gptr<u32x4> B, uint32_t b_tiles, uint32_t wg, uint32_t (&m)[2][4]) {
#pragma unroll
        for (uint32_t a = 0; a < 2; a++) {
            const uint32_t w = wv * 2 + a;
#pragma unroll
            for (uint32_t b = 0; b < 4; b++) {
                const gptr<uint32_t> p = reinterpret_cast<gptr<uint32_t>>(B - lane + ((uint64_t)b * b_tiles + wg) * 64);
                m[a][b] = p[((lane & 31u) + 32u * (w >> 2)) * 4u + (w & 3u)];
            }
        }
    };
    uint64_t u = blockIdx.x;
    if (u >= units) return;
    gptr<u32x4> A, B;
    uint32_t b_tiles, wg;
    unit(u, A, B, b_tiles, wg);
    uint32_t m[2][4];
    mask(B, b_tiles, wg, m);
    u32x4 xa[2], xb[4];
#pragma unroll
    for (uint32_t a = 0; a < 2; a++) xa[a] = A[(uint64_t)a * r_tiles * 64];
#pragma unroll
    for (uint32_t b = 0; b < 4; b++) xb[b] = B[(uint64_t)b * b_tiles * 64];
    uint64_t total = 0;
    for (;;) {
        u += gridDim.x;
        // the next unit (this one again at the end: loaded, not used)
        gptr<u32x4> nA = A, nB = B;
        uint32_t nb_tiles = b_tiles, nwg = wg;
        if (u < units) unit(u, nA, nB, nb_tiles, nwg);
        uint32_t any = 0;
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) any |= m[a][b];
        const bool work = __ballot(any != 0) != 0;  // wave-uniform
        uint32_t cm[2][4];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) cm[a][b] = m[a][b];
        if (work) {
            f32x16 acc[2][4];
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 4; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
            gptr<u32x4> pa = A, pb = B;
            uint32_t sb = b_tiles;
            for (uint32_t kb = 0; kb <= wg; kb++) {  // R's rows w have bits up to column w
                pa += 64;
                pb += 64;
                if (kb == wg) {  // on to the next unit
                    pa = nA;
                    pb = nB;
                    sb = nb_tiles;
                    mask(nB, nb_tiles, nwg, m);
                }
                u32x4 ya[2], yb[4];
#pragma unroll
                for (uint32_t a = 0; a < 2; a++) ya[a] = pa[(uint64_t)a * r_tiles * 64];
#pragma unroll
                for (uint32_t b = 0; b < 4; b++) yb[b] = pb[(uint64_t)b * sb * 64];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    i32x8 oa[2];
#pragma unroll
                    for (int a = 0; a < 2; a++) oa[a] = dense_operand_w(xa[a][s]);
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        const i32x8 ob = dense_operand_v(xb[b][s]);
#pragma unroll
                        for (int a = 0; a < 2; a++)
                            acc[a][b] =
                                __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(oa[a], ob, acc[a][b], 4, 4, 0, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int a = 0; a < 2; a++) xa[a] = ya[a];
#pragma unroll
                for (int b = 0; b < 4; b++) xb[b] = yb[b];
            }
            // lane l holds column v = l % 32 and rows w = 8 (r / 4) + 4 (l / 32) + r % 4 of each block
            float sum = 0.0f;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const uint32_t mm = cm[a][b] >> (4u * (lane >> 5));
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int bit = 8 * (r >> 2) + (r & 3);
                        const int keep = ((int)(mm << (31 - bit))) >> 31;
                        sum += __int_as_float(__float_as_int(acc[a][b][r]) & keep);
                    }
                }
            total += (uint64_t)(uint32_t)sum;
        } else {
            mask(nB, nb_tiles, nwg, m);
#pragma unroll
            for (uint32_t a = 0; a < 2; a++) xa[a] = nA[(uint64_t)a * r_tiles * 64];
#pragma unroll
            for (uint32_t b = 0; b < 4; b++) xb[b] = nB[(uint64_t)b * nb_tiles * 64];
        }
        if (u >= units) break;  // block-uniform
        A = nA;
        B = nB;
        b_tiles = nb_tiles;
        wg = nwg;
        __syncthreads();  // the waves stay near each other, for the cache
    }
    total = wave_sum(total);
    if (lane == 0 && total) line_add(lines, kLineHits, total);
}

// ---------------------------------------------------------------- launches

hipError_t launch_dense_class(const GraphDesc *desc, const SplitDesc *sd, const DenseDesc *dd, int ob, uint32_t n,
                              uint32_t nblocks, uint64_t *part_in, unsigned long long *counts, uint64_t *lines,
                              hipStream_t st) {
    const uint32_t ib = (nblocks + kBlock - 1) / kBlock;
    k_dense_init<<<dim3(ib < 64 ? ib : 64), dim3(kBlock), 0, st>>>(dd, part_in, nblocks, counts, lines);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // a grid's threads in one direction are below 2^32
    const uint32_t blocks = (uint32_t)(((uint64_t)n + kBlock - 1) / kBlock);
    constexpr uint32_t kX = 1u << 23;
    const dim3 grid(blocks < kX ? blocks : kX, (blocks + kX - 1) / kX);
    return WTC_LAUNCH_OFF(ob, k_dense_class, grid, dim3(kBlock), 0, st, desc, sd, dd, part_in);
}

hipError_t launch_dense_count(const GraphDesc *desc, const DenseDesc *dd, int ob, uint32_t core, int num_cus,
                              uint64_t *lines, hipStream_t st) {
    const uint32_t cus = (uint32_t)(num_cus > 0 ? num_cus : 1);
    // a block's LDS holds 32 rows: 64 KB for 16,384 columns, 8 KB for 2,048
    constexpr uint32_t kShort = 3;
    const uint32_t cols = core < (kDenseCore0 << (kShort - 1)) ? core : kDenseCore0 << (kShort - 1);
    hipError_t e = WTC_LAUNCH_OFF(ob, k_dense_rows, dim3(cus * 4), dim3(kRowsThreads), (size_t)cols * 4, st, desc, dd, 0u, kShort,
                                  core <= cols);
    if (e != hipSuccess) return e;
    if (core > cols) {
        const uint32_t lds = core * 4, per_cu = 163840u / lds < 4u ? 163840u / lds : 4u;
        e = WTC_LAUNCH_OFF(ob, k_dense_rows, dim3(cus * per_cu), dim3(kRowsThreads), lds, st, desc, dd, kShort, kDenseClasses, true);
        if (e != hipSuccess) return e;
    }
    k_dense_mm<<<dim3(cus * 2), dim3(kBlock), 0, st>>>(dd, lines);
    return hipGetLastError();
}

}  // namespace wtc
