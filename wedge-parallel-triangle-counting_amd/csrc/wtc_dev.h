// wtc_dev.h -- device helpers shared by the HIP translation units: binomial
// counts, wave-uniform broadcasts and wave64/block scans.
#pragma once
#include "wtc_kernels.h"

// Launches KERNEL<uint64_t> or KERNEL<uint32_t> by the set's offset width and
// returns the launch status.
#define WTC_LAUNCH_OFF(ob, KERNEL, GRID, BLOCK, SHMEM, STREAM, ...)               \
    [&]() -> hipError_t {                                                         \
        if ((ob) == 8)                                                            \
            KERNEL<uint64_t><<<GRID, BLOCK, SHMEM, STREAM>>>(__VA_ARGS__);        \
        else                                                                      \
            KERNEL<uint32_t><<<GRID, BLOCK, SHMEM, STREAM>>>(__VA_ARGS__);        \
        return hipGetLastError();                                                 \
    }()

namespace wtc {

__device__ __forceinline__ uint64_t binom2_d(uint64_t x) {
    return (x & 1u) ? x * ((x - 1u) >> 1) : (x >> 1) * (x - 1u);
}

// C(x,2) of a 32-bit x: x(x-1) < 2^64, so one 32x32->64 multiply and a shift.
__device__ __forceinline__ uint64_t binom2_u32(uint32_t x) { return ((uint64_t)x * (uint64_t)(x - 1u)) >> 1; }

// The top-a bitmap (tc.cu:262-272, 329-346) as a square a x a bit matrix over
// the ranks [thr, thr + a), row-major in 32-bit words (a is a multiple of 32,
// so every row starts on a word boundary): the bit of (w, u) is bit
// (u - thr) % 32 of word (w - thr) * a/32 + (u - thr) / 32.  Only the strict
// upper triangle u > w is ever set or read.  a32 = a/32.
__device__ __forceinline__ uint64_t bm_word(uint32_t w, uint32_t u, uint32_t thr, uint32_t a32) {
    return (uint64_t)(w - thr) * a32 + ((u - thr) >> 5);
}
__device__ __forceinline__ uint32_t bm_test(const uint32_t *__restrict__ bitmap, uint32_t w, uint32_t u,
                                            uint32_t thr, uint32_t a32) {
    return (bitmap[bm_word(w, u, thr, a32)] >> ((u - thr) & 31u)) & 1u;
}

__device__ __forceinline__ uint32_t uni32(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// The lane-read builtins return int: each 32-bit half goes back through
// uint32_t before it is widened, so the low half is never sign-extended.
__device__ __forceinline__ uint64_t uni64(uint64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32));
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t uni(uint32_t x) { return uni32(x); }
__device__ __forceinline__ uint64_t uni(uint64_t x) { return uni64(x); }

// Value of x in lane `src`, which must be the same in every lane.
__device__ __forceinline__ uint64_t readlane_u64(uint64_t x, uint32_t src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, (int)src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), (int)src);
    return ((uint64_t)hi << 32) | lo;
}

// Value of x in lane src (ds_bpermute), for 64- and 32-bit values; every
// lane of the wave must execute it.
__device__ __forceinline__ uint64_t shfl_u64(uint64_t x, uint32_t src) {
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)x, (int)src, kWave);
    const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(x >> 32), (int)src, kWave);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint32_t shfl_off(uint32_t x, uint32_t src) {
    return (uint32_t)__shfl((int)x, (int)src, kWave);
}
__device__ __forceinline__ uint64_t shfl_off(uint64_t x, uint32_t src) { return shfl_u64(x, src); }
// Value of x in lane (lane - d), or the lane's own x for lanes below d.
__device__ __forceinline__ uint64_t shfl_up_u64(uint64_t x, int d) {
    const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)x, d, kWave);
    const uint32_t hi = (uint32_t)__shfl_up((int)(uint32_t)(x >> 32), d, kWave);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t wave_incl_scan(uint64_t x) {
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        uint64_t y = __shfl_up(x, (unsigned)o, kWave);
        if (lane >= o) x += y;
    }
    return x;
}

__device__ __forceinline__ uint64_t wave_sum(uint64_t x) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, kWave);
    return x;
}

// Exclusive scan over the 256 lanes of a block; s_tot holds 4 wave totals.
__device__ __forceinline__ uint64_t block_excl_scan(uint64_t x, uint64_t *s_tot, uint64_t &total) {
    const uint64_t inc = wave_incl_scan(x);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_tot[w] = inc;
    __syncthreads();
    uint64_t off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kWavesPerBlock; i++) {
        const uint64_t t = s_tot[i];
        off += (i < w) ? t : 0;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return off + inc - x;
}

// Exclusive prefix over the kScanChunk values of a block, from `carry` on: in
// each of four rounds a thread holds four neighbours, x[4 r .. 4 r + 3] being
// values (r * kBlock + thread) * 4 of the block; one barrier in all (sixteen
// rounds of one value each took 15 us a block, this 6).  Returns carry and the
// block's values summed.
constexpr int kScanRounds = kScanItems / 4;
__device__ __forceinline__ uint64_t chunk_scan(uint64_t (&x)[kScanItems], uint64_t carry,
                                               uint64_t (*s_tot)[kWavesPerBlock]) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x >> 6;
    uint64_t sum[kScanRounds], inc[kScanRounds];
#pragma unroll
    for (int r = 0; r < kScanRounds; r++) {
        sum[r] = x[4 * r] + x[4 * r + 1] + x[4 * r + 2] + x[4 * r + 3];
        inc[r] = wave_incl_scan(sum[r]);
        if (lane == kWave - 1) s_tot[r][wv] = inc[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kScanRounds; r++) {
        uint64_t at = carry + inc[r] - sum[r];
        for (uint32_t w = 0; w < (uint32_t)kWavesPerBlock; w++) {
            at += w < wv ? s_tot[r][w] : 0;
            carry += s_tot[r][w];
        }
#pragma unroll
        for (int z = 0; z < 4; z++) {
            const uint64_t y = x[4 * r + z];
            x[4 * r + z] = at;
            at += y;
        }
    }
    return carry;
}

// Value 4 r + z of a thread in a chunk_scan, from the block's first.
__device__ __forceinline__ uint64_t chunk_at(int r, int z) { return ((uint64_t)r * kBlock + threadIdx.x) * 4 + z; }

// Global-memory views of the CSR, prefix and bitmap arrays.  Their pointers
// are read from descriptors in memory, so without the cast the compiler must
// treat them as generic addresses: flat loads, which also count against the
// LDS counter and make every wait cover the LDS traffic too.
template <class T>
using gptr = const __attribute__((address_space(1))) T *;
template <class T>
__device__ __forceinline__ gptr<T> to_global(const T *p) {
    return (gptr<T>)p;
}
// Constant-address-space views of the same read-only arrays, for reads whose
// address is wave-uniform: they become scalar loads into SGPRs, so the
// arithmetic that follows stays on the scalar unit.
template <class T>
using cptr = const __attribute__((address_space(4))) T *;
template <class T>
__device__ __forceinline__ cptr<T> to_const(const T *p) {
    return (cptr<T>)p;
}

// Rightmost v in [lo, hi] with ws[v] <= t, given ws[lo] <= t.  Called with
// wave-uniform arguments (scalar loads) and per lane (vector loads).
template <class P>
__device__ __forceinline__ uint32_t rightmost_le(P ws, uint32_t lo, uint32_t hi, uint64_t t) {
    uint32_t s = lo + 1, e = hi + 1;
    while (s < e) {
        const uint32_t mid = s + ((e - s) >> 1);
        if (ws[mid] <= t) s = mid + 1;
        else e = mid;
    }
    return s - 1;
}

// Adds x to word `word` of the block's sum line.
__device__ __forceinline__ void line_add(uint64_t *lines, uint32_t word, uint64_t x) {
    atomicAdd(reinterpret_cast<unsigned long long *>(&lines[(blockIdx.x % kSumLines) * kLineWords + word]),
              (unsigned long long)x);
}

// The next tile of `of` counters at line `first`, for one thread of a block
// (a counter for each block at most: every one needs blocks).
__device__ __forceinline__ uint64_t line_tile(uint64_t *lines, uint32_t first, uint32_t of) {
    of = of < gridDim.x ? of : gridDim.x;
    const uint32_t c = blockIdx.x % of;
    return c + of * atomicAdd(reinterpret_cast<unsigned long long *>(&lines[(first + c) * kLineWords]), 1ull);
}

// Rightmost r in [0, hi] with f(r) <= t for a non-decreasing f with f(0) <=
// t, by a whole wave: 64 probes a round.
template <class F>
__device__ __forceinline__ uint32_t wave_rightmost_le(uint32_t hi, uint64_t t, F f) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t lo = 0;  // f(lo) <= t
    while (lo < hi) {
        const uint32_t step = (hi - lo - 1) / kWave + 1;
        const uint64_t at = (uint64_t)lo + (uint64_t)(lane + 1) * step;
        const bool le = at <= hi && f((uint32_t)at) <= t;
        const uint32_t k = (uint32_t)__builtin_popcountll(__ballot(le));  // a prefix of the lanes
        const uint64_t end = (uint64_t)lo + (uint64_t)(k + 1) * step - 1;
        lo += k * step;
        hi = end < hi ? (uint32_t)end : hi;
    }
    return uni32(lo);
}

}  // namespace wtc
