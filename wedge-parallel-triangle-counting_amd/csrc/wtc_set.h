// wtc_set.h -- sets of ids in LDS for the slab and row counts: a row of ids
// owns a region of buckets of four slots in a table of words.
#pragma once

#include "wtc_dev.h"
#include "wtc_kernels.h"

namespace wtc {

// Four ids loaded by one 16-byte load.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kSetWays = 4;             // slots per bucket
constexpr uint32_t kSetMore = 0x80000000u;  // on a bucket's last slot: ids of the bucket are in the next, too
// A free slot.  kWide: sets of ids that may need all 32 bits, with none left
// for the mark; every full bucket then sends a lookup on to the next (of buckets
// with one id on average 1.9% are full, 0.4% marked).
template <bool kWide>
constexpr uint32_t kSetFree = kWide ? kSentinel : kSetIdsEnd;

// Bucket of id u in a region of len buckets (len < 2^16): a multiplicative
// hash of u's low 24 bits, in 24-bit multiplications (32-bit ones take four
// times as long, and the compiler makes them of a product that it needs the
// low bits of only).
__device__ __forceinline__ uint32_t set_bucket(uint32_t u, uint32_t len) {
    uint32_t h, b;
    asm("v_mul_u32_u24_e32 %0, %1, %2" : "=v"(h) : "s"(0x9e3779u), "v"(u));
    asm("v_mul_hi_u32_u24_e32 %0, %1, %2" : "=v"(b) : "v"(h), "v"(len << 8));
    return b;
}

// Id u into the region of len buckets at `first` (free slots kSetFree).
template <bool kWide = false>
__device__ __forceinline__ void set_insert(uint32_t *tab, uint32_t first, uint32_t len, uint32_t u) {
    uint32_t bk = first + set_bucket(u, len);
    for (;;) {
        uint32_t z = 0;
        while (z < kSetWays && atomicCAS(&tab[bk * kSetWays + z], kSetFree<kWide>, u) != kSetFree<kWide>) z++;
        if (z < kSetWays) return;
        if (!kWide) atomicOr(&tab[bk * kSetWays + kSetWays - 1], kSetMore);  // full: on to the next
        bk = bk + 1 == first + len ? first : bk + 1;
    }
}

// How many of kN ids are in the region; the ids from number `left` on are not
// counted.  Each id's first bucket is read for all at once, one 16-byte LDS
// read each; the slots are compared without branches, and only a bucket marked
// full goes on to the next.
template <bool kWide = false, int kN>
__device__ __forceinline__ uint32_t set_hits(const uint32_t *tab, const uint32_t (&u)[kN], uint32_t left, uint32_t first,
                                             uint32_t len) {
    const u32x4 *tab4 = reinterpret_cast<const u32x4 *>(tab);
    // the id in a bucket's last slot, and whether ids of the bucket may be in the next
    auto last = [](uint32_t x) -> uint32_t { return kWide ? x : x & ~kSetMore; };
    auto more = [](uint32_t x) -> bool { return kWide ? x != kSetFree<true> : (int)x < 0; };
    uint32_t bk[kN], h = 0;
    u32x4 v[kN];
#pragma unroll
    for (int z = 0; z < kN; z++) {
        bk[z] = first + set_bucket(u[z], len);
        v[z] = tab4[bk[z]];
    }
#pragma unroll
    for (int z = 0; z < kN; z++) {
        const bool in = left > (uint32_t)z;
        const bool f = (v[z][0] == u[z]) | (v[z][1] == u[z]) | (v[z][2] == u[z]) | (last(v[z][3]) == u[z]);
        h += (in & f) ? 1u : 0u;
        if (in & !f & more(v[z][3])) {
            uint32_t b2 = bk[z];
            for (;;) {
                b2 = b2 + 1 == first + len ? first : b2 + 1;
                const u32x4 w = tab4[b2];
                const bool f2 = (w[0] == u[z]) | (w[1] == u[z]) | (w[2] == u[z]) | (last(w[3]) == u[z]);
                h += f2 ? 1u : 0u;
                if (f2 | !more(w[3])) break;
            }
        }
    }
    return h;
}

}  // namespace wtc
