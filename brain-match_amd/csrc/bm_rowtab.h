/*
 * Row tables: one hash table per adjacency row (male and female, out and in),
 * in 16-byte buckets.  A bucket holds four 4-byte slots (key << 15) | weight
 * ("packed": ids below 2^17, weights of both graphs in 0..32767) or two
 * 8-byte slots {key, weight}; slot 0 = empty (ids start at 1).  A key's home
 * bucket is a multiplicative hash; an insert takes the first empty slot from
 * its home bucket on, so a lookup reads one bucket per round and ends at the
 * key or at a bucket with an empty slot.  At a load of at most 1/2 nine of ten
 * absent keys end in the first round, and a row of 216 entries is 2 KB.  A
 * row's descriptor is (first bucket << 6) | log2(buckets); empty rows share
 * the always empty bucket 0, so no lookup needs a test for them.
 */
#ifndef BM_ROWTAB_H
#define BM_ROWTAB_H

#include "bm_device.h"
#include "bm_devutil.h"

namespace bmd {

template <bool PACKED>
struct RowSlots {
    static constexpr uint32_t kPerBucket = PACKED ? 4u : 2u;
};

__device__ __forceinline__ uint32_t row_home(int32_t key, uint32_t lb) {
    return (((uint32_t)key * 0x9E3779B1u) >> (31u - lb)) >> 1;
}

/* One bucket of a lookup: w = key's weight if the bucket holds it (else
 * BM_ABSENT); returns whether the lookup ends here.  key must not be 0. */
template <bool PACKED>
__device__ __forceinline__ bool row_bucket(const uint4& v, int32_t key, int32_t& w) {
    if (PACKED) {
        const uint32_t k = (uint32_t)key;
        const bool h0 = (v.x >> 15) == k, h1 = (v.y >> 15) == k, h2 = (v.z >> 15) == k, h3 = (v.w >> 15) == k;
        const uint32_t e = h0 ? v.x : (h1 ? v.y : (h2 ? v.z : v.w));
        const bool hit = h0 || h1 || h2 || h3;
        w = hit ? (int32_t)(e & 0x7fffu) : BM_ABSENT;
        /* slots fill in order, so the last one tells whether one is empty */
        return hit || v.w == 0u;
    }
    const bool h0 = (int32_t)v.x == key, h1 = (int32_t)v.z == key;
    w = h0 ? (int32_t)v.y : (h1 ? (int32_t)v.w : BM_ABSENT);
    return h0 || h1 || v.z == 0u;
}

/* Weight of key (not 0) in the row with descriptor d, or BM_ABSENT, `skip`
 * buckets past its home on. */
template <bool PACKED>
__device__ __forceinline__ int32_t row_find_from(const uint4* __restrict__ tab, uint64_t d, int32_t key, uint32_t skip) {
    const uint32_t lb = (uint32_t)(d & 63u), mask = (1u << lb) - 1u;
    const uint4* T = tab + (d >> 6);
    uint32_t b = (row_home(key, lb) + skip) & mask;
    for (;;) {
        int32_t w;
        if (row_bucket<PACKED>(T[b], key, w)) return w;
        b = (b + 1u) & mask;
    }
}

/* Weight of key in the row with descriptor d, or BM_ABSENT (key 0: absent). */
template <bool PACKED>
__device__ __forceinline__ int32_t row_find(const uint4* __restrict__ tab, uint64_t d, int32_t key) {
    return key == 0 ? BM_ABSENT : row_find_from<PACKED>(tab, d, key, 0u);
}

}  // namespace bmd

#endif
