// pga_lookback.h - the place of a sort tile among the tiles before it.
//
// A radix sort pass in one launch (k_sweep, pga_lbvh.hip; the decoupled
// look-back of Merrill and Garland 2016) lets every tile publish, per digit, a
// status word: its own count (kCount) or the count with all tiles before it
// (kPrefix). A tile adds the words of the tiles before it, nearest first, up
// to the first kPrefix. Host code can call it too: the CPU tests drive it with
// words that come late or never.
#ifndef PGA_LOOKBACK_H
#define PGA_LOOKBACK_H

#include <cstdint>

#ifdef __HIPCC__
#define PGA_LB_FN __host__ __device__ __forceinline__
#else
#define PGA_LB_FN inline
#endif

namespace bvhk {

typedef unsigned long long u64;

// One 64-bit word carries flag and value (the low 62 bits), so that relaxed
// accesses order themselves.
constexpr u64 kCount = 1ull << 62, kPrefix = 2ull << 62, kValue = (1ull << 62) - 1ull;

// Sum over the tiles before `tile`. load(k): the status word of tile k;
// idle(): between two looks at a word that has not come; count(k): the count
// of tile k taken from the keys themselves. The words are read kBack at a
// time: they are independent loads, and one at a time the tiles of a million
// keys would be a chain of up to 245 round trips to memory.
// The wait is bounded: after `patience` idle looks in all, a word that has not
// come is counted instead of waited for. A word comes within microseconds as
// long as the tiles before this one run; it never does when something else
// clears the words or the tickets meanwhile (builds that share one scratch
// array and overlap), and a wait without a bound would then hold the GPU.
template <class Load, class Idle, class Count>
PGA_LB_FN uint32_t look_back(uint32_t tile, uint32_t patience, Load load, Idle idle, Count count) {
    constexpr int kBack = 8;
    uint32_t before = 0;
    int64_t k = (int64_t)tile - 1;                  // the nearest tile not yet added
    while (k >= 0) {
        u64 v[kBack];
#ifdef __HIPCC__
#pragma unroll
#endif
        for (int b = 0; b < kBack; ++b) v[b] = load((uint32_t)(k - b > 0 ? k - b : 0));
        bool open = true;                           // every nearer word has been there
#ifdef __HIPCC__
#pragma unroll
#endif
        for (int b = 0; b < kBack; ++b) {
            if (!open || k < 0) continue;
            if (v[b] < kCount) { open = false; continue; }
            before += (uint32_t)(v[b] & kValue);
            k = v[b] >= kPrefix ? -1 : k - 1;
        }
        if (open) continue;
        if (patience != 0u) {
            --patience;
            idle();
        } else {
            before += count((uint32_t)k);
            --k;
        }
    }
    return before;
}

} // namespace bvhk

#endif
