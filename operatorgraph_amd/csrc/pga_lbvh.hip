// pga_lbvh.hip - linear BVH over terminal AABBs on gfx950 (wave64).
//
// The construction of GPUBVHConstructor.cuh (Karras 2012) in three steps:
//   1. k_morton  - AABB centre normalised to the scene box, 10 bits per axis
//                  interleaved into a 30-bit Morton code (GPUBVHConstructor.cuh:
//                  44-86), written as the reference's unique 64-bit key
//                  (code << 32 | index), with the digit histograms of all four
//                  sort passes;
//   2. LSD radix sort of the keys' codes, four 8-bit passes (thrust::sort,
//                  :311-312, orders the same keys): k_digit_totals, then one
//                  k_sweep per pass, which ranks a tile, finds the tile's place
//                  by looking back over the tiles before it, and scatters it.
//                  A stable sort of the codes of ascending indices gives the
//                  order of the keys. Up to kSmallLeaves leaves one workgroup
//                  sorts in LDS (k_sort_small);
//   3. the tree  - the radix tree (buildRadixTree, :88-213) and its boxes
//                  (propagateBVH, :215-261) in one climb from the leaves
//                  (after Apetrei 2014): a subtree over the sorted leaves
//                  [l, r] continues on the side of the closer neighbour, the
//                  first child to reach a split leaves its end and box there,
//                  the second unites both and goes on. k_tree_leaves climbs
//                  inside a workgroup's tile of leaves, k_tree_roots inside a
//                  group of the subtrees the previous level could not finish,
//                  until one group is left; every exchange goes through LDS.
//                  The numbering is the reference's: a right child [l, r] is
//                  node l, a left child node r, the root node 0.
// Children are encoded as in the reference: >= 0 a leaf (sorted position),
// < 0 an internal node (negated index); node 0 is the root.
//
// Device-count mode: every kernel that reads the leaf count n takes the host
// bound n (grid size) and an optional device word nd; with nd the count is
// min(*nd, n), so a gather of the derived terminals, the scene box and the
// whole build run from device state without a host round trip, and can be
// recorded in a HIP graph and replayed while the terminal counts change.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "../../include/pga.h"
#include "pga_lookback.h"

namespace bvhk {

constexpr uint32_t kThreads = 1024;              // sort and tree workgroups
constexpr uint32_t kWaves = kThreads / 64u;
constexpr uint32_t kItems = 4;
constexpr uint32_t kTile = kThreads * kItems;   // keys per sort workgroup
constexpr uint32_t kSmallLeaves = kTile;        // up to here one workgroup sorts all keys in LDS
constexpr uint32_t kDigits = 256, kPasses = 4;  // 30-bit codes: digits at bits 32, 40, 48, 56 of the key
constexpr uint32_t kHistBlocks = 512;           // most workgroups of k_morton
constexpr uint32_t kGatherBlocks = 8192;         // grid-stride workgroups of the terminal gather
constexpr uint32_t kTreeTile = 1024;             // sorted leaves per workgroup of the tree's first level
constexpr uint32_t kTreeGroup = 32;              // workgroups of one level whose open subtrees one of the next takes
constexpr uint32_t kMaxRoots = 128;              // open subtrees a workgroup may leave (see k_tree_leaves)
// two floats of a box record: boxes are 24-byte records that a caller may align to 4 bytes only
typedef float box2 __attribute__((ext_vector_type(2), aligned(4)));

// leaf count: the host bound, or the device word when there is one
__device__ __forceinline__ uint32_t leaf_count(uint32_t n, const uint32_t* nd) {
    return nd ? min(*nd, n) : n;
}

__device__ __forceinline__ uint32_t f2u_rd(float x) {
    if (!(x > 0.0f)) return 0u;
    if (x >= 4294967296.0f) return 0xFFFFFFFFu;
    return (uint32_t)x;
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {     // GPUBVHConstructor.cuh:48-54
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t morton30(float x, float y, float z) {   // :56-64
    uint32_t vx = min(f2u_rd(x * 1023.0f), 1023u);
    uint32_t vy = min(f2u_rd(y * 1023.0f), 1023u);
    uint32_t vz = min(f2u_rd(z * 1023.0f), 1023u);
    return spread10(vx) | (spread10(vy) << 1) | (spread10(vz) << 2);
}

// AABB of the unit cube (or, planar, the unit square z = 0) under an
// instance's model rows: centre = translation, half extent of row r =
// 0.5 (|m_r0| + |m_r1| (+ |m_r2|)).
__global__ void __launch_bounds__(256) k_instance_aabbs(const pga_instance* __restrict__ inst, uint32_t n,
                                                        uint32_t planar, float* __restrict__ aabbs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4* m = reinterpret_cast<const float4*>(inst + i);
    const float4 r0 = m[0], r1 = m[1], r2 = m[2];
    float h0 = fabsf(r0.x) + fabsf(r0.y), h1 = fabsf(r1.x) + fabsf(r1.y), h2 = fabsf(r2.x) + fabsf(r2.y);
    if (!planar) { h0 = h0 + fabsf(r0.z); h1 = h1 + fabsf(r1.z); h2 = h2 + fabsf(r2.z); }
    h0 = h0 * 0.5f; h1 = h1 * 0.5f; h2 = h2 * 0.5f;
    float* o = aabbs + (size_t)i * 6u;
    o[0] = r0.w - h0; o[1] = r1.w - h1; o[2] = r2.w - h2;
    o[3] = r0.w + h0; o[4] = r1.w + h1; o[5] = r2.w + h2;
}

// Boxes of the instances of terminal types 0..ntypes-1, concatenated in type
// order (each buffer in its own order): counts come from the derivation's
// device counters, each clamped to its buffer's capacity. Writes the leaf
// count min(total, capacity) and an overflow flag.
struct GatherArgs {
    const pga_instance* buf[PGA_MAX_TERMINALS];
    unsigned long long cap[PGA_MAX_TERMINALS];
    uint32_t ntypes, planar_mask, capacity;
};

__global__ void __launch_bounds__(256) k_gather_boxes(GatherArgs g, const unsigned long long* __restrict__ counts,
                                                      float* __restrict__ aabbs, uint32_t* __restrict__ nd,
                                                      uint32_t* __restrict__ overflow) {
    __shared__ unsigned long long start[PGA_MAX_TERMINALS + 1];
    if (threadIdx.x == 0) {
        unsigned long long s = 0;
        for (uint32_t t = 0; t < g.ntypes; ++t) {
            start[t] = s;
            const unsigned long long c = counts[t];
            s += c < g.cap[t] ? c : g.cap[t];
        }
        start[g.ntypes] = s;
        if (blockIdx.x == 0) {
            *nd = (uint32_t)(s < g.capacity ? s : g.capacity);
            *overflow = s > g.capacity ? 1u : 0u;
        }
    }
    __syncthreads();
    const unsigned long long total = start[g.ntypes] < g.capacity ? start[g.ntypes] : g.capacity;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (unsigned long long)gridDim.x * blockDim.x) {
        uint32_t t = 0;                       // the last type whose range starts at or before i
        for (uint32_t step = 32; step > 0; step >>= 1)
            if (t + step < g.ntypes && start[t + step] <= i) t += step;
        const float4* m = reinterpret_cast<const float4*>(g.buf[t] + (i - start[t]));
        const float4 r0 = m[0], r1 = m[1], r2 = m[2];
        float h0 = fabsf(r0.x) + fabsf(r0.y), h1 = fabsf(r1.x) + fabsf(r1.y), h2 = fabsf(r2.x) + fabsf(r2.y);
        if (!((g.planar_mask >> t) & 1u)) { h0 = h0 + fabsf(r0.z); h1 = h1 + fabsf(r1.z); h2 = h2 + fabsf(r2.z); }
        h0 = h0 * 0.5f; h1 = h1 * 0.5f; h2 = h2 * 0.5f;
        float* o = aabbs + i * 6u;
        o[0] = r0.w - h0; o[1] = r1.w - h1; o[2] = r2.w - h2;
        o[3] = r0.w + h0; o[4] = r1.w + h1; o[5] = r2.w + h2;
    }
}

// Per-workgroup min/max of the AABB corners (scene box), then one workgroup
// folds the partials.
__global__ void __launch_bounds__(256) k_bounds(const float* __restrict__ aabbs, uint32_t n, const uint32_t* nd,
                                                float* __restrict__ part) {
    __shared__ float red[6][256];
    n = leaf_count(n, nd);
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float* a = aabbs + (size_t)i * 6u;
        for (int q = 0; q < 3; ++q) { b[q] = fminf(b[q], a[q]); b[q + 3] = fmaxf(b[q + 3], a[q + 3]); }
    }
    for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = b[q];
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int q = 0; q < 6; ++q)
                red[q][threadIdx.x] = q < 3 ? fminf(red[q][threadIdx.x], red[q][threadIdx.x + s])
                                            : fmaxf(red[q][threadIdx.x], red[q][threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6u + threadIdx.x] = red[threadIdx.x][0];
}
__global__ void __launch_bounds__(256) k_bounds_fold(float* part, uint32_t nparts) {
    __shared__ float red[6][256];
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t b = threadIdx.x; b < nparts; b += blockDim.x)
        for (int q = 0; q < 6; ++q) v[q] = q < 3 ? fminf(v[q], part[b * 6u + q]) : fmaxf(v[q], part[b * 6u + q]);
    for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = v[q];
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h)
            for (int q = 0; q < 6; ++q)
                red[q][threadIdx.x] = q < 3 ? fminf(red[q][threadIdx.x], red[q][threadIdx.x + h])
                                            : fmaxf(red[q][threadIdx.x], red[q][threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x < 6) part[threadIdx.x] = red[threadIdx.x][0];
}

// Adds one to h[d] for every lane of `valid`: sorted or clustered input gives
// whole waves one digit, which then costs one LDS atomic instead of 64 on the
// same address.
__device__ __forceinline__ void hist_add(uint32_t* h, uint32_t d, bool valid) {
    const u64 m = __ballot(valid);
    if (m == 0ull) return;
    const int lead = __ffsll((long long)m) - 1;
    const uint32_t d0 = __shfl(d, lead);
    if (__ballot(valid && d != d0) == 0ull) {
        if ((int)(threadIdx.x & 63u) == lead) atomicAdd(&h[d0], (uint32_t)__popcll(m));
    } else if (valid) {
        atomicAdd(&h[d], 1u);
    }
}

// Morton code of box i: the scene box from the host (mn, ex) or, with `box`,
// from the device: min xyz, max xyz, an empty extent taken as 1.
struct Scene {
    float mn0, mn1, mn2, ex0, ex1, ex2;
    const float* box;
};
__device__ __forceinline__ Scene scene_of(Scene sc) {
    if (sc.box) {
        const float* box = sc.box;
        sc.mn0 = box[0]; sc.mn1 = box[1]; sc.mn2 = box[2];
        sc.ex0 = box[3] - sc.mn0; sc.ex1 = box[4] - sc.mn1; sc.ex2 = box[5] - sc.mn2;
        sc.ex0 = sc.ex0 > 0.0f ? sc.ex0 : 1.0f; sc.ex1 = sc.ex1 > 0.0f ? sc.ex1 : 1.0f;
        sc.ex2 = sc.ex2 > 0.0f ? sc.ex2 : 1.0f;
    }
    return sc;
}
__device__ __forceinline__ u64 morton_key(const float* __restrict__ aabbs, uint32_t i, const Scene& sc) {
    const float* b = aabbs + (size_t)i * 6u;
    const float cx = (b[0] + b[3]) * 0.5f, cy = (b[1] + b[4]) * 0.5f, cz = (b[2] + b[5]) * 0.5f;
    const uint32_t code = morton30((cx - sc.mn0) / sc.ex0, (cy - sc.mn1) / sc.ex1, (cz - sc.mn2) / sc.ex2);
    return ((u64)code << 32) | (u64)i;
}

// ---- radix sort: stable, 8-bit digits, one launch per pass ----
// Keys of all leaves, and each workgroup's histograms of the four digits
// (rows[block][pass * 256 + digit]). Also clears what the sweeps share: the
// tile tickets and, per pass, tile and digit, the status words.
__global__ void __launch_bounds__(kThreads) k_morton(const float* __restrict__ aabbs, uint32_t n, const uint32_t* nd,
                                                     Scene scene, u64* __restrict__ keys, uint32_t* __restrict__ rows,
                                                     u64* __restrict__ status, uint32_t nstatus,
                                                     uint32_t* __restrict__ tickets) {
    __shared__ uint32_t h[kPasses * kDigits];
    n = leaf_count(n, nd);
    h[threadIdx.x] = 0u;                       // kPasses * kDigits == kThreads
    if (blockIdx.x == 0u && threadIdx.x < kPasses) tickets[threadIdx.x] = 0u;
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < nstatus; i += gridDim.x * kThreads) status[i] = 0ull;
    __syncthreads();
    const Scene sc = scene_of(scene);
    for (uint32_t base = blockIdx.x * kThreads; base < n; base += gridDim.x * kThreads) {
        const uint32_t i = base + threadIdx.x;
        const bool valid = i < n;
        u64 key = 0ull;
        if (valid) {
            key = morton_key(aabbs, i, sc);
            keys[i] = key;
        }
#pragma unroll
        for (uint32_t p = 0; p < kPasses; ++p)
            hist_add(h + p * kDigits, (uint32_t)(key >> (32u + 8u * p)) & 0xFFu, valid);
    }
    __syncthreads();
    rows[(size_t)blockIdx.x * kThreads + threadIdx.x] = h[threadIdx.x];
}
static_assert(kPasses * kDigits == kThreads, "one histogram word per thread");

// totals[pass * 256 + digit]: the histogram rows summed; a workgroup takes 64
// columns, 16 row groups side by side.
__global__ void __launch_bounds__(kThreads) k_digit_totals(const uint32_t* __restrict__ rows, uint32_t nrows,
                                                           uint32_t* __restrict__ totals) {
    __shared__ uint32_t part[kWaves][64];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t col = blockIdx.x * 64u + lane;
    uint32_t s = 0;
#pragma unroll 8
    for (uint32_t r = w; r < nrows; r += kWaves) s += rows[(size_t)r * kThreads + col];
    part[w][lane] = s;
    __syncthreads();
    if (w == 0u) {
        for (uint32_t k = 1; k < kWaves; ++k) s += part[k][lane];
        totals[col] = s;
    }
}

struct SortLDS {
    u64 key[kTile];                     // the tile in the order of this pass's digit
    uint32_t wave[kWaves][kDigits];     // per wave: count, then offset of each digit
    uint32_t first[kDigits];            // tile position of each digit's first key
    uint32_t base[kDigits];             // output position of each digit's first key, less `first`
    uint32_t sums[8];
    uint32_t tile;
};

// Exclusive prefix over the first 256 threads (four waves; `sums` holds a
// word per wave). Every thread of the workgroup calls it.
__device__ __forceinline__ uint32_t scan256(uint32_t v, uint32_t* sums) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if ((int)lane >= d) x += y;
    }
    if (w < 4u && lane == 63u) sums[w] = x;
    __syncthreads();
    uint32_t off = 0;
    for (uint32_t k = 0; k < 4u; ++k) off += k < w ? sums[k] : 0u;
    __syncthreads();
    return off + x - v;
}

// Ranks the tile's keys by the digit at `shift`: S.first (first tile position
// of each digit), rank[] (position of each key in the tile); thread d < 256
// returns the tile's count of digit d. Wave w holds the keys w * 256 ..
// w * 256 + 255 in tile order, 64 a step: within a step a lane's rank among
// the lanes of its digit comes from eight ballots, and the wave's running
// counts are its own, so the four steps need no barrier.
__device__ __forceinline__ uint32_t rank_tile(SortLDS& S, const u64 key[kItems], uint32_t nvalid, uint32_t shift,
                                              uint32_t rank[kItems]) {
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    // LDS pointer of its own address space: volatile accesses through a generic
    // one would be flat loads and stores
    typedef __attribute__((address_space(3))) volatile uint32_t lds_u32;
    lds_u32* mine = (lds_u32*)S.wave[w];
    for (uint32_t k = lane; k < kDigits; k += 64u) mine[k] = 0u;
    const u64 lt = (1ull << lane) - 1ull;
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const bool valid = w * 256u + it * 64u + lane < nvalid;
        const uint32_t d = (uint32_t)(key[it] >> shift) & 0xFFu;
        u64 peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const u64 on = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? on : ~on;
        }
        const uint32_t before = mine[d], r = (uint32_t)__popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();       // every lane has read the count its digit had
        if (valid && r == 0u) mine[d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[it] = before + r;
    }
    __syncthreads();
    uint32_t total = 0;
    if (t < kDigits)
        for (uint32_t k = 0; k < kWaves; ++k) {
            const uint32_t c = S.wave[k][t];
            S.wave[k][t] = total;
            total += c;
        }
    const uint32_t f = scan256(total, S.sums);
    if (t < kDigits) S.first[t] = f;
    __syncthreads();
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const uint32_t d = (uint32_t)(key[it] >> shift) & 0xFFu;
        rank[it] += S.first[d] + S.wave[w][d];
    }
    return total;
}

// Idle looks of the look-back before it counts a tile's digit itself: 10 to 20
// ms, a thousand times what a word takes to come.
constexpr uint32_t kPatience = 1u << 14;

// One pass: the tile's keys ranked in LDS, the tile's place in the output of
// every digit found by looking back over the tiles before it, the keys
// written in tile order (runs of consecutive keys per digit). A tile waits
// for lower tiles only, and tiles are numbered by ticket in the order in
// which workgroups start, so the lowest unfinished tile is always running and
// never waits; and no wait is longer than kPatience looks (look_back). A
// million keys sort in 4 x 16.7 us; a histogram, three scan launches and a
// scatter a pass took 181 us (20 launches).
__global__ void __launch_bounds__(kThreads) k_sweep(const u64* __restrict__ in, u64* __restrict__ out, uint32_t n,
                                                    const uint32_t* nd, uint32_t pass,
                                                    const uint32_t* __restrict__ totals, u64* status,
                                                    uint32_t* tickets) {
    __shared__ SortLDS S;
    n = leaf_count(n, nd);
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6, shift = 32u + 8u * pass;
    if (t == 0u) S.tile = atomicAdd(&tickets[pass], 1u);
    __syncthreads();
    const uint32_t tile = S.tile;
    if ((uint64_t)tile * kTile >= n) return;            // whole workgroup: no keys here
    const uint32_t s = tile * kTile, cnt = min(kTile, n - s);
    u64 key[kItems];
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const uint32_t q = w * 256u + it * 64u + lane;
        key[it] = q < cnt ? in[s + q] : 0ull;
    }
    uint32_t rank[kItems];
    const uint32_t total = rank_tile(S, key, cnt, shift, rank);
    u64* st = status + t;                               // word of tile k: st[k * 256]
    if (t < kDigits)
        __hip_atomic_store(&st[(size_t)tile * kDigits], (tile ? kCount : kPrefix) | total, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it)
        if (w * 256u + it * 64u + lane < cnt) S.key[rank[it]] = key[it];
    const uint32_t g = scan256(t < kDigits ? totals[pass * kDigits + t] : 0u, S.sums);
    if (t < kDigits) {
        const uint32_t before = look_back(
            tile, kPatience,
            [&](uint32_t k) {
                return __hip_atomic_load(&st[(size_t)k * kDigits], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            },
            [] { __builtin_amdgcn_s_sleep(1); },
            [&](uint32_t k) {                           // tile k < tile: all its keys are there
                uint32_t c = 0;
#pragma unroll 8
                for (uint32_t q = 0; q < kTile; ++q) c += ((uint32_t)(in[(size_t)k * kTile + q] >> shift) & 0xFFu) == t;
                return c;
            });
        if (tile)
            __hip_atomic_store(&st[(size_t)tile * kDigits], kPrefix | (u64)(before + total), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        S.base[t] = g + before - S.first[t];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const uint32_t q = it * kThreads + t;
        if (q < cnt) {
            const u64 x = S.key[q];
            const uint32_t off = S.base[(uint32_t)(x >> shift) & 0xFFu] + q;
            if (off < n) out[off] = x;                  // always true for a build that has its scratch to itself
        }
    }
}

// Up to kSmallLeaves leaves (one sort tile): keys and sort in one workgroup,
// 17.8 us for 3,001 leaves, where the launches above would take about 45 us
// (9 us a pass at a few tiles) and the separate scans took 120.
__global__ void __launch_bounds__(kThreads) k_sort_small(const float* __restrict__ aabbs, uint32_t n,
                                                         const uint32_t* nd, Scene scene, u64* __restrict__ keys) {
    __shared__ SortLDS S;
    n = min(leaf_count(n, nd), kSmallLeaves);
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const Scene sc = scene_of(scene);
    u64 key[kItems];
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const uint32_t i = w * 256u + it * 64u + lane;
        key[it] = i < n ? morton_key(aabbs, i, sc) : 0ull;
    }
#pragma unroll 1
    for (uint32_t pass = 0; pass < kPasses; ++pass) {
        uint32_t rank[kItems];
        (void)rank_tile(S, key, n, 32u + 8u * pass, rank);
#pragma unroll
        for (uint32_t it = 0; it < kItems; ++it)
            if (w * 256u + it * 64u + lane < n) S.key[rank[it]] = key[it];
        __syncthreads();
#pragma unroll
        for (uint32_t it = 0; it < kItems; ++it) {
            const uint32_t i = w * 256u + it * 64u + lane;
            if (i < n) key[it] = S.key[i];
        }
        // the next pass writes S.key after its barriers
    }
#pragma unroll
    for (uint32_t it = 0; it < kItems; ++it) {
        const uint32_t i = w * 256u + it * 64u + lane;
        if (i < n) keys[i] = key[it];
    }
}

// ---- the tree ----
// The union is taken in child order, left box first: min(L, R) = R < L ? R : L
// and max(L, R) = L < R ? R : L, as std::min / std::max fold them.
__device__ __forceinline__ void unite(const float b[6], const float o[6], bool mine_left, float u[6]) {
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const float L = mine_left ? b[q] : o[q], R = mine_left ? o[q] : b[q];
        u[q] = q < 3 ? (R < L ? R : L) : (L < R ? R : L);
    }
}

struct TreeOut {
    int32_t *left, *right, *parent, *leaf_parent;
    int32_t* other_end;                 // the end of node i's leaf range other than i (NULL: not wanted)
    float* node_aabb;
};

// A subtree over the sorted leaves [l, r] whose parent reaches beyond the
// workgroup that completed it, with its box.
struct __align__(16) Root {
    uint32_t l, r;
    float2 b0, b1, b2;
};

// The items of a workgroup, in leaf order: leaves (CAP = kTreeTile), or the
// open subtrees of the level before (CAP = kTreeGroup * kMaxRoots).
template <uint32_t CAP>
struct TreeLDS {
    float2 box[CAP * 3u];               // the box a subtree left for its sibling, at the end the sibling meets
    uint32_t slot[CAP];                 // split between items q and q + 1: the far end (+ 1) of the child that came first
    uint16_t mark[CAP];                 // open subtree starting at item q: its end + 1 | 0x8000 for a right child
    int8_t delta[CAP + 4u];             // common prefix of the keys either side of item q's start (-1: none)
    uint32_t sums[kWaves];
};
// ... and what the first level writes out at the end, by tile position
struct LeafOut {
    uint16_t node[kTreeTile];           // node: split | kLeftLeaf | kRightLeaf (kNoNode: made elsewhere)
    uint16_t parent[kTreeTile];         // parent of node / leaf (kNoNode: made elsewhere)
    uint16_t leaf_parent[kTreeTile];
    uint16_t other_end[kTreeTile];
};
constexpr uint32_t kLeftLeaf = 0x4000u, kRightLeaf = 0x8000u, kNoNode = 0xFFFFu;   // split < kTreeTile <= 0x4000
// ... and the first leaf of each item above it ([m]: the leaf after the last item)
struct RootIn {
    uint32_t first[kTreeGroup * kMaxRoots + 1u];
    uint32_t pre[kTreeGroup + 1u];
};

// Common prefix length of the keys of leaves x - 1 and x, -1 at the ends.
__device__ __forceinline__ int key_delta(const u64* __restrict__ keys, uint32_t x, uint32_t n) {
    return x == 0u || x >= n ? -1 : __clzll((long long)(keys[x - 1u] ^ keys[x]));
}

// Climbs from item q with box b until the sibling has not come yet, the
// parent reaches beyond the workgroup's m items (mark), or the root is done.
// A subtree [ql, qr] is the right child of its parent when its first key
// shares more bits with the key before it than its last with the key after
// it; the two are never equal, as the keys are unique. Both children meet at
// the split between them. A subtree leaves its box at its end next to the
// split, before the exchange of the slot: two subtrees with that end are
// nested, and the inner one's box was taken before the outer one existed.
// That end is the subtree's node number, so at the end box[] holds the boxes
// of the nodes made here.
// The climb is a chain of LDS round trips (the exchange, then the sibling's
// box and the key distance at its far end), at two workgroups of 16 waves a
// compute unit. The first level's nodes go out afterwards, in order, instead
// of seven scattered stores a step with a few lanes left: k_tree_leaves over
// a million leaves 53 -> 45 us. A Karras search per node and a separate refit
// through global memory (three kernels, which read the topology back) took
// 142 us for what the levels here do in 45 + 46.
template <bool LEAVES, uint32_t CAP>
__device__ __forceinline__ void climb(TreeLDS<CAP>& T, LeafOut* lo, const RootIn* in, const TreeOut& out, uint32_t n,
                                      uint32_t m, uint32_t q, float2 b0, float2 b1, float2 b2) {
    uint32_t ql = q, qr = q;
    uint32_t L = LEAVES ? q : in->first[q], R1 = LEAVES ? q + 1u : in->first[q + 1u];   // leaves [L, R1)
    int dl = T.delta[ql], dr = T.delta[qr + 1u];
    bool made = false;                  // [ql, qr] is a node made here: split before leaf P, children leaves or nodes
    uint32_t P = 0;
    bool lleaf = false, rleaf = false;
    for (;;) {
        const bool root = dl < 0 && dr < 0, right = dl > dr;
        if (made) {
            const uint32_t node = root ? 0u : (right ? L : R1 - 1u);
            if (LEAVES) {
                lo->node[node] = (uint16_t)((P - 1u) | (lleaf ? kLeftLeaf : 0u) | (rleaf ? kRightLeaf : 0u));
                uint16_t* pl = lleaf ? lo->leaf_parent : lo->parent;
                uint16_t* pr = rleaf ? lo->leaf_parent : lo->parent;
                pl[P - 1u] = (uint16_t)node;
                pr[P] = (uint16_t)node;
                lo->other_end[node] = (uint16_t)(node == L ? R1 - 1u : L);
            } else if (node < n - 1u && P - 1u < n - 1u && (rleaf || P < n - 1u)) {
                // (always; the open subtrees come from memory that a build which
                // breaks the rule of pga_lbvh_build_noalloc writes, too)
                const int32_t lc = lleaf ? (int32_t)(P - 1u) : -(int32_t)(P - 1u), rc = rleaf ? (int32_t)P : -(int32_t)P;
                out.left[node] = lc;
                out.right[node] = rc;
                (lleaf ? out.leaf_parent : out.parent)[P - 1u] = (int32_t)node;
                (rleaf ? out.leaf_parent : out.parent)[P] = (int32_t)node;
                if (root) out.parent[0] = -1;
                if (out.other_end) out.other_end[node] = (int32_t)(node == L ? R1 - 1u : L);
                box2* o = reinterpret_cast<box2*>(out.node_aabb + (size_t)node * 6u);
                o[0] = box2{b0.x, b0.y};
                o[1] = box2{b1.x, b1.y};
                o[2] = box2{b2.x, b2.y};
            }
        }
        float2* mine = &T.box[(root ? 0u : (right ? ql : qr)) * 3u];
        mine[0] = b0;
        mine[1] = b1;
        mine[2] = b2;
        if (root) return;
        if (right ? ql == 0u : qr + 1u == m) {
            T.mark[ql] = (uint16_t)((qr + 1u) | (right ? 0x8000u : 0u));
            return;
        }
        const uint32_t sp = right ? ql - 1u : qr;
        // only LDS needs ordering: the box is in place before the slot is
        // exchanged, and the sibling's is read after it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint32_t v = __hip_atomic_exchange(&T.slot[sp], (right ? qr : ql) + 1u, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");
        if (v == 0u) return;            // the sibling's thread goes on from here
        T.slot[sp] = 0u;                // both have come
        const float2* src = &T.box[(right ? sp : sp + 1u) * 3u];
        const float2 s0 = src[0], s1 = src[1], s2 = src[2];
        const uint32_t far = v - 1u;    // the sibling's far end
        const int d = T.delta[right ? far : far + 1u];
        const uint32_t F = LEAVES ? (right ? far : far + 1u) : in->first[right ? far : far + 1u];
        const float bb[6] = {b0.x, b0.y, b1.x, b1.y, b2.x, b2.y}, o[6] = {s0.x, s0.y, s1.x, s1.y, s2.x, s2.y};
        float u[6];
        unite(bb, o, !right, u);
        b0 = make_float2(u[0], u[1]);
        b1 = make_float2(u[2], u[3]);
        b2 = make_float2(u[4], u[5]);
        if (right) {
            P = L;
            rleaf = R1 - L == 1u;
            lleaf = L - F == 1u;
            L = F; ql = far; dl = d;
        } else {
            P = R1;
            lleaf = R1 - L == 1u;
            rleaf = F - R1 == 1u;
            R1 = F; qr = far; dr = d;
        }
        made = true;
    }
}

// The open subtrees of the workgroup, in leaf order: those marked, and those
// whose sibling has not come to their split. Every thread calls it after all
// climbs. A level's roots are at most kMaxRoots: they are the siblings that
// hang off the two paths from the tree's root to the workgroup's first and
// last leaf, and a radix tree over unique 64-bit keys whose top two bits are
// zero is at most 62 levels deep.
template <uint32_t CAP>
__device__ __forceinline__ void leave_roots(TreeLDS<CAP>& T, const RootIn* in, uint32_t s, uint32_t m,
                                            Root* __restrict__ roots, uint32_t* __restrict__ nroots) {
    constexpr uint32_t K = CAP / kThreads;      // in: first leaves of the items (NULL: item q is leaf s + q)
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    __syncthreads();
    for (uint32_t q = t; q < m; q += kThreads) {
        const uint32_t v = T.slot[q];
        if (v == 0u) continue;
        if (v - 1u <= q) T.mark[v - 1u] = (uint16_t)(q + 1u);      // the left child [v - 1, q]
        else T.mark[q + 1u] = (uint16_t)(v | 0x8000u);             // the right child [q + 1, v - 1]
    }
    __syncthreads();
    uint32_t c = 0;
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) c += t * K + k < m && T.mark[t * K + k] != 0u ? 1u : 0u;
    uint32_t x = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if ((int)lane >= d) x += y;
    }
    if (lane == 63u) T.sums[w] = x;
    __syncthreads();
    uint32_t off = x - c, all = 0;
    for (uint32_t k = 0; k < kWaves; ++k) {
        off += k < w ? T.sums[k] : 0u;
        all += T.sums[k];
    }
    if (t == 0u) *nroots = min(all, kMaxRoots);
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        const uint32_t q = t * K + k;
        if (q >= m || T.mark[q] == 0u) continue;
        const uint32_t e = T.mark[q] & 0x7FFFu, at = (T.mark[q] & 0x8000u) ? q : e - 1u;
        if (off < kMaxRoots) {
            Root r;
            r.l = in ? in->first[q] : s + q;
            r.r = (in ? in->first[e] : s + e) - 1u;
            r.b0 = T.box[at * 3u];
            r.b1 = T.box[at * 3u + 1u];
            r.b2 = T.box[at * 3u + 2u];
            roots[off] = r;
        }
        ++off;
    }
}

// First level: a workgroup per tile of kTreeTile sorted leaves, one leaf per
// thread (41 KB of LDS, two workgroups of 16 waves per compute unit). What
// bounds it is the gather of the leaf boxes through the sorted keys (24 bytes
// from a 128-byte line each) and the length of the climbs in LDS; the tile's
// nodes are written in order afterwards.
__global__ void __launch_bounds__(kThreads) k_tree_leaves(const float* __restrict__ aabbs,
                                                          const u64* __restrict__ keys, uint32_t n, const uint32_t* nd,
                                                          TreeOut out, Root* __restrict__ roots,
                                                          uint32_t* __restrict__ nroots) {
    __shared__ __align__(16) TreeLDS<kTreeTile> T;
    __shared__ LeafOut O;
    static_assert(kTreeTile == kThreads, "one leaf per thread");
    n = leaf_count(n, nd);
    const uint32_t q = threadIdx.x, s = blockIdx.x * kTreeTile;
    if (s >= n) {
        if (q == 0u) nroots[blockIdx.x] = 0u;
        return;
    }
    const uint32_t m = min(kTreeTile, n - s);
    const uint32_t i = s + min(q, m - 1u);
    const u64 key = keys[i];
    const box2* src = reinterpret_cast<const box2*>(aabbs + (size_t)min((uint32_t)key, n - 1u) * 6u);
    const box2 g0 = src[0], g1 = src[1], g2 = src[2];
    T.slot[q] = 0u;
    T.mark[q] = 0u;
    O.node[q] = O.parent[q] = O.leaf_parent[q] = (uint16_t)kNoNode;
    if (q < m) T.delta[q] = (int8_t)(i == 0u ? -1 : __clzll((long long)(keys[i - 1u] ^ key)));
    if (q == 0u) T.delta[m] = (int8_t)key_delta(keys, s + m, n);
    __syncthreads();
    if (q < m)
        climb<true>(T, &O, nullptr, out, n, m, q, make_float2(g0.x, g0.y), make_float2(g1.x, g1.y),
                    make_float2(g2.x, g2.y));
    leave_roots(T, nullptr, s, m, roots + (size_t)blockIdx.x * kMaxRoots, nroots + blockIdx.x);
    if (q >= m) return;
    const uint32_t node = O.node[q], par = O.parent[q], lpar = O.leaf_parent[q];
    if (lpar != kNoNode) out.leaf_parent[i] = (int32_t)(s + lpar);
    if (par != kNoNode) out.parent[i] = (int32_t)(s + par);
    if (node != kNoNode) {
        const int32_t p = (int32_t)(s + (node & 0x3FFFu));
        out.left[i] = (node & kLeftLeaf) ? p : -p;
        out.right[i] = (node & kRightLeaf) ? p + 1 : -(p + 1);
        if (out.other_end) out.other_end[i] = (int32_t)(s + O.other_end[q]);
        box2* o = reinterpret_cast<box2*>(out.node_aabb + (size_t)i * 6u);
        const float2 a = T.box[q * 3u], b = T.box[q * 3u + 1u], c = T.box[q * 3u + 2u];
        o[0] = box2{a.x, a.y};
        o[1] = box2{b.x, b.y};
        o[2] = box2{c.x, c.y};
        if (i == 0u) out.parent[0] = -1;        // the whole tree is one tile
    }
}

// The levels above: a workgroup takes the open subtrees of kTreeGroup
// workgroups of the level before.
__global__ void __launch_bounds__(kThreads) k_tree_roots(const u64* __restrict__ keys, uint32_t n, const uint32_t* nd,
                                                         TreeOut out, const Root* __restrict__ in,
                                                         const uint32_t* __restrict__ nin, uint32_t groups,
                                                         Root* __restrict__ roots, uint32_t* __restrict__ nroots) {
    constexpr uint32_t CAP = kTreeGroup * kMaxRoots;
    __shared__ __align__(16) TreeLDS<CAP> T;
    __shared__ RootIn I;
    n = leaf_count(n, nd);
    const uint32_t t = threadIdx.x, g0 = blockIdx.x * kTreeGroup;
    if (t < 64u) {                      // one wave: prefix of the groups' counts
        const uint32_t c = t < kTreeGroup && g0 + t < groups ? min(nin[g0 + t], kMaxRoots) : 0u;
        uint32_t x = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d);
            if ((int)t >= d) x += y;
        }
        if (t <= kTreeGroup) I.pre[t] = x - c;
    }
    __syncthreads();
    const uint32_t m = I.pre[kTreeGroup];
    if (m == 0u) {
        if (t == 0u) nroots[blockIdx.x] = 0u;
        return;
    }
    for (uint32_t x = t; x < CAP; x += kThreads) {
        const uint32_t c = x / kMaxRoots, q = I.pre[c] + x % kMaxRoots;
        if (q >= I.pre[c + 1u]) continue;
        const Root r = in[(size_t)g0 * kMaxRoots + x];
        I.first[q] = r.l;
        T.box[q * 3u] = r.b0;
        T.box[q * 3u + 1u] = r.b1;
        T.box[q * 3u + 2u] = r.b2;
        T.delta[q] = (int8_t)key_delta(keys, r.l, n);
        T.slot[q] = 0u;
        T.mark[q] = 0u;
        if (q + 1u == m) {
            I.first[m] = r.r + 1u;
            T.delta[m] = (int8_t)key_delta(keys, r.r + 1u, n);
        }
    }
    __syncthreads();
    for (uint32_t q = t; q < m; q += kThreads)
        climb<false>(T, nullptr, &I, out, n, m, q, T.box[q * 3u], T.box[q * 3u + 1u], T.box[q * 3u + 2u]);
    leave_roots(T, &I, 0u, m, roots + (size_t)blockIdx.x * kMaxRoots, nroots + blockIdx.x);
}

// The tree with four children a node, for walks (collider_hit): binary node i
// takes its children's children, or a child itself where it is a leaf. One
// thread per binary node (a walk from the root meets those at even depths).
// A child of more than a third of the node's leaves stands first: a walk
// pushes the children in this order and goes on with the last, so that it is
// in such a child only when no sibling of it waits on the stack. With 17 words
// waiting (no room for four more), at least six levels have some, and the walk
// is in at most 3^-6 = 1/729 of the leaves. Nodes of up to 32 leaves, which
// are quickly scanned, keep the order of the curve: it finds a collision
// sooner (16,384-lot city block 764 us, 766 with this rule, 773 with it for
// all nodes, 769 with all four children sorted by size).
__global__ void __launch_bounds__(256) k_wide(const u64* __restrict__ keys, uint32_t n, const uint32_t* nd,
                                              const int32_t* __restrict__ left, const int32_t* __restrict__ right,
                                              const int32_t* __restrict__ other_end,
                                              const float* __restrict__ node_aabb, const float* __restrict__ aabbs,
                                              const float4* __restrict__ coll, float4* __restrict__ wide) {
    const uint32_t nn = leaf_count(n, nd);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (nn < 2u || i >= nn - 1u) return;
    // a left child of [l, r] ends, and a right child begins, at the split
    const uint32_t far = (uint32_t)other_end[i], l = min(i, far), r = max(i, far);
    int32_t g[4];                        // the slots' subtrees
    uint32_t size[4];                    // their leaves, 0: no subtree
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int32_t c = h == 0 ? left[i] : right[i];
        const uint32_t at = (uint32_t)abs(c), first = h == 0 ? l : at, last = h == 0 ? at : r;
        g[2 * h] = c < 0 ? left[at] : c;
        g[2 * h + 1] = c < 0 ? right[at] : 0;
        size[2 * h] = c < 0 ? (uint32_t)abs(g[2 * h]) - first + 1u : 1u;
        size[2 * h + 1] = c < 0 ? last - (uint32_t)abs(g[2 * h + 1]) + 1u : 0u;
    }
    uint32_t big = 0, most = size[0];
#pragma unroll
    for (uint32_t q = 1; q < 4u; ++q) {
        big = size[q] > most ? q : big;
        most = max(most, size[q]);
    }
    if (r - l < 32u || most <= (r - l + 1u) / 3u) big = 0u;
#pragma unroll
    for (uint32_t q = 1; q < 4u; ++q) {
        const bool swap = q == big;
        const uint32_t s0 = size[0];
        const int32_t g0 = g[0];
        size[0] = swap ? size[q] : s0;
        g[0] = swap ? g[q] : g0;
        size[q] = swap ? s0 : size[q];
        g[q] = swap ? g0 : g[q];
    }
    float b[4][6];
    uint32_t ref[4], tag[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool there = size[q] != 0u;
        const float* src = nullptr;
        ref[q] = 0xFFFFFFFFu;            // kWideNone
        tag[q] = 0u;
        if (there && g[q] >= 0) {
            const uint32_t item = (uint32_t)keys[g[q]];
            ref[q] = item | 0x80000000u;        // kWideLeaf
            tag[q] = __float_as_uint(coll[(size_t)item * 5u + 3u].w) & 0xFFFFu;
            src = aabbs + (size_t)item * 6u;
        } else if (there) {
            ref[q] = (uint32_t)-g[q];
            src = node_aabb + (size_t)(-g[q]) * 6u;
        }
#pragma unroll
        for (int z = 0; z < 6; ++z) b[q][z] = there ? src[z] : (z < 3 ? INFINITY : -INFINITY);
    }
    float4* o = wide + (size_t)i * 8u;
#pragma unroll
    for (int z = 0; z < 6; ++z) o[z] = make_float4(b[0][z], b[1][z], b[2][z], b[3][z]);
    o[6] = make_float4(__uint_as_float(ref[0]), __uint_as_float(ref[1]), __uint_as_float(ref[2]),
                       __uint_as_float(ref[3]));
    o[7] = make_float4(__uint_as_float(l), __uint_as_float(r + 1u),
                       __uint_as_float(tag[0] | tag[1] << 16), __uint_as_float(tag[2] | tag[3] << 16));
}

} // namespace bvhk

// ---- host API ----
namespace {

using namespace bvhk;

uint32_t ceil_div(uint32_t a, uint32_t b) { return a / b + (a % b ? 1u : 0u); }

// A build's scratch for up to n leaves, in 8-byte words of one array: the
// other key buffer of the sort, its histogram rows and status words, and the
// open subtrees of the tree's levels.
struct Scratch {
    u64* keys = nullptr;
    u64* status = nullptr;
    Root* roots[2] = {nullptr, nullptr};     // written by even / odd levels
    uint32_t *rows = nullptr, *totals = nullptr, *tickets = nullptr, *nroots[2] = {nullptr, nullptr};
};
constexpr size_t hist_rows(size_t n) {
    const size_t b = (n + kThreads - 1u) / kThreads;
    return b < kHistBlocks ? b : kHistBlocks;
}
constexpr size_t scratch_words(size_t n) {
    const size_t tiles = (n + kTile - 1u) / kTile, wgs = (n + kTreeTile - 1u) / kTreeTile;
    const size_t up = (wgs + kTreeGroup - 1u) / kTreeGroup;
    return n + 2u + kPasses * kDigits * tiles + hist_rows(n) * (kThreads / 2u) + kThreads / 2u + 8u +
           (wgs + up) * (kMaxRoots * sizeof(Root) / 8u) + wgs / 2u + up / 2u + 8u;
}
Scratch scratch_at(void* base, size_t n) {
    const size_t tiles = (n + kTile - 1u) / kTile, wgs = (n + kTreeTile - 1u) / kTreeTile;
    const size_t up = (wgs + kTreeGroup - 1u) / kTreeGroup;
    Scratch c;
    u64* p = static_cast<u64*>(base);
    c.roots[0] = reinterpret_cast<Root*>(p); p += wgs * (kMaxRoots * sizeof(Root) / 8u);
    c.roots[1] = reinterpret_cast<Root*>(p); p += up * (kMaxRoots * sizeof(Root) / 8u);
    c.keys = p; p += n + 2u;
    c.status = p; p += kPasses * kDigits * tiles;
    c.rows = reinterpret_cast<uint32_t*>(p); p += hist_rows(n) * (kThreads / 2u);
    c.totals = reinterpret_cast<uint32_t*>(p); p += kThreads / 2u;
    c.tickets = reinterpret_cast<uint32_t*>(p); p += 8u;
    c.nroots[0] = reinterpret_cast<uint32_t*>(p); p += wgs / 2u + 4u;
    c.nroots[1] = reinterpret_cast<uint32_t*>(p);
    return c;
}

} // namespace

struct pga_lbvh {
    uint32_t capacity = 0;
    int device = 0;
    hipStream_t stream = nullptr;
    void* scratch_mem = nullptr;
    Scratch scratch;
    int32_t* other_end = nullptr;   // counted builds (pga_lbvh_enqueue_counted): see TreeOut
    float* bounds = nullptr;        // bounds partials; [0, 6) the folded scene box
    uint32_t* dev_words = nullptr;  // [0] leaf count of the last gather, [1] its overflow flag
    hipEvent_t e0 = nullptr, e1 = nullptr;
    std::string error;
};

namespace {

pga_status lfail(pga_lbvh* b, pga_status st, const std::string& m) {
    if (b) b->error = m;
    return st;
}

#define LHIP(b, expr)                                                                  \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess) return lfail(b, PGA_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Morton keys, sort and tree for n leaves (nd: the device count, n its
// bound), with a host scene box (mn, ex) or the device box `box`. other_end:
// see TreeOut.
hipError_t enqueue_build(const Scratch& c, hipStream_t s, const float* aabbs, uint32_t n, const uint32_t* nd,
                         const float mn[3], const float ex[3], const float* box, uint64_t* keys_out, int32_t* left,
                         int32_t* right, int32_t* parent, int32_t* leaf_parent, float* node_aabb,
                         int32_t* other_end) {
    const Scene scene{mn[0], mn[1], mn[2], ex[0], ex[1], ex[2], box};
    u64* keys = reinterpret_cast<u64*>(keys_out);
    if (n <= kSmallLeaves) {
        hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(kThreads), 0, s, aabbs, n, nd, scene, keys);
    } else {
        const uint32_t nb = ceil_div(n, kTile), rows = (uint32_t)hist_rows(n);
        hipLaunchKernelGGL(k_morton, dim3(rows), dim3(kThreads), 0, s, aabbs, n, nd, scene, keys, c.rows, c.status,
                           kPasses * kDigits * nb, c.tickets);
        hipLaunchKernelGGL(k_digit_totals, dim3(kPasses * kDigits / 64u), dim3(kThreads), 0, s, c.rows, rows,
                           c.totals);
        for (uint32_t pass = 0; pass < kPasses; ++pass)     // an even number of passes: the last one writes `keys`
            hipLaunchKernelGGL(k_sweep, dim3(nb), dim3(kThreads), 0, s, pass & 1u ? c.keys : keys,
                               pass & 1u ? keys : c.keys, n, nd, pass, c.totals,
                               c.status + (size_t)pass * kDigits * nb, c.tickets);
    }
    const TreeOut out{left, right, parent, leaf_parent, other_end, node_aabb};
    uint32_t groups = ceil_div(n, kTreeTile), level = 0;
    hipLaunchKernelGGL(k_tree_leaves, dim3(groups), dim3(kThreads), 0, s, aabbs, keys, n, nd, out, c.roots[0],
                       c.nroots[0]);
    while (groups > 1u) {
        const uint32_t next = ceil_div(groups, kTreeGroup), from = level & 1u;
        hipLaunchKernelGGL(k_tree_roots, dim3(next), dim3(kThreads), 0, s, keys, n, nd, out, c.roots[from],
                           c.nroots[from], groups, c.roots[from ^ 1u], c.nroots[from ^ 1u]);
        groups = next;
        ++level;
    }
    return hipGetLastError();
}

// ---- the allocation-free build (pga_lbvh_build_noalloc) ----
// Its scratch is this file-scope device array, for at most kNoAllocLeaves
// leaves (about 16.1 MiB, held by every GPU the library runs on until the
// process ends). Host code uses the address that hipGetSymbolAddress gives on
// each device, never the array's name.
constexpr uint32_t kNoAllocLeaves = PGA_LBVH_NOALLOC_MAX_LEAVES;
static __device__ __align__(256) u64 scratch[scratch_words(kNoAllocLeaves)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {nullptr};   // the array's address on each device
thread_local std::string g_noalloc_error;      // message of the last failed call on this thread

pga_status noalloc_fail(pga_status st, const std::string& m) {
    g_noalloc_error = m;
    return st;
}

// The array's address on the current device, looked up once per device.
pga_status scratch_on_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return noalloc_fail(PGA_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return noalloc_fail(PGA_ERR_UNSUPPORTED, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return noalloc_fail(PGA_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return PGA_OK;
}

} // namespace

extern "C" {

PGA_API pga_status pga_lbvh_build_noalloc(const float* aabbs, uint32_t n, const float scene_min[3],
                                          const float scene_max[3], uint64_t* keys, int32_t* left, int32_t* right,
                                          int32_t* parent, int32_t* leaf_parent, float* node_aabb, void* stream) {
    if (!aabbs || !scene_min || !scene_max || !keys || !left || !right || !parent || !leaf_parent || !node_aabb)
        return noalloc_fail(PGA_ERR_INVALID_ARG, "null argument");
    if (n < 2u || n > kNoAllocLeaves)
        return noalloc_fail(PGA_ERR_INVALID_ARG, "pga_lbvh_build_noalloc: need 2 <= n <= " +
                                                     std::to_string(kNoAllocLeaves) + " leaves, got " +
                                                     std::to_string(n));
    const float ex[3] = {scene_max[0] - scene_min[0], scene_max[1] - scene_min[1], scene_max[2] - scene_min[2]};
    if (!(ex[0] > 0.0f) || !(ex[1] > 0.0f) || !(ex[2] > 0.0f)) return noalloc_fail(PGA_ERR_INVALID_ARG, "empty scene box");
    void* base = nullptr;
    pga_status st = scratch_on_device(&base);
    if (st) return st;
    const hipError_t e = enqueue_build(scratch_at(base, kNoAllocLeaves), (hipStream_t)stream, aabbs, n, nullptr,
                                       scene_min, ex, nullptr, keys, left, right, parent, leaf_parent, node_aabb,
                                       nullptr);
    if (e != hipSuccess) return noalloc_fail(PGA_ERR_HIP, std::string("launch: ") + hipGetErrorString(e));
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_create(uint32_t capacity, int32_t device, void* stream, pga_lbvh** out) {
    if (!out || capacity < 2u || capacity > 0x7FFFFFFFu) return PGA_ERR_INVALID_ARG;
    pga_lbvh* b = new pga_lbvh();
    *out = b;
    b->capacity = capacity;
    if (device >= 0) LHIP(b, hipSetDevice(device));
    LHIP(b, hipGetDevice(&b->device));
    b->stream = (hipStream_t)stream;
    LHIP(b, hipMalloc(&b->scratch_mem, scratch_words(capacity) * 8u));
    b->scratch = scratch_at(b->scratch_mem, capacity);
    LHIP(b, hipMalloc((void**)&b->other_end, (size_t)capacity * 4u));
    LHIP(b, hipMalloc((void**)&b->bounds, 1024u * 6u * 4u));
    LHIP(b, hipMalloc((void**)&b->dev_words, 64u));
    LHIP(b, hipMemset(b->dev_words, 0, 64u));
    LHIP(b, hipEventCreate(&b->e0));
    LHIP(b, hipEventCreate(&b->e1));
    return PGA_OK;
}

PGA_API void pga_lbvh_destroy(pga_lbvh* b) {
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    else (void)hipDeviceSynchronize();
    (void)hipFree(b->scratch_mem); (void)hipFree(b->bounds);
    (void)hipFree(b->dev_words); (void)hipFree(b->other_end);
    if (b->e0) (void)hipEventDestroy(b->e0);
    if (b->e1) (void)hipEventDestroy(b->e1);
    delete b;
}

PGA_API const char* pga_lbvh_last_error(const pga_lbvh* b) { return b ? b->error.c_str() : g_noalloc_error.c_str(); }

PGA_API pga_status pga_lbvh_instance_aabbs(pga_lbvh* b, const pga_instance* instances, uint32_t n, int32_t planar,
                                           float* aabbs) {
    if (!b || (n && (!instances || !aabbs))) return lfail(b, PGA_ERR_INVALID_ARG, "null buffer");
    if (n == 0) return PGA_OK;
    hipLaunchKernelGGL(k_instance_aabbs, dim3((n + 255u) / 256u), dim3(256), 0, b->stream, instances, n,
                       planar ? 1u : 0u, aabbs);
    LHIP(b, hipGetLastError());
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_bounds(pga_lbvh* b, const float* aabbs, uint32_t n, float bounds[6]) {
    if (!b || !aabbs || !bounds || n == 0) return lfail(b, PGA_ERR_INVALID_ARG, "bad bounds arguments");
    const uint32_t blocks = std::min<uint32_t>(1024u, (n + 255u) / 256u);
    hipLaunchKernelGGL(k_bounds, dim3(blocks), dim3(256), 0, b->stream, aabbs, n, nullptr, b->bounds);
    hipLaunchKernelGGL(k_bounds_fold, dim3(1), dim3(256), 0, b->stream, b->bounds, blocks);
    LHIP(b, hipGetLastError());
    LHIP(b, hipMemcpyAsync(bounds, b->bounds, 6u * 4u, hipMemcpyDeviceToHost, b->stream));
    LHIP(b, hipStreamSynchronize(b->stream));
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_build(pga_lbvh* b, const float* aabbs, uint32_t n, const float scene_min[3],
                                  const float scene_max[3], uint64_t* keys, int32_t* left, int32_t* right,
                                  int32_t* parent, int32_t* leaf_parent, float* node_aabb) {
    if (!b || !aabbs || !scene_min || !scene_max || !keys || !left || !right || !parent || !leaf_parent || !node_aabb)
        return lfail(b, PGA_ERR_INVALID_ARG, "null argument");
    if (n < 2u || n > b->capacity)
        return lfail(b, PGA_ERR_INVALID_ARG, "need 2 <= n <= capacity (" + std::to_string(b->capacity) + ")");
    const float ex[3] = {scene_max[0] - scene_min[0], scene_max[1] - scene_min[1], scene_max[2] - scene_min[2]};
    if (!(ex[0] > 0.0f) || !(ex[1] > 0.0f) || !(ex[2] > 0.0f)) return lfail(b, PGA_ERR_INVALID_ARG, "empty scene box");
    LHIP(b, hipEventRecord(b->e0, b->stream));
    LHIP(b, enqueue_build(b->scratch, b->stream, aabbs, n, nullptr, scene_min, ex, nullptr, keys, left, right, parent,
                          leaf_parent, node_aabb, nullptr));
    LHIP(b, hipEventRecord(b->e1, b->stream));
    LHIP(b, hipStreamSynchronize(b->stream));
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_gather_instances(pga_lbvh* b, const pga_instance* const* buffers,
                                             const uint64_t* capacities, uint32_t n_types,
                                             const uint64_t* device_counts, uint32_t planar_mask, float* aabbs) {
    if (!b || !buffers || !capacities || !device_counts || !aabbs || n_types == 0 || n_types > PGA_MAX_TERMINALS)
        return lfail(b, PGA_ERR_INVALID_ARG, "bad gather arguments");
    GatherArgs g{};
    for (uint32_t t = 0; t < n_types; ++t) {
        if (!buffers[t] && capacities[t]) return lfail(b, PGA_ERR_INVALID_ARG, "null buffer with nonzero capacity");
        g.buf[t] = buffers[t];
        g.cap[t] = capacities[t];
    }
    g.ntypes = n_types;
    g.planar_mask = planar_mask;
    g.capacity = b->capacity;
    const uint32_t blocks = std::min<uint32_t>(kGatherBlocks, (b->capacity + 255u) / 256u);
    hipLaunchKernelGGL(k_gather_boxes, dim3(blocks), dim3(256), 0, b->stream, g,
                       reinterpret_cast<const unsigned long long*>(device_counts), aabbs, b->dev_words,
                       b->dev_words + 1);
    LHIP(b, hipGetLastError());
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_build_device(pga_lbvh* b, const float* aabbs, const float* scene_min,
                                         const float* scene_max, uint64_t* keys, int32_t* left, int32_t* right,
                                         int32_t* parent, int32_t* leaf_parent, float* node_aabb) {
    if (!b || !aabbs || !keys || !left || !right || !parent || !leaf_parent || !node_aabb)
        return lfail(b, PGA_ERR_INVALID_ARG, "null argument");
    if (!scene_min != !scene_max) return lfail(b, PGA_ERR_INVALID_ARG, "give both scene corners or neither");
    const uint32_t n = b->capacity;
    const uint32_t* nd = b->dev_words;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    LHIP(b, hipStreamIsCapturing(b->stream, &cs));
    const bool timed = cs == hipStreamCaptureStatusNone;
    if (timed) LHIP(b, hipEventRecord(b->e0, b->stream));
    if (scene_min) {
        const float ex[3] = {scene_max[0] - scene_min[0], scene_max[1] - scene_min[1], scene_max[2] - scene_min[2]};
        if (!(ex[0] > 0.0f) || !(ex[1] > 0.0f) || !(ex[2] > 0.0f))
            return lfail(b, PGA_ERR_INVALID_ARG, "empty scene box");
        LHIP(b, enqueue_build(b->scratch, b->stream, aabbs, n, nd, scene_min, ex, nullptr, keys, left, right, parent,
                              leaf_parent, node_aabb, nullptr));
    } else {
        const uint32_t blocks = std::min<uint32_t>(1024u, (n + 255u) / 256u);
        hipLaunchKernelGGL(k_bounds, dim3(blocks), dim3(256), 0, b->stream, aabbs, n, nd, b->bounds);
        hipLaunchKernelGGL(k_bounds_fold, dim3(1), dim3(256), 0, b->stream, b->bounds, blocks);
        const float zero[3] = {0.0f, 0.0f, 0.0f}, one[3] = {1.0f, 1.0f, 1.0f};
        LHIP(b, enqueue_build(b->scratch, b->stream, aabbs, n, nd, zero, one, b->bounds, keys, left, right, parent,
                              leaf_parent, node_aabb, nullptr));
    }
    if (timed) LHIP(b, hipEventRecord(b->e1, b->stream));
    return PGA_OK;
}

} // extern "C"

// The device-count build over a caller's count word (the colliders a
// multi-phase derivation stored, built between its phases by pga_api.cpp):
// min(*nd, capacity) leaves, the scene box from the device.
hipError_t pga_lbvh_enqueue_counted(pga_lbvh* b, const float* aabbs, const uint32_t* nd, uint64_t* keys,
                                    int32_t* left, int32_t* right, int32_t* parent, int32_t* leaf_parent,
                                    float* node_aabb, const float4* coll, float4* wide) {
    const uint32_t n = b->capacity;
    const uint32_t blocks = std::min<uint32_t>(1024u, (n + 255u) / 256u);
    hipLaunchKernelGGL(k_bounds, dim3(blocks), dim3(256), 0, b->stream, aabbs, n, nd, b->bounds);
    hipLaunchKernelGGL(k_bounds_fold, dim3(1), dim3(256), 0, b->stream, b->bounds, blocks);
    const float zero[3] = {0.0f, 0.0f, 0.0f}, one[3] = {1.0f, 1.0f, 1.0f};
    const hipError_t e = enqueue_build(b->scratch, b->stream, aabbs, n, nd, zero, one, b->bounds, keys, left, right,
                                       parent, leaf_parent, node_aabb, b->other_end);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_wide, dim3(ceil_div(n, 256u)), dim3(256), 0, b->stream, reinterpret_cast<const u64*>(keys), n,
                       nd, left, right, b->other_end, node_aabb, aabbs, coll, wide);
    return hipGetLastError();
}

extern "C" {

PGA_API pga_status pga_lbvh_leaf_count(pga_lbvh* b, uint32_t* n, int32_t* overflow) {
    if (!b || !n) return lfail(b, PGA_ERR_INVALID_ARG, "null argument");
    uint32_t w[2] = {0u, 0u};
    LHIP(b, hipMemcpyAsync(w, b->dev_words, sizeof(w), hipMemcpyDeviceToHost, b->stream));
    LHIP(b, hipStreamSynchronize(b->stream));
    *n = w[0];
    if (overflow) *overflow = w[1] ? 1 : 0;
    return PGA_OK;
}

PGA_API pga_status pga_lbvh_seconds(pga_lbvh* b, double* seconds) {
    if (!b || !seconds) return PGA_ERR_INVALID_ARG;
    float ms = 0.0f;
    LHIP(b, hipEventElapsedTime(&ms, b->e0, b->e1));
    *seconds = ms * 1e-3;
    return PGA_OK;
}

} // extern "C"
