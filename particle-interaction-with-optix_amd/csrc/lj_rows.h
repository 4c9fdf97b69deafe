// lj_rows.h -- sorting the rows of a CSR neighbour list: 16 lanes a row in registers, or a
// workgroup a row in the memory that holds it.
//
// The list calls find each particle's partners in walk order (cells, or the tree's
// leaves) and promise rows in ascending index order.  The reference has no lists; its
// OptiX programs visit a particle's partners in the order the hardware reports them
// (SDK/optixMultiSphereAABB/optixLJ.cu:134-176).
#pragma once

#include "lj_internal.h"
#include "lj_pair.h"

namespace lj {

constexpr int kSortThreads = 256;
constexpr int kRowLanes = 16;                                // lanes of a row: one DPP row
constexpr int kShortLanes = 4;                               // lanes of a short row
constexpr uint32_t kShortRow = 4 * kShortLanes;              // longest row that they sort
constexpr int kBlockRows = kSortThreads / kShortLanes;       // rows of a workgroup
constexpr uint32_t kRegRow = 16 * kRowLanes;                 // longest row sorted in registers
constexpr uint32_t kLdsRow = 4096;                           // longest row sorted in LDS

// One exchange across lanes: element r of a lane against element r (or, mirrored, K - 1
// - r) of its partner; the lanes with `bit` clear keep the smaller one.
template <int K, int CTRL, bool MIRROR>
__device__ inline void cross(uint32_t (&a)[K], unsigned bit) {
    const bool upper = (threadIdx.x & bit) != 0;
    uint32_t o[K];
#pragma unroll
    for (int r = 0; r < K; ++r) o[r] = from_lane<CTRL>(a[MIRROR ? K - 1 - r : r]);
#pragma unroll
    for (int r = 0; r < K; ++r) a[r] = upper ? max(a[r], o[r]) : min(a[r], o[r]);
}

// Exchange with the lane 4 away: the two halves of each 8 lanes mirrored, then each
// half mirrored back.
template <int K>
__device__ inline void cross4(uint32_t (&a)[K]) {
    const bool upper = (threadIdx.x & 4u) != 0;
    uint32_t o[K];
#pragma unroll
    for (int r = 0; r < K; ++r) o[r] = from_lane<kMirror4>(from_lane<kMirror8>(a[r]));
#pragma unroll
    for (int r = 0; r < K; ++r) a[r] = upper ? max(a[r], o[r]) : min(a[r], o[r]);
}

__device__ inline void order(uint32_t& lo, uint32_t& hi) {
    const uint32_t x = lo, y = hi;
    lo = min(x, y);
    hi = max(x, y);
}

// The exchanges at distances D, D / 2, ..., 1 inside a lane's K elements.
template <int K, int D>
__device__ inline void within(uint32_t (&a)[K]) {
    if constexpr (D >= 1) {
#pragma unroll
        for (int r = 0; r < K; ++r)
            if ((r & D) == 0) order(a[r], a[r + D]);
        within<K, D / 2>(a);
    }
}

// Stages 2, 4, ..., K of the sort inside a lane: each first compares mirrored elements
// of a block, then halves the distance, so every comparison puts the smaller first.
template <int K, int S>
__device__ inline void lane_stages(uint32_t (&a)[K]) {
    if constexpr (S <= K) {
#pragma unroll
        for (int b = 0; b < K; b += S)
#pragma unroll
            for (int r = 0; r < S / 2; ++r) order(a[b + r], a[b + S - 1 - r]);
        within<K, S / 4>(a);
        lane_stages<K, S * 2>(a);
    }
}

// Sorts the LANES K elements of a row (LANES 4 or 16), element lane K + r in register r of
// its lane (Batcher's bitonic sort, "Sorting networks and their applications", AFIPS 1968,
// in the form whose merges start with a mirrored comparison).
template <int K, int LANES>
__device__ inline void sort_regs(uint32_t (&a)[K]) {
    static_assert(LANES == 4 || LANES == 16, "lanes of a row");
    lane_stages<K, 2>(a);
    cross<K, kXor1, true>(a, 1u);  // blocks of 2 lanes
    within<K, K / 2>(a);
    cross<K, kMirror4, true>(a, 2u);  // of 4
    cross<K, kXor1, false>(a, 1u);
    within<K, K / 2>(a);
    if constexpr (LANES == 16) {
        cross<K, kMirror8, true>(a, 4u);  // of 8
        cross<K, kXor2, false>(a, 2u);
        cross<K, kXor1, false>(a, 1u);
        within<K, K / 2>(a);
        cross<K, kMirror16, true>(a, 8u);  // of 16
        cross4<K>(a);
        cross<K, kXor2, false>(a, 2u);
        cross<K, kXor1, false>(a, 1u);
        within<K, K / 2>(a);
    }
}

// K consecutive entries at any 4-byte address as one store of up to 16 bytes each.
struct __attribute__((packed, aligned(4))) Four {
    uint32_t v[4];
};

// Sorts from[0, m) (the row itself or a copy in LDS) into row[0, m), m <= LANES K.
template <int K, int LANES = kRowLanes>
__device__ inline void sort_row(const uint32_t* from, uint32_t* row, uint32_t m) {
    const uint32_t lane = threadIdx.x % LANES;
    uint32_t a[K];
    // striped loads (the order before the sort does not matter); places past the row's
    // end hold the largest value and stay behind every entry
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const uint32_t at = r * LANES + lane;
        a[r] = at < m ? from[at] : 0xffffffffu;
    }
    sort_regs<K, LANES>(a);
    const uint32_t first = lane * K;
#pragma unroll
    for (int r = 0; r < K; r += 4) {
        if (K >= 4 && first + r + 4 <= m) {
            *reinterpret_cast<Four*>(row + first + r) = Four{{a[r], a[r + 1], a[r + 2], a[r + 3]}};
        } else {
#pragma unroll
            for (int u = 0; u < 4 && r + u < K; ++u)
                if (first + r + u < m) row[first + r + u] = a[r + u];
        }
    }
}

// The wave's four rows (one per 16 lanes, m <= kRegRow) by the longest of them.
__device__ inline void sort_four_rows(const uint32_t* from, uint32_t* row, uint32_t m) {
    if (__any(m > 128u)) sort_row<16>(from, row, m);
    else if (__any(m > 64u)) sort_row<8>(from, row, m);
    else if (__any(m > 32u)) sort_row<4>(from, row, m);
    else if (__any(m > 0u)) sort_row<2>(from, row, m);
}

// The wave's sixteen rows (one per four lanes, m <= kShortRow) by the longest of them.
__device__ inline void sort_short_rows(const uint32_t* from, uint32_t* row, uint32_t m) {
    if (__any(m > 8u)) sort_row<4, 4>(from, row, m);
    else if (__any(m > 4u)) sort_row<2, 4>(from, row, m);
    else if (__any(m > 0u)) sort_row<1, 4>(from, row, m);
}

// The same sort over v[0, m) by the whole workgroup, for memory that its threads share
// (LDS or the row itself); a comparison with a place at or past m never exchanges.
__device__ inline void block_sort(uint32_t* v, uint32_t m) {
    uint32_t top = 2;
    while (top < m) top <<= 1;  // m <= 2^31
    for (uint32_t s = 2; s != 0 && s <= top; s <<= 1)
        for (uint32_t d = s >> 1; d > 0; d >>= 1) {
            for (uint32_t c = threadIdx.x; c < (top >> 1); c += kSortThreads) {
                const uint32_t in = c & (d - 1u), lo = ((c - in) << 1) + in;
                const uint32_t hi = d == (s >> 1) ? ((c - in) << 1) + (s - 1u) - in : lo + d;
                if (hi < m) {
                    const uint32_t x = v[lo], y = v[hi];
                    if (x > y) {
                        v[lo] = y;
                        v[hi] = x;
                    }
                }
            }
            __syncthreads();
        }
}

}  // namespace lj
