// Bounds of any range of leaf slots from a binary tree of boxes over them:
// level 0 is one box per slot, entry j of level k the union of entries 2j and
// 2j + 1 of level k - 1.  A range is the union of at most two entries a level,
// all independent loads, so the boxes of every node of a BVH whose subtrees
// are slot ranges come from one launch -- instead of one dependent launch per
// tree level, or a bottom-up climb through device-scope counters, which
// flushes an XCD's L2 at every step.
//
// Min/max are the select forms of glm::min/max (aabb::grow,
// libgi/intersect.h:9-15) from an empty box (+inf, -inf): a NaN coordinate
// never enters a box, and the union does not depend on its order.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rt {
namespace dev {

struct box6 {
    float lo[3], hi[3];
};

__device__ __forceinline__ box6 empty_box6() {
    return box6{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
}

__device__ __forceinline__ void box_grow(box6 &b, float x, float y, float z) {
    b.lo[0] = (x < b.lo[0]) ? x : b.lo[0];
    b.lo[1] = (y < b.lo[1]) ? y : b.lo[1];
    b.lo[2] = (z < b.lo[2]) ? z : b.lo[2];
    b.hi[0] = (b.hi[0] < x) ? x : b.hi[0];
    b.hi[1] = (b.hi[1] < y) ? y : b.hi[1];
    b.hi[2] = (b.hi[2] < z) ? z : b.hi[2];
}

__device__ __forceinline__ void box_merge(box6 &b, const box6 &c) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = (c.lo[k] < b.lo[k]) ? c.lo[k] : b.lo[k];
        b.hi[k] = (b.hi[k] < c.hi[k]) ? c.hi[k] : b.hi[k];
    }
}

// Boxes of all levels over n slots (each level half the one below, rounded
// up, one after the other).
inline size_t box_tree_entries(uint32_t n) {
    size_t sum = 0;
    for (size_t m = n; m > 1; m = (m + 1) / 2) sum += m;
    return sum + 1;
}

// The union of slots [a, b) of n.
__device__ __forceinline__ box6 box_of_range(const box6 *level, uint32_t n, uint32_t a, uint32_t b) {
    box6 r = empty_box6();
    while (a < b) {
        if (a & 1u) box_merge(r, level[a++]);
        if (b & 1u) box_merge(r, level[--b]);
        level += n;
        n = (n + 1) >> 1;
        a >>= 1;
        b >>= 1;
    }
    return r;
}

constexpr int kBoxBlock = 1024;   // slots (and threads) per block of a level-building kernel

// Ten levels above the entries [blockIdx.x * kBoxBlock, + kBoxBlock) of a
// level of n entries that starts at `level`; thread t holds entry t (an empty
// box past the end) and has written it.  Every thread of the block calls it.
__device__ __forceinline__ void box_levels(box6 mine, box6 *level, uint32_t n) {
    __shared__ box6 wave_box[kBoxBlock / 64];
    const uint32_t t = threadIdx.x, lane = t & 63u;
    uint32_t j = blockIdx.x * (uint32_t)kBoxBlock + t;
#pragma unroll
    for (int k = 1; k <= 6; ++k) {
        if (n <= 1) return;   // the top is written (uniform over the grid)
        level += n;
        n = (n + 1) >> 1;
        j >>= 1;
        box6 other;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            other.lo[c] = __shfl_down(mine.lo[c], 1u << (k - 1), 64);
            other.hi[c] = __shfl_down(mine.hi[c], 1u << (k - 1), 64);
        }
        box_merge(mine, other);   // only lanes that are multiples of 2^k hold a box of this level
        if ((lane & ((1u << k) - 1u)) == 0 && j < n) level[j] = mine;
    }
    if (lane == 0) wave_box[t >> 6] = mine;
    __syncthreads();
#pragma unroll
    for (int k = 1; k <= 4; ++k) {
        if (n <= 1) return;
        level += n;
        n = (n + 1) >> 1;
        const uint32_t per = 16u >> k, e = blockIdx.x * per + t;
        box6 b;
        const bool mine_too = t < per;
        if (mine_too) {
            b = wave_box[2 * t];
            box_merge(b, wave_box[2 * t + 1]);
        }
        __syncthreads();
        if (mine_too) {
            wave_box[t] = b;
            if (e < n) level[e] = b;
        }
        __syncthreads();
    }
}

// The levels above level 10 of a tree over n slots whose first ten levels a
// kernel of kBoxBlock-slot blocks has written.
hipError_t launch_box_tree_top(box6 *tree, uint32_t n, hipStream_t stream);

} // namespace dev
} // namespace rt
