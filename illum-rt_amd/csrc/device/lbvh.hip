// Linear BVH built on the device (Karras, "Maximizing parallelism in the
// construction of BVHs, octrees, and k-d trees", HPG 2012), written straight
// into the flattened layout the trace kernels read.
//
//   1. per triangle: shading record and vertex indices, bounding box, index
//      and material checks, and the centre of the box (the reduction of the
//      centres' bounds runs in two passes, one partial per block);
//   2. 63-bit Morton code of the centre, 21 bits per axis over those bounds;
//   3. radix sort of (code, triangle) pairs (rocPRIM);
//   4. triangle records in Morton order, and the box tree over them
//      (box_tree.h);
//   5. the binary radix tree over the sorted codes, one thread per inner node;
//      equal codes are told apart by their sorted positions.  A node is its
//      leaf range and split; a subtree of at most `max_leaf` triangles becomes
//      one leaf of its parent (one slot range);
//   6. pre-order numbering of the emitted nodes: a node's number is the count
//      of emitted nodes that begin before its range, plus the longer ones that
//      begin with it.  The nodes that begin at one position are a chain of
//      left children below a right child (or the root), which one thread
//      walks; an exclusive scan of the chains' lengths gives the numbers, the
//      difference to the scan of the chains that end at a position the number
//      of nodes above each leaf, so the depth;
//   7. nodes written in that order, each child's box a range of the box tree;
//      the surfaces of inner and leaf boxes, summed per block, go to the host.
//
// What bounds it is the latency of its launches (20 of them the sort's) and
// of short dependent loads; no step waits on another wavefront.  The hall's
// 262,144 triangles: 207 us on the device, 334 us a call.  The climb from the leaves to the
// root through acquire/release counters that gave boxes and subtree sizes
// before took 981 us of 1,300 (and the call 4.7 ms, most of it the copy of
// the tree to the host and its check there): at device scope every step writes back and
// invalidates the XCD's L2.
//
// Leaf boxes bound whole triangles.  Min/max are the select forms of
// glm::min/max starting from empty boxes, so a NaN coordinate never enters a
// box.  This tree is not the reference's SAH tree: closest hits agree with
// brute force up to equal-t ties and grazing hits, not bit for bit.
#include "lbvh_kernels.h"

#include "../core/records.h"
#include "box_tree.h"

#include <cstring>

#include <rocprim/rocprim.hpp>

namespace rt {
namespace dev {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kEmitBlock = 1024;   // few area sums to read back
constexpr uint32_t kMortonBits = 21;
constexpr uint32_t kScanTile = 1024;   // positions per block of the numbering scan

// Scratch layout (offsets in bytes, 256-aligned), for n triangles, m = n - 1.
struct scratch_map {
    size_t tri_box, partial, bounds, keys0, keys1, vals0, vals1, other, split, rank, chains, tiles, begins, boxes,
        sort_tmp, sort_bytes, total;
};

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

scratch_map map_scratch(uint32_t n, size_t sort_bytes) {
    scratch_map s{};
    size_t m = n > 1 ? n - 1 : 1, nb = (n + kBlock - 1) / kBlock + 1, off = 0;
    auto take = [&](size_t bytes) {
        size_t at = off;
        off = align256(off + bytes);
        return at;
    };
    s.tri_box = take(sizeof(box6) * (size_t)n);
    s.partial = take(sizeof(box6) * nb);
    s.bounds = take(sizeof(box6));
    s.keys0 = take(8ull * n);
    s.keys1 = take(8ull * n);
    s.vals0 = take(4ull * n);
    s.vals1 = take(4ull * n);
    s.other = take(4 * m);
    s.split = take(4 * m);
    s.rank = take(4 * m);
    s.chains = take(8ull * n);
    s.tiles = take(8 * ((size_t)n / kScanTile + 1));
    s.begins = take(4ull * n);
    s.boxes = take(sizeof(box6) * box_tree_entries(n));
    s.sort_bytes = sort_bytes;
    s.sort_tmp = take(sort_bytes);
    s.total = off;
    return s;
}

size_t sort_storage(uint32_t n) {
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, (uint64_t *)nullptr, (uint64_t *)nullptr, (uint32_t *)nullptr,
                                    (uint32_t *)nullptr, n, 0, 3 * kMortonBits);
    return bytes;
}

template <class T> T *at(void *base, size_t off) {
    return reinterpret_cast<T *>(static_cast<char *>(base) + off);
}

// ---- 1. triangle boxes, checks, shading copy, partial bounds of the box centres ----
__global__ __launch_bounds__(kBlock) void k_tri_boxes(lbvh_in in, lbvh_out out, box6 *tri_box, box6 *partial) {
    __shared__ box6 sh[kBlock / 64];
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    box6 c = empty_box6();
    if (i < in.n_tris) {
        box6 b = empty_box6();
        bool bad = false;
        float4 *geo = reinterpret_cast<float4 *>(out.tri_geo) + 3ull * i;
        const uint32_t m = in.mat ? in.mat[i] : 0u;
        for (int k = 0; k < 3; ++k) {
            uint32_t v = in.vidx[3ull * i + k];
            out.tri_vidx[3ull * i + k] = v;
            if (v >= in.n_vert) {
                bad = true;
                v = 0;
            }
            const float x = in.pos[3ull * v], y = in.pos[3ull * v + 1], z = in.pos[3ull * v + 2];
            geo[k] = make_float4(x, y, z, k ? 0.0f : __uint_as_float(m));
            box_grow(b, x, y, z);
        }
        if (bad) atomicAdd(out.result->counts + 2, 1u);
        if (m >= in.n_mats) atomicAdd(out.result->counts + 4, 1u);
        tri_box[i] = b;
        box_grow(c, 0.5f * (b.lo[0] + b.hi[0]), 0.5f * (b.lo[1] + b.hi[1]), 0.5f * (b.lo[2] + b.hi[2]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        box6 o;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            o.lo[k] = __shfl_down(c.lo[k], off, 64);
            o.hi[k] = __shfl_down(c.hi[k], off, 64);
        }
        box_merge(c, o);
    }
    if ((threadIdx.x & 63u) == 0) sh[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; ++w) box_merge(c, sh[w]);
        partial[blockIdx.x] = c;
    }
}

__global__ __launch_bounds__(kBoxBlock) void k_reduce_bounds(const box6 *partial, uint32_t n_part, box6 *bounds) {
    __shared__ box6 sh[kBoxBlock];
    box6 c = empty_box6();
    for (uint32_t i = threadIdx.x; i < n_part; i += kBoxBlock) box_merge(c, partial[i]);
    sh[threadIdx.x] = c;
    __syncthreads();
    for (int w = kBoxBlock / 2; w > 0; w >>= 1) {
        if (threadIdx.x < (unsigned)w) box_merge(sh[threadIdx.x], sh[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) *bounds = sh[0];
}

// ---- 2. Morton codes ----
__device__ __forceinline__ uint64_t spread21(uint32_t x) {
    uint64_t v = x & 0x1fffffu;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

__global__ __launch_bounds__(kBlock) void k_morton(const box6 *tri_box, const box6 *bounds, uint32_t n,
                                                   uint64_t *keys, uint32_t *vals) {
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const box6 b = tri_box[i];
    const box6 bb = *bounds;
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        float ext = bb.hi[k] - bb.lo[k];
        float scale = ext > 0.0f ? (float)((1u << kMortonBits) - 1) / ext : 0.0f;
        float x = (0.5f * (b.lo[k] + b.hi[k]) - bb.lo[k]) * scale;
        x = fminf(fmaxf(x, 0.0f), (float)((1u << kMortonBits) - 1));   // NaN -> 0
        q[k] = (uint32_t)x;
    }
    keys[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    vals[i] = i;
}

// ---- 5. binary radix tree ----
// Common-prefix length of sorted codes a and b; -1 outside [0, n).
__device__ __forceinline__ int delta(const uint64_t *keys, int n, int a, int b) {
    if (b < 0 || b >= n) return -1;
    uint64_t ka = keys[a], kb = keys[b];
    if (ka == kb) return 64 + __clz((uint32_t)a ^ (uint32_t)b);
    return __clzll(ka ^ kb);
}

// Inner node i covers the leaves between i and other[i]; its left child ends
// at split[i].
__global__ __launch_bounds__(kBlock) void k_karras(const uint64_t *keys, int n, int32_t *other, int32_t *split) {
    int i = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    other[i] = j;
    split[i] = i + s * d + (d < 0 ? -1 : 0);
}

// The left child of a node with split g covers first .. g and is inner node g
// (or leaf g), the right one g + 1 .. last, inner node (or leaf) g + 1.
struct tree_view {
    int n, max_leaf;
    const int32_t *other, *split;
};
__device__ __forceinline__ bool emitted(const tree_view &v, int first, int last) {
    return last - first + 1 > v.max_leaf;
}

// ---- 6. pre-order numbers ----
// Thread p walks the chain of emitted nodes that begin at leaf p from its
// longest (inner node p, when it covers p .. other[p]) down the left
// children, giving each its place in the chain, and counts the chain of
// those that end at p (inner node p, when it covers other[p] .. p; the root's
// right children for the last leaf).  chains[p] = (begin here) << 32 | end
// here; tiles: their sums over kScanTile positions.
__global__ __launch_bounds__(kScanTile) void k_chains(tree_view v, int32_t *rank, uint64_t *chains, uint64_t *tiles) {
    __shared__ uint64_t sum;
    if (threadIdx.x == 0) sum = 0;
    __syncthreads();
    const int p = (int)(blockIdx.x * kScanTile + threadIdx.x);
    uint32_t begins = 0, ends = 0;
    if (p < v.n) {
        const int o = p < v.n - 1 ? v.other[p] : 0;
        if (p < v.n - 1 && o > p) {
            // a chain is at most v.n long: every step shortens the range
            for (int i = p, last = o; emitted(v, p, last);) {
                rank[i] = (int32_t)begins++;
                last = v.split[i];
                if (last <= p || last >= v.n - 1) break;
                i = last;
            }
        }
        // the chain ending at p: its longest node is inner node p, the root for the last leaf
        int i = p < v.n - 1 ? (o < p ? p : -1) : 0, first = p < v.n - 1 ? o : 0;
        while (i >= 0 && emitted(v, first, p)) {
            ++ends;
            first = v.split[i] + 1;
            if (first >= p) break;
            i = first;
        }
        chains[p] = ((uint64_t)begins << 32) | ends;
    }
    uint64_t x = ((uint64_t)begins << 32) | ends;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down((unsigned long long)x, off, 64);
    if ((threadIdx.x & 63u) == 0) atomicAdd(reinterpret_cast<unsigned long long *>(&sum), (unsigned long long)x);
    __syncthreads();
    if (threadIdx.x == 0) tiles[blockIdx.x] = sum;
}

__device__ __forceinline__ uint64_t wave_inclusive(uint64_t x, uint32_t lane) {
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint64_t u = __shfl_up((unsigned long long)x, off, 64);
        if (lane >= off) x += u;
    }
    return x;
}

// Exclusive sums of the block's values (kScanTile threads); `total` the whole.
__device__ __forceinline__ uint64_t block_exclusive(uint64_t x, uint64_t *sh, uint64_t &total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t incl = wave_inclusive(x, lane);
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    uint64_t before = 0;
    total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kScanTile / 64; ++w) {
        const uint64_t s = sh[w];
        before += w < wave ? s : 0;
        total += s;
    }
    __syncthreads();
    return before + incl - x;
}

// The tiles' exclusive sums, in place; the number of emitted nodes.
__global__ __launch_bounds__(kScanTile) void k_scan_tiles(uint64_t *tiles, uint32_t n_tiles, uint32_t *counts) {
    __shared__ uint64_t sh[kScanTile / 64];
    uint64_t carry = 0, total;
    for (uint32_t base = 0; base < n_tiles; base += kScanTile) {
        const uint32_t j = base + threadIdx.x;
        const uint64_t e = block_exclusive(j < n_tiles ? tiles[j] : 0, sh, total);
        if (j < n_tiles) tiles[j] = carry + e;
        carry += total;
    }
    if (threadIdx.x == 0) counts[0] = (uint32_t)(carry >> 32);
}

// begins[p] = emitted nodes that begin before leaf p; the largest number of
// emitted nodes above one leaf is the depth.
__global__ __launch_bounds__(kScanTile) void k_number(const uint64_t *chains, const uint64_t *tiles, uint32_t n,
                                                      uint32_t *begins, uint32_t *counts) {
    __shared__ uint64_t sh[kScanTile / 64];
    __shared__ uint32_t deepest;
    const uint32_t p = blockIdx.x * kScanTile + threadIdx.x;
    if (threadIdx.x == 0) deepest = 0;
    const uint64_t mine = p < n ? chains[p] : 0;
    uint64_t total;
    const uint64_t e = tiles[blockIdx.x] + block_exclusive(mine, sh, total);
    uint32_t depth = 0;
    if (p < n) {
        begins[p] = (uint32_t)(e >> 32);
        depth = (uint32_t)(e >> 32) + (uint32_t)(mine >> 32) - (uint32_t)e;   // begun up to p, not ended before p
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) depth = max(depth, __shfl_down(depth, off, 64));
    if ((threadIdx.x & 63u) == 0) atomicMax(&deepest, depth);
    __syncthreads();
    // atomics on one word take 11 ns each: only a block that raises it adds one
    if (threadIdx.x == 0 && deepest > __hip_atomic_load(counts + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(counts + 1, deepest);
}

// ---- 7. flattened nodes and triangle records ----
// Child covering leaves [first, last] of inner node index c.
__device__ __forceinline__ int32_t child_ref(const tree_view &v, const int32_t *rank, const uint32_t *begins, int first,
                                             int last, int c) {
    if (!emitted(v, first, last)) return make_leaf_ref((uint32_t)first, (uint32_t)(last - first + 1));
    return (int32_t)(begins[first] + (uint32_t)rank[c]);
}

__device__ __forceinline__ float half_area(const box6 &b) {
    const float x = b.hi[0] - b.lo[0], y = b.hi[1] - b.lo[1], z = b.hi[2] - b.lo[2];
    return x >= 0.0f && y >= 0.0f && z >= 0.0f ? x * y + (x + y) * z : 0.0f;
}

// Inner node i; area.x and area.y: half the surface of its inner children's
// boxes and of its leaves'.
__device__ __forceinline__ void emit_node(const tree_view &v, int i, const int32_t *rank, const uint32_t *begins,
                                          const box6 *boxes, node2 *nodes, lbvh_result *result, float2 &area) {
    uint32_t *counts = result->counts;
    const int o = v.other[i], first = min(i, o), last = max(i, o), g = v.split[i];
    if (!emitted(v, first, last)) return;
    // what the host checks of an uploaded tree: the node and its inner
    // children inside the array, children after their parent, and slots
    // inside the records
    if (first < 0 || last >= v.n || g < first || g >= last) {
        atomicAdd(counts + 3, 1u);
        return;
    }
    const uint32_t total = counts[0], at = begins[first] + (uint32_t)rank[i];
    const int32_t l = child_ref(v, rank, begins, first, g, g), r = child_ref(v, rank, begins, g + 1, last, g + 1);
    if (at >= total || (l >= 0 && ((uint32_t)l <= at || (uint32_t)l >= total)) ||
        (r >= 0 && ((uint32_t)r <= at || (uint32_t)r >= total))) {
        atomicAdd(counts + 3, 1u);
        return;
    }
    const box6 bl = box_of_range(boxes, (uint32_t)v.n, (uint32_t)first, (uint32_t)g + 1u);
    const box6 br = box_of_range(boxes, (uint32_t)v.n, (uint32_t)g + 1u, (uint32_t)last + 1u);
    float4 *out = reinterpret_cast<float4 *>(nodes + at);
    out[0] = make_float4(bl.lo[0], bl.hi[0], bl.lo[1], bl.hi[1]);
    out[1] = make_float4(br.lo[0], br.hi[0], br.lo[1], br.hi[1]);
    out[2] = make_float4(bl.lo[2], bl.hi[2], br.lo[2], br.hi[2]);
    out[3] = make_float4(__int_as_float(l), __int_as_float(r), 0.0f, 0.0f);
    if (i == 0) {
        result->root_ref = 0;
        float4 *copy = reinterpret_cast<float4 *>(&result->root);
        for (int k = 0; k < 4; ++k) copy[k] = out[k];
    }
    const float al = half_area(bl), ar = half_area(br);
    area.x = (l >= 0 ? al : 0.0f) + (r >= 0 ? ar : 0.0f);
    area.y = (l >= 0 ? 0.0f : al) + (r >= 0 ? 0.0f : ar);
}

__global__ __launch_bounds__(kEmitBlock) void k_emit(tree_view v, const int32_t *rank, const uint32_t *begins,
                                                 const box6 *boxes, node2 *nodes, lbvh_result *result, float2 *areas) {
    __shared__ float2 sum[kEmitBlock / 64];
    const int i = (int)(blockIdx.x * kEmitBlock + threadIdx.x);
    float2 area = make_float2(0.0f, 0.0f);
    if (i < v.n - 1) emit_node(v, i, rank, begins, boxes, nodes, result, area);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        area.x += __shfl_down(area.x, off, 64);
        area.y += __shfl_down(area.y, off, 64);
    }
    if ((threadIdx.x & 63u) == 0) sum[threadIdx.x >> 6] = area;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kEmitBlock / 64; ++w) {
            area.x += sum[w].x;
            area.y += sum[w].y;
        }
        areas[blockIdx.x] = area;
    }
}

// ---- 4. records in Morton order and the lower levels of the box tree ----
__global__ __launch_bounds__(kBoxBlock) void k_records(lbvh_in in, lbvh_out out, const uint32_t *vals,
                                                       box6 *boxes) {
    const uint32_t k = blockIdx.x * (uint32_t)kBoxBlock + threadIdx.x;
    box6 box = empty_box6();
    if (k < in.n_tris) {
        const uint32_t t = vals[k];
        // the shading record holds the corners
        const float4 *geo = reinterpret_cast<const float4 *>(out.tri_geo) + 3ull * t;
        const float4 a = geo[0], b = geo[1], c = geo[2];
        const vec3f A{a.x, a.y, a.z}, B{b.x, b.y, b.z}, C{c.x, c.y, c.z};
        out.tris[k] = in.tri == TRI_WOOP ? make_woop_rec(A, B, C) : make_exact_rec(A, B, C, t);
        out.slot_ids[k] = t;
        box_grow(box, A.x, A.y, A.z);
        box_grow(box, B.x, B.y, B.z);
        box_grow(box, C.x, C.y, C.z);
        boxes[k] = box;
    }
    box_levels(box, boxes, in.n_tris);
}

// Trees of at most max_leaf triangles (including one triangle): the root is a leaf.
__global__ void k_root_leaf(uint32_t n, lbvh_result *result) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        result->root_ref = n ? make_leaf_ref(0u, n) : kInvalidRef;
        result->counts[0] = 0;
        result->counts[1] = 0;
    }
}

__global__ void k_clear(uint32_t *counts) {
    if (threadIdx.x < 5) counts[threadIdx.x] = 0u;
}

inline dim3 grid_for(uint32_t n) { return dim3((n + kBlock - 1) / kBlock); }

} // namespace

uint32_t lbvh_area_blocks(uint32_t n_tris) { return n_tris > 1 ? (n_tris - 1 + kEmitBlock - 1) / kEmitBlock : 0u; }

size_t lbvh_scratch_bytes(uint32_t n_tris) {
    if (n_tris == 0) return 256;
    return map_scratch(n_tris, sort_storage(n_tris)).total;
}

hipError_t launch_lbvh(const lbvh_in &in, const lbvh_out &out, void *scratch, hipStream_t s) {
    const uint32_t n = in.n_tris;
    uint32_t *counts = out.result->counts;   // an address, not read here
    hipLaunchKernelGGL(k_clear, dim3(1), dim3(64), 0, s, counts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (n == 0) {
        hipLaunchKernelGGL(k_root_leaf, dim3(1), dim3(64), 0, s, 0u, out.result);
        return hipGetLastError();
    }
    const scratch_map sm = map_scratch(n, sort_storage(n));
    box6 *tri_box = at<box6>(scratch, sm.tri_box), *partial = at<box6>(scratch, sm.partial);
    box6 *bounds = at<box6>(scratch, sm.bounds), *boxes = at<box6>(scratch, sm.boxes);
    uint64_t *keys0 = at<uint64_t>(scratch, sm.keys0), *keys1 = at<uint64_t>(scratch, sm.keys1);
    uint32_t *vals0 = at<uint32_t>(scratch, sm.vals0), *vals1 = at<uint32_t>(scratch, sm.vals1);
    const uint32_t nb = (n + kBlock - 1) / kBlock;

    hipLaunchKernelGGL(k_tri_boxes, grid_for(n), dim3(kBlock), 0, s, in, out, tri_box, partial);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_reduce_bounds, dim3(1), dim3(kBoxBlock), 0, s, partial, nb, bounds);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_morton, grid_for(n), dim3(kBlock), 0, s, tri_box, bounds, n, keys0, vals0);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    size_t sort_bytes = sm.sort_bytes;
    e = rocprim::radix_sort_pairs(at<void>(scratch, sm.sort_tmp), sort_bytes, keys0, keys1, vals0, vals1, n, 0,
                                  3 * kMortonBits, s);
    if (e != hipSuccess) return e;

    // records in Morton order (every slot is one triangle)
    hipLaunchKernelGGL(k_records, dim3((n + kBoxBlock - 1) / kBoxBlock), dim3(kBoxBlock), 0, s, in, out, vals1, boxes);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (n <= (uint32_t)in.max_leaf) {
        hipLaunchKernelGGL(k_root_leaf, dim3(1), dim3(64), 0, s, n, out.result);
        return hipGetLastError();
    }
    if ((e = launch_box_tree_top(boxes, n, s)) != hipSuccess) return e;

    int32_t *other = at<int32_t>(scratch, sm.other), *split = at<int32_t>(scratch, sm.split);
    int32_t *rank = at<int32_t>(scratch, sm.rank);
    uint64_t *chains = at<uint64_t>(scratch, sm.chains), *tiles = at<uint64_t>(scratch, sm.tiles);
    uint32_t *begins = at<uint32_t>(scratch, sm.begins);
    const tree_view v{(int)n, in.max_leaf, other, split};
    const uint32_t n_tiles = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_karras, grid_for(n - 1), dim3(kBlock), 0, s, keys1, (int)n, other, split);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_chains, dim3(n_tiles), dim3(kScanTile), 0, s, v, rank, chains, tiles);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kScanTile), 0, s, tiles, n_tiles, counts);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_number, dim3(n_tiles), dim3(kScanTile), 0, s, chains, tiles, n, begins, counts);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_emit, dim3(lbvh_area_blocks(n)), dim3(kEmitBlock), 0, s, v, rank, begins, boxes, out.nodes, out.result,
                       out.areas);
    return hipGetLastError();
}

} // namespace dev
} // namespace rt
