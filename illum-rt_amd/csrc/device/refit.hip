// Refit: new vertex positions, unchanged triangles and topology.
//
// Records are rebuilt per leaf slot with the host flattener's own functions
// (core/records.h), so a refit to the committed positions reproduces the
// committed records bit for bit.  A leaf child's box is the bounding box of
// its triangles' vertices, an inner child's box that of every triangle below
// it.  Leaf boxes therefore bound whole triangles even where the builder's
// early split clipping had bounded fragments (a fragment box lies inside the
// triangle's box, so every hit stays reachable).
//
// The builders partition their triangle lists in place, so the slots below a
// child are one range: its box is a range of the box tree (box_tree.h) that
// the record kernel builds over the slots as it goes.  What bounds it is
// latency: three launches, the gathers slot -> triangle -> vertices, and up to
// 2 log2(slots) independent box loads per child.  One launch per tree level,
// deepest first, took 22 dependent launches for the hall's tree (262,144
// triangles): 155 us, this 40 us.
//
// Min/max are select forms that never let a NaN coordinate into a box, so
// refit boxes are NaN-free.
#include "refit_kernels.h"

#include "../core/records.h"

namespace rt {
namespace dev {

namespace {

__device__ __forceinline__ vec3f vertex(const float *pos, uint32_t v) {
    return vec3f{pos[3ull * v], pos[3ull * v + 1], pos[3ull * v + 2]};
}

// One thread per slot (and per triangle, for the shading copy).
__global__ __launch_bounds__(kBoxBlock) void k_refit_records(refit_args a) {
    const uint32_t i = blockIdx.x * (uint32_t)kBoxBlock + threadIdx.x;
    box6 box = empty_box6();
    if (i < a.n_slots) {
        uint32_t t = a.slot_ids[i];
        vec3f A = vertex(a.pos, a.vidx[3ull * t]);
        vec3f B = vertex(a.pos, a.vidx[3ull * t + 1]);
        vec3f C = vertex(a.pos, a.vidx[3ull * t + 2]);
        a.tris[i] = a.tri == TRI_WOOP ? make_woop_rec(A, B, C) : make_exact_rec(A, B, C, t);
        box_grow(box, A.x, A.y, A.z);
        box_grow(box, B.x, B.y, B.z);
        box_grow(box, C.x, C.y, C.z);
        a.boxes[i] = box;
    }
    if (a.tri_geo && i < a.n_tris) {
        float *g = a.tri_geo + 12ull * i;
        for (int c = 0; c < 3; ++c) {
            vec3f p = vertex(a.pos, a.vidx[3ull * i + c]);
            g[4 * c] = p.x;
            g[4 * c + 1] = p.y;
            g[4 * c + 2] = p.z;
        }
    }
    if (blockIdx.x * (uint32_t)kBoxBlock < a.n_slots) box_levels(box, a.boxes, a.n_slots);   // uniform per block
}

// One thread per child.
__global__ __launch_bounds__(256) void k_refit_nodes(refit_args a) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t width = a.bvh == BVH2 ? 2u : 4u;
    if (i >= a.n_nodes * width) return;
    const uint2 r = a.ranges[i];
    const box6 b = box_of_range(a.boxes, a.n_slots, r.x, r.y);
    if (a.bvh == BVH2) {
        node2 &nd = static_cast<node2 *>(a.nodes)[i >> 1];
        float4 xy = make_float4(b.lo[0], b.hi[0], b.lo[1], b.hi[1]);
        float2 z = make_float2(b.lo[2], b.hi[2]);
        if (i & 1u) {
            *reinterpret_cast<float4 *>(&nd.rxlo) = xy;
            *reinterpret_cast<float2 *>(&nd.rzlo) = z;
        } else {
            *reinterpret_cast<float4 *>(&nd.lxlo) = xy;
            *reinterpret_cast<float2 *>(&nd.lzlo) = z;
        }
    } else {
        node4 &nd = static_cast<node4 *>(a.nodes)[i >> 2];
        const uint32_t c = i & 3u;
        nd.lox[c] = b.lo[0];
        nd.hix[c] = b.hi[0];
        nd.loy[c] = b.lo[1];
        nd.hiy[c] = b.hi[1];
        nd.loz[c] = b.lo[2];
        nd.hiz[c] = b.hi[2];
    }
}

} // namespace

hipError_t launch_refit(const refit_args &a, hipStream_t stream) {
    const uint32_t n = a.n_slots > a.n_tris ? a.n_slots : a.n_tris;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_refit_records, dim3((n + kBoxBlock - 1) / kBoxBlock), dim3(kBoxBlock), 0, stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.n_nodes == 0) return e;
    e = launch_box_tree_top(a.boxes, a.n_slots, stream);
    if (e != hipSuccess) return e;
    const uint32_t children = a.n_nodes * (a.bvh == BVH2 ? 2u : 4u);
    hipLaunchKernelGGL(k_refit_nodes, dim3((children + 255) / 256), dim3(256), 0, stream, a);
    return hipGetLastError();
}

} // namespace dev
} // namespace rt
