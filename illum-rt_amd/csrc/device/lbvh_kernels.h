// Device BVH construction (linear BVH) straight into the flattened layout of
// core/layout.h.
#pragma once

#include <hip/hip_runtime.h>

#include "../core/layout.h"

#include <cstdint>

namespace rt {
namespace dev {

struct lbvh_in {
    const float *pos;        // 3 floats per vertex
    const uint32_t *vidx;    // 3 vertex indices per triangle
    const uint32_t *mat;     // material id per triangle, or null (all 0)
    uint32_t n_vert, n_tris, n_mats;
    int max_leaf;            // leaf size bound (1..32)
    int tri;                 // tri_format of the records
};

struct lbvh_out {
    node2 *nodes;            // n_tris - 1 entries reserved (at most that many are written)
    tri_rec *tris;           // n_tris records, slot k = k-th triangle in Morton order
    uint32_t *slot_ids;      // n_tris
    float *tri_geo;          // 12 floats per triangle: A.xyz + material bits, B.xyz, C.xyz (w words 0)
    uint32_t *tri_vidx;      // copy of the 3 vertex indices per triangle
    struct lbvh_result *result;   // device memory
    float2 *areas;                // lbvh_area_blocks: sums of half the surface of inner children's boxes and of leaves'
                                  // (written for trees with inner nodes)
};

// What the host reads back of a build.
struct lbvh_result {
    int32_t root_ref;        // root inner node 0, or the leaf reference of a one-leaf tree
    uint32_t counts[5];      // emitted inner nodes, depth (inner nodes on the longest path), triangles with a bad
                             // vertex index, nodes that failed the layout check, triangles with a bad material id
    uint32_t pad[2];
    node2 root;              // copy of inner node 0 (trees that have one)
};

uint32_t lbvh_area_blocks(uint32_t n_tris);

// Scratch the build needs, in bytes, for n_tris triangles.
size_t lbvh_scratch_bytes(uint32_t n_tris);

// Builds the tree on `stream`; `scratch` holds lbvh_scratch_bytes(n_tris)
// bytes.  Results are valid once the stream reaches the end of the build.
hipError_t launch_lbvh(const lbvh_in &in, const lbvh_out &out, void *scratch, hipStream_t stream);

} // namespace dev
} // namespace rt
