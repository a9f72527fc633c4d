// Device refit of a committed scene to new vertex positions: same triangles,
// same tree topology, new triangle records and node boxes.
#pragma once

#include <hip/hip_runtime.h>

#include "../core/layout.h"
#include "box_tree.h"

#include <cstdint>

namespace rt {
namespace dev {

struct refit_args {
    void *nodes;               // node2[] or node4[]
    int bvh;                   // bvh_format
    uint32_t n_nodes;
    tri_rec *tris;             // one record per leaf slot
    const uint32_t *slot_ids;  // slot -> triangle id
    int tri;                   // tri_format
    uint32_t n_slots;
    float *tri_geo;            // 12 floats per triangle (A.xyz + material bits, B.xyz, C.xyz), or null
    uint32_t n_tris;
    const float *pos;          // 3 floats per vertex
    const uint32_t *vidx;      // 3 vertex indices per triangle
    const uint2 *ranges;       // leaf slots [x, y) below each child, 2 or 4 per node (empty: absent child)
    box6 *boxes;               // box_tree_entries(n_slots)
};

// Records, shading vertices and every node box from the new positions: three
// launches up to a million slots.
hipError_t launch_refit(const refit_args &a, hipStream_t stream);

} // namespace dev
} // namespace rt
