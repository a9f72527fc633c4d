// Plain while-while trace kernels: one ray per lane, one wavefront per block,
// grid sized to the batch, the stack in LDS, sized for the tree.  This is the
// per-bounce launch form the batched persistent kernels are measured against,
// and the exact-order kernel the parity tests hold to the CPU tracer bit for
// bit.
//
// Traversal order follows binary_bvh_tracer::closest_hit/any_hit
// (rt/cpu/bvh2.cpp:72-189): at an inner node both child boxes are tested; if
// both are hit the nearer is entered next (left when dist_l < dist_r, else
// right) and the other pushed; leaf slots are tested in index order and a hit
// replaces the best one only when strictly closer.
//
// Bound: VALU issue at partial lane occupancy (2.07 M rays and more; smaller
// batches go to the group trace).  The wavefront leaves its node loop once at
// most kNodeLanes lanes still descend, so that 60 lanes with a leaf in hand
// do not wait for the last four: each lane's own order is unchanged.  Hall,
// 1920 x 1080, closest hit, camera / bounce / random rays: 1250 / 2262 / 2412
// us with 8 lanes, 1453 / 2945 / 2828 waiting for all, 1283 / 2298 / 2396
// with 4, 1256 / 2390 / 2571 with 16; 1594 / 3323 / 3160 with the stack in
// private memory, four-wavefront blocks and no vote.  Blocks that hand their
// idle lanes new rays from an LDS counter (2 to 16 rays a lane) gained 6-20%
// on incoherent rays and lost 20-60% on camera rays.
#include "kernels.h"
#include "trace_core.h"

namespace rt {
namespace dev {

template <int TRI, bool ANY, bool COUNT>
__global__ __launch_bounds__(64) void k_trace_plain(scene_desc sc, ray_soa rays, hit_soa hits, uint8_t *occluded,
                                                    uint32_t n, unsigned long long *stats) {
    extern __shared__ int32_t lds_stack[];   // the tree's stack need entries per lane, lane-minor
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x, 16u) * 64u + threadIdx.x;
    if (i >= n) return;
    int32_t *col = lds_stack + threadIdx.x;
    const dray r = load_ray(rays, i);
    // the select-based box test only where some ray of the wavefront (or the
    // scene) has a non-finite component; both decide identically otherwise
    const bool exact = !sc.nan_free || __ballot(!ray_is_finite(r)) != 0;
    const node2 *nodes = static_cast<const node2 *>(sc.nodes);
    int32_t cur = sc.root_ref;
    int sp = 0;
    dhit h{};
    h.t = ANY ? INFINITY : FLT_MAX;
    uint32_t c_nodes = 0, c_tris = 0;
    while (cur != kInvalidRef) {
        while (cur >= 0 && cur != kInvalidRef) {
            if (COUNT) ++c_nodes;
            const float4 *np = reinterpret_cast<const float4 *>(nodes + cur);
            float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
            float dl, dr;
            bool hl = box_test<ANY>(exact, n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, h.t, dl);
            bool hr = box_test<ANY>(exact, n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, h.t, dr);
            int32_t rl = __float_as_int(n3.x), rr = __float_as_int(n3.y);
            if (hl && hr) {
                bool left_first = dl < dr;
                col[64 * sp++] = left_first ? rr : rl;
                cur = left_first ? rl : rr;
            } else if (hl) {
                cur = rl;
            } else if (hr) {
                cur = rr;
            } else {
                cur = sp > 0 ? col[64 * --sp] : kInvalidRef;
            }
            if (__popcll(__builtin_amdgcn_ballot_w64(cur >= 0 && cur != kInvalidRef)) <= kNodeLanes) break;
        }
        while (cur < 0) {
            const uint32_t slot = leaf_slot(cur), cnt = leaf_count(cur);
            cur = sp > 0 ? col[64 * --sp] : kInvalidRef;
            for (uint32_t k = 0; k < cnt; ++k) {
                float t, u, v;
                if (COUNT) ++c_tris;
                if (test_slot<TRI>(sc, slot + k, r, h.t, t, u, v) &&
                    (!sc.alpha || alpha_opaque(sc, slot_tri_id<TRI>(sc, slot + k), u, v))) {
                    h.found = true;
                    h.slot = slot + k;
                    if (ANY) {
                        cur = kInvalidRef;
                        break;
                    }
                    h.t = t;
                    h.u = u;
                    h.v = v;
                }
            }
        }
    }
    if (COUNT) {
        atomicAdd(stats, (unsigned long long)c_nodes);
        atomicAdd(stats + 1, (unsigned long long)c_tris);
    }
    if (ANY) {
        if (occluded) occluded[i] = h.found ? 1 : 0;
        // The reference's CPU adapter marks an occluded ray with
        // t = ref = (unsigned)-1 and resets the others (rt/cpu/wavefront.cpp:60-70).
        if (hits.t) store_hit(hits, i, h.found ? 4294967295.0f : FLT_MAX, 0.0f, 0.0f, h.found ? 0xffffffffu : 0u);
    } else if (h.found) {
        store_hit(hits, i, h.t, h.u, h.v, slot_tri_id<TRI>(sc, h.slot));
    } else {
        store_hit(hits, i, FLT_MAX, 0.0f, 0.0f, 0u);
    }
}

namespace {
template <int TRI, bool ANY>
void launch_tri_any(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded, uint32_t n,
                    uint32_t depth, unsigned long long *stats, hipStream_t stream) {
    dim3 grid((n + 63u) / 64u), block(64);
    const size_t lds = 256u * depth;
    if (stats) hipLaunchKernelGGL((k_trace_plain<TRI, ANY, true>), grid, block, lds, stream, sc, rays, hits, occluded, n, stats);
    else hipLaunchKernelGGL((k_trace_plain<TRI, ANY, false>), grid, block, lds, stream, sc, rays, hits, occluded, n, stats);
}
} // namespace

hipError_t launch_trace_plain(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                              uint32_t n, bool any, int need, hipStream_t stream, unsigned long long *stats) {
    if (n == 0) return hipSuccess;
    const uint32_t depth = (uint32_t)(need > 1 ? need : 1);   // LDS entries per lane
    if (sc.tri == TRI_EXACT) {
        if (any) launch_tri_any<TRI_EXACT, true>(sc, rays, hits, occluded, n, depth, stats, stream);
        else launch_tri_any<TRI_EXACT, false>(sc, rays, hits, occluded, n, depth, stats, stream);
    } else {
        if (any) launch_tri_any<TRI_WOOP, true>(sc, rays, hits, occluded, n, depth, stats, stream);
        else launch_tri_any<TRI_WOOP, false>(sc, rays, hits, occluded, n, depth, stats, stream);
    }
    return hipGetLastError();
}

} // namespace dev
} // namespace rt
