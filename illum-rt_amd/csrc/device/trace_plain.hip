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
// Postponed leaves.  One ray per lane leaves lanes idle wherever their rays
// differ, so a lane that reaches a leaf parks it (up to kPark) and goes on
// descending until every lane of the wavefront holds one.  Meanwhile the box
// tests see a best t that is older than the reference's, which may open nodes
// the reference would have culled.  The hits are still the reference's, bit
// for bit:
//   * Parked leaves are tested in the order they were reached.  The first is
//     the reference's next leaf.  A leaf that was met with none parked, and
//     an entry pushed then, was decided by the reference's own best t.
//   * Every other leaf is kept with its box's entry distance q and tested only
//     if q < best when its turn comes -- the reference's test of that box (of
//     two sibling leaves the far one is held to the best t before the near
//     one, when the reference tested both).  Its ancestors' tests agree:
//     their boxes hold the leaf's box, and slab distances are monotone in the
//     bounds under IEEE rounding.
//   * The stack has no room for q.  A leaf that would be pushed while others
//     are parked makes its node wait until they are done (`hold`), so entries
//     on the stack are nodes, whose children are tested again, or leaves the
//     reference visits.
// Rays with non-finite components and trees whose boxes are not nested (an
// uploaded layout may be any) do not park; the counting variant does not
// either and counts the reference's visits.  Any-hit needs no order: it parks
// one leaf and tests it without conditions.
//
// Without parking, the wavefront leaves its node loop once at most kNodeLanes
// lanes still descend: each lane's own order is unchanged.
//
// Bound: VALU issue at partial lane occupancy, and wavefronts in flight (26
// of 32 per CU with the hall's 24 words a lane; 21 wavefronts cost 6%, which
// rules out parked leaves or distances in LDS).  More than 1 M rays come
// here; smaller batches go to the group trace.  Hall, closest hit, camera /
// bounce / random rays, 1920 x 1080: 1181 / 2069 / 2171 us, before (no
// parking) 1262 / 2253 / 2345; 3840 x 2160: 3466 / 7121 / 7464, before 3633 /
// 7902 / 8208; any-hit 1920 x 1080 1071 / 2155 / 2119, before 1198 / 2179 /
// 2225.  3 parked leaves instead of 4: 1217 / 2129 / 2192; making every far
// leaf's node wait, siblings too: 1213 / 2218 / 2249; one pushed leaf with its
// distance in registers instead of waiting: 6% slower; registers capped for 8
// waves per SIMD: 1219 / 2101 / 2243.  Without parking: 1453 waiting for every
// lane, 1283 with a vote of 4, 1256 with 16.  Blocks that hand their idle
// lanes new rays from an LDS counter (2 to 16 rays a lane) gained 6-20% on
// incoherent rays and lost 20-60% on camera rays.
#include "kernels.h"
#include "trace_core.h"

namespace rt {
namespace dev {

namespace {

// Leaves a lane may park.
template <bool ANY, bool COUNT> constexpr int kPark = COUNT ? 0 : (ANY ? 1 : 4);

} // namespace

template <int TRI, bool ANY, bool COUNT>
__global__ __launch_bounds__(64) void k_trace_plain(scene_desc sc, ray_soa rays, hit_soa hits, uint8_t *occluded,
                                                    uint32_t n, unsigned long long *stats) {
    extern __shared__ int32_t lds_stack[];   // per lane: two sentinels, the tree's stack need; lane-minor
    constexpr int P = kPark<ANY, COUNT>;
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x, 16u) * 64u + threadIdx.x;
    if (i >= n) return;
    int32_t *col = lds_stack + threadIdx.x;
    col[0] = kInvalidRef;
    col[64] = kInvalidRef;
    const dray r = load_ray(rays, i);
    // the select-based box test only where some ray of the wavefront (or the
    // scene) has a non-finite component; both decide identically otherwise
    const bool exact = !sc.nan_free || wave_mask(!ray_is_finite(r)) != 0;
    const bool park = P > 0 && (ANY || (sc.nested && !exact));
    const node2 *nodes = static_cast<const node2 *>(sc.nodes);
    int32_t cur = sc.root_ref;
    int sp = 128;             // word of the column the next entry goes to
    float cq = -INFINITY;     // distance of the leaf in hand (below)
    // parked leaves and their distances, [0] the newest
    int32_t pl[P > 0 ? P : 1] = {};
    float pq[P > 0 ? P : 1] = {};
    uint32_t pairs = 0;       // bit k: the k-th leaf of the next leaf phase is the far sibling of the one before it
    int pc = 0;
    dhit h{};
    h.t = ANY ? INFINITY : FLT_MAX;
    uint32_t c_nodes = 0, c_tris = 0;
    while (wave_mask(cur != kInvalidRef) != 0) {
        bool hold = false;    // the node in hand has to wait for the parked leaves
        // ---- inner nodes: until every lane has a leaf (parking), or at most kNodeLanes still descend ----
        for (int least = 0;;) {
            const bool inner = (uint32_t)cur < (uint32_t)kInvalidRef;
            const bool step = (inner && (ANY || !hold)) || (park && cur < 0 && pc < P);
            if ((int)__popcll(wave_mask(step && pc == 0)) <= least) break;
            if (!park) least = kNodeLanes;
            if (step) {
                const int32_t t0 = col[sp - 64], t1 = P ? col[sp - 128] : 0;
                int32_t c = cur, next = t0;   // what the lane is at after this step, and the entry below it
                float c_q = cq, next_q = -INFINITY;
                int d = 0;
                if (inner) {
                    if (COUNT) ++c_nodes;
                    const float4 *np = reinterpret_cast<const float4 *>(nodes + cur);
                    const float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
                    float dl, dr;
                    bool hl, hr;
                    if (exact) {
                        hl = box_exact<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, h.t, dl);
                        hr = box_exact<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, h.t, dr);
                    } else {
                        hl = box_min3<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, h.t, dl);
                        hr = box_min3<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, h.t, dr);
                    }
                    const int32_t rl = __float_as_int(n3.x), rr = __float_as_int(n3.y);
                    const bool both = hl && hr, any = hl || hr, left = hl && (!hr || dl < dr);
                    const int32_t near_ref = left ? rl : rr, far_ref = left ? rr : rl;
                    bool push = both;
                    if (!ANY && P > 0) {
                        hold = pc > 0 && both && far_ref < 0 && !(near_ref < 0 && pc < P);
                        push = both && !hold;
                        c_q = left ? dl : dr;
                        next_q = both && pc > 0 ? (left ? dr : dl) : -INFINITY;
                        if (both && near_ref < 0 && far_ref < 0 && pc < P) pairs |= 2u << pc;
                    }
                    if (push) col[sp] = far_ref;
                    c = any ? near_ref : t0;
                    next = both ? far_ref : (any ? t0 : t1);
                    d = both ? 64 : (any ? 0 : -64);
                    if (!ANY && P > 0) {
                        c_q = any ? c_q : -INFINITY;
                        c = hold ? cur : c;
                        d = hold ? 0 : d;
                    }
                }
                const bool keep = park && c < 0 && pc < P;
#pragma unroll
                for (int k = P - 1; k > 0; --k) {
                    pl[k] = keep ? pl[k - 1] : pl[k];
                    pq[k] = keep ? pq[k - 1] : pq[k];
                }
                if (P > 0) pl[0] = keep ? c : pl[0];
                if (P > 1) {
                    pq[0] = keep ? c_q : pq[0];
                    cq = keep ? next_q : c_q;
                }
                pc += keep ? 1 : 0;
                cur = keep ? next : c;
                sp += d - (keep ? 64 : 0);
            }
        }
        // ---- leaves: the parked ones, oldest first, then those in hand ----
        float before = h.t;   // best t before the latest leaf
        for (bool first = true;; first = false) {   // the first is visited whatever its distance
            int32_t lf;
            float lq = -INFINITY;
            if (pc > 0) {
                lf = pl[0];
                lq = P > 1 ? pq[0] : 0.0f;
#pragma unroll
                for (int k = 1; k < P; ++k) {
                    lf = pc > k ? pl[k] : lf;
                    lq = pc > k ? pq[k] : lq;
                }
                --pc;
            } else if (cur < 0) {
                lf = cur;
                if (P > 1) lq = cq;
                cq = -INFINITY;
                sp -= 64;
                cur = col[sp];
            } else {
                break;
            }
            const uint32_t slot = leaf_slot(lf);
            const uint32_t cnt = !ANY && P > 1 && !first && !(lq < (pairs & 1u ? before : h.t)) ? 0u : leaf_count(lf);
            before = h.t;
            pairs >>= 1;
            for (uint32_t k = 0; k < cnt; ++k) {
                float t, u, v;
                if (COUNT) ++c_tris;
                if (test_slot<TRI>(sc, slot + k, r, h.t, t, u, v) &&
                    (!sc.alpha || alpha_opaque(sc, slot_tri_id<TRI>(sc, slot + k), u, v))) {
                    h.found = true;
                    h.slot = slot + k;
                    if (ANY) {
                        cur = kInvalidRef;
                        pc = 0;
                        break;
                    }
                    h.t = t;
                    h.u = u;
                    h.v = v;
                }
            }
            if (ANY && h.found) break;
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
    const size_t lds = 256u * (depth + 2u);
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
