// Group trace kernels: K lanes of a wavefront (8 or 16) trace one ray.
//
// A small batch is bound by the latency of its slowest wavefront.  One ray
// per lane makes a wavefront walk the union of 64 rays' node and leaf visits
// one after another: 3,072 camera rays of the 262,144-triangle hall took
// 670 us (plain) or 430 us (dynamic) while a single ray takes 34 us, and a
// 320 x 240 image took no less.  Here a group of K lanes takes the K newest
// entries of its ray's stack in one step -- each lane fetches one inner node
// and tests both child boxes -- so a ray of 100 node visits is done in 20 to
// 30 steps, and only 64 / K rays share a wavefront.
//
//   * The stack is a list of (reference, distance) in LDS, kept in the
//     reference's depth-first order: a step replaces the K newest entries by
//     their hit children, nearer child above, in the entries' own order
//     (positions from two ballots and population counts).  The node at depth
//     j of the K is opened before the ones above it are finished, so it is
//     tested against an older best t than the reference would use: the list
//     holds every entry the reference pushes, and some it would have culled.
//   * Leaves wait until they are on top.  Then K / 4 of them are tested at
//     once, four triangles each (a larger leaf: K triangles at a time), and
//     the group keeps the smallest t, the earliest in stack order on a tie.
//   * The result is the reference's, bit for bit.  An entry carries the
//     largest entry distance D of its node and all ancestors.  The reference
//     visits a leaf for certain when D < best at that point, since best was
//     never smaller before; a leaf with D >= best, which it may have culled,
//     changes nothing unless one of its triangles is hit closer than best
//     (t < D: rounding, or a ray in a box face).  If that happens the ray
//     starts over one entry at a time, which is the reference's traversal.
//     Any-hit needs neither order nor distances.
//   * Steps take all K entries while the list holds fewer than `soft`; above
//     that they shrink, down to one, so `soft` + the tree's stack need
//     entries always suffice.
//
// Bound: VALU issue once the chip is full (about 105 VALU instructions a
// node step, 110 a leaf step; of 8 lanes 5.0 hold an inner node on camera
// rays and 4.0 on bounce rays; 29 and 33 node steps, 11 and 15 leaf steps per
// wavefront of 8 rays), the latency of the dependent node fetches below that.
// Measured, closest hit, hall, one ray per lane (plain kernel before its vote
// and LDS stack) against this one: 64 x 48 camera rays 670 -> 38 us (K = 16),
// 320 x 240 743 -> 124 us, 640 x 480 813 -> 352 us, 1281 x 719 1108 -> 832 us
// (K = 8); bounce rays 581 -> 35, 787 -> 131, 1034 -> 381, 1801 -> 910 us.  K = 4 was slower than
// 8 at the sizes this kernel serves (640 x 480: 554 against 468 us), fetching
// the nodes before the leaf step the same within 2% at fewer waves, refilling
// idle groups from a work counter slower (1280 x 720: 1290 against 1069 us: a
// group's ray is too short to pay for the fetch).
#include "kernels.h"
#include "trace_core.h"

namespace rt {
namespace dev {

namespace {

// One stack entry: a child reference and the largest entry distance of it
// and its ancestors.
struct alignas(8) group_entry {
    int32_t ref;
    float dist;
};

struct group_args {
    scene_desc sc;
    ray_soa rays;
    hit_soa hits;
    uint8_t *occluded;
    uint32_t n;
    const uint32_t *count_ptr;
    const batch_desc *table;
    uint32_t n_desc;
    ray_gather gather;
    uint32_t cap, soft;   // entries per ray; list length up to which steps take K entries
};

// This group's bits of a wave mask.
template <int K> __device__ __forceinline__ uint32_t group_bits(uint64_t mask, uint32_t shift) {
    return (uint32_t)(mask >> shift) & ((1u << K) - 1u);
}

template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

} // namespace

template <int K, int TRI, bool ANY, bool MULTI>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MULTI ? 7 : 8)))
void k_trace_group(group_args a) {
    extern __shared__ group_entry lds_entries[];
    const uint32_t n = a.count_ptr ? min(*a.count_ptr, a.n) : a.n;
    const uint32_t lane = threadIdx.x, gl = lane & (K - 1), shift = lane & ~(uint32_t)(K - 1);
    constexpr uint32_t kRays = 64u / K;   // rays per block
    const uint32_t low = (1u << gl) - 1u;
    group_entry *st = lds_entries + (threadIdx.x / K) * a.cap;

    const uint32_t nb = (n + kRays - 1) / kRays;
    if (blockIdx.x >= nb) return;
    const uint32_t idx = xcd_block(blockIdx.x, nb, 16u) * kRays + threadIdx.x / K;
    const bool has = idx < n;

    uint32_t ray_id = 0, desc = 0;
    dray r{};
    const node2 *nodes = static_cast<const node2 *>(a.sc.nodes);
    const tri_rec *tris = a.sc.tris;
    const uint32_t *slot_ids = a.sc.slot_ids;
    int32_t root = a.sc.root_ref;
    bool nan_free = a.sc.nan_free != 0, alpha_on = a.sc.alpha != 0;
    if (has) {
        ray_id = idx;
        if (MULTI) {
            desc = find_desc(a.table, a.n_desc, idx);
            const batch_desc &bd = a.table[desc];
            nodes = static_cast<const node2 *>(bd.scene.nodes);
            tris = bd.scene.tris;
            slot_ids = bd.scene.slot_ids;
            root = bd.scene.root_ref;
            nan_free = bd.scene.nan_free != 0;
            alpha_on = bd.scene.alpha != 0;
            ray_id = idx - bd.first;
            r = load_ray(bd.rays, ray_id);
        } else if (a.gather.aos) {
            r = load_ray_aos(a.gather.aos, a.gather.perm ? a.gather.perm[idx] : idx, a.gather.stride,
                             a.gather.fixed_t != 0);
        } else {
            r = load_ray(a.rays, idx);
        }
    }
    const bool exact = wave_mask(has && !(nan_free && ray_is_finite(r))) != 0;
    int sp = has && root != kInvalidRef ? 1 : 0;
    if (sp && gl == 0) st[0] = group_entry{root, -INFINITY};
    float best = ANY ? INFINITY : FLT_MAX, hu = 0.0f, hv = 0.0f;
    uint32_t hslot = 0;
    bool owner = false;    // this lane holds the ray's hit so far
    bool found = false;    // group-uniform
    bool serial = false;   // group-uniform: reference order, one entry at a time

    while (wave_mask(sp > 0)) {
        // LDS entries pass between the lanes of one wavefront, whose LDS
        // operations execute in order: only the compiler must keep it
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int m = serial ? min(sp, 1) : min(sp, min(K, max(1, (int)a.soft - sp)));
        const int base = sp - m;
        const bool valid = (int)gl < m;
        group_entry e{kInvalidRef, 0.0f};
        if (valid) e = st[base + (int)gl];
        const bool inner = valid && e.ref >= 0;
        const uint64_t leaf_lanes = wave_mask(e.ref < 0);
        const uint32_t leaves = group_bits<K>(leaf_lanes, shift);
        const bool top_leaf = m > 0 && ((leaves >> (m - 1)) & 1u);
        const uint64_t tops = wave_mask(top_leaf);
        int taken = 0;     // leaf entries this step takes off the top
        bool restart = false;
        if (tops) {
            // lane 4 q + j tests triangle j of the q-th leaf of the run of
            // leaves at the top
            const int lead = top_leaf ? __clz((int)~(leaves << (32 - m))) : 0;
            int q = (int)(gl >> 2);
            uint32_t j = gl & 3u;
            bool mine = q < lead;
            group_entry le{-1, 0.0f};
            if (mine) le = st[sp - 1 - q];
            uint32_t cnt = mine ? leaf_count(le.ref) : 0u;
            bool wide = false;
            taken = min(lead, K / 4);
            const uint64_t bigs = wave_mask(cnt > 4);
            if (bigs) {
                // a leaf of more than four triangles: all K lanes take it
                // once it is at the top, K triangles at a time
                const uint32_t big = group_bits<K>(bigs, shift);
                if (big) {
                    const int fq = (__ffs((int)big) - 1) >> 2;
                    if (fq == 0) {
                        wide = true;
                        j = gl;
                        le = st[sp - 1];
                        cnt = leaf_count(le.ref);
                        mine = true;
                        taken = 1;
                        if (cnt > (uint32_t)K) {
                            taken = 0;
                            if ((int)gl == m - 1) e.ref = make_leaf_ref(leaf_slot(e.ref) + K, cnt - K);
                        }
                    } else {
                        taken = fq;
                        if (q >= fq) cnt = 0;
                    }
                }
            }
            float t = INFINITY, u = 0.0f, v = 0.0f;
            const uint32_t slot = leaf_slot(le.ref) + j;
            bool hit = false;
            if (j < cnt) {
                const float4 *p = reinterpret_cast<const float4 *>(tris + slot);
                float4 r0 = p[0], r1 = p[1], r2 = p[2];
                hit = TRI == TRI_EXACT ? tri_exact(r0, r1, r2, r, best, t, u, v) : tri_woop(r0, r1, r2, r, best, t, u, v);
                if (hit && alpha_on)
                    hit = alpha_opaque(MULTI ? a.table[desc].scene : a.sc,
                                       TRI == TRI_EXACT ? __float_as_uint(r0.w) : slot_ids[slot], u, v);
            }
            const uint64_t hit_lanes = wave_mask(hit);
            if (hit_lanes) {
                const uint32_t hits = group_bits<K>(hit_lanes, shift);
                if (ANY) {
                    if (hits) {
                        found = true;
                        restart = true;
                        sp = 0;
                    }
                } else {
                    const float tm = hit ? t : INFINITY;
                    // running best before this lane's leaf, in stack order
                    float before = best;
                    float all = min_of(tm, dpp<0xB1>(tm));      // quad_perm 1 0 3 2
                    all = min_of(all, dpp<0x4E>(all));          // quad_perm 2 3 0 1
                    if (K > 4) {
                        const float o = dpp<0x141>(all);        // row_half_mirror
                        if (!wide && (gl & 4u)) before = min_of(before, o);
                        all = min_of(all, o);
                    }
                    if (K > 8) {
                        const float o = dpp<0x140>(all);        // row_mirror
                        if (!wide && (gl & 8u)) before = min_of(before, o);
                        all = min_of(all, o);
                    }
                    const uint32_t lates = group_bits<K>(wave_mask(hit && t < before && le.dist >= before), shift);
                    const uint32_t won = group_bits<K>(wave_mask(hit && t == all), shift);
                    if (hits) {
                        if (lates && !serial) {
                            // a leaf the reference may have culled gave a hit: start over in its order
                            serial = true;
                            restart = true;
                            sp = 1;
                            best = FLT_MAX;
                            owner = false;
                            found = false;
                        } else {
                            best = all;
                            found = true;
                            owner = (won & low) == 0 && hit && t == all;
                            if (owner) {
                                hu = u;
                                hv = v;
                                hslot = slot;
                            }
                        }
                    }
                }
            }
        }
        // ---- inner entries ----
        int32_t rn = e.ref, rf = kInvalidRef;
        float dn = e.dist, df = 0.0f;
        bool one = valid && !inner && (int)gl < m - taken, two = false;
        if (inner) {
            float dl, dr;
            bool hl, hr;
            const float4 *np = reinterpret_cast<const float4 *>(nodes + (uint32_t)e.ref);
            const float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
            if (exact) {
                hl = box_exact<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, best, dl);
                hr = box_exact<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, best, dr);
            } else {
                hl = box_min3<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, best, dl);
                hr = box_min3<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, best, dr);
            }
            const int32_t rl = __float_as_int(n3.x), rr = __float_as_int(n3.y);
            const bool left = hl && (!hr || dl < dr);
            rn = left ? rl : rr;
            rf = left ? rr : rl;
            if (!ANY) {
                dn = max_of(left ? dl : dr, e.dist);
                df = max_of(left ? dr : dl, e.dist);
            }
            one = hl || hr;
            two = hl && hr;
        }
        if (restart) one = two = false;
        const uint32_t b1 = group_bits<K>(wave_mask(one), shift), b2 = group_bits<K>(wave_mask(two), shift);
        int pos = base + __popc(b1 & low) + __popc(b2 & low);
        if (two) st[pos++] = group_entry{rf, df};
        if (one) st[pos] = group_entry{rn, dn};
        if (restart) {
            if (!ANY && gl == 0) st[0] = group_entry{root, -INFINITY};
        } else {
            sp = base + __popc(b1) + __popc(b2);
        }
    }

    if (!has) return;
    hit_soa ho = a.hits;
    uint8_t *occ = a.occluded;
    if (MULTI) {
        ho = a.table[desc].hits;
        occ = a.table[desc].occluded;
    }
    if (ANY) {
        if (gl == 0) {
            if (occ) occ[ray_id] = found ? 1 : 0;
            if (ho.t) store_hit(ho, ray_id, found ? 4294967295.0f : FLT_MAX, 0.0f, 0.0f, found ? 0xffffffffu : 0u);
        }
    } else if (owner) {
        const uint32_t id = TRI == TRI_EXACT ? __float_as_uint(reinterpret_cast<const float4 *>(tris + hslot)[0].w)
                                             : slot_ids[hslot];
        store_hit(ho, ray_id, best, hu, hv, id);
    } else if (!found && gl == 0) {
        store_hit(ho, ray_id, FLT_MAX, 0.0f, 0.0f, 0u);
    }
}

namespace {

template <int K, int TRI, bool ANY, bool MULTI>
hipError_t launch_k(const group_args &a, hipStream_t s) {
    constexpr uint32_t kRays = 64u / K;
    const uint32_t blocks = (a.n + kRays - 1) / kRays;
    const size_t lds = kRays * a.cap * sizeof(group_entry);
    hipLaunchKernelGGL((k_trace_group<K, TRI, ANY, MULTI>), dim3(blocks), dim3(64), lds, s, a);
    return hipGetLastError();
}

template <int K, bool MULTI>
hipError_t dispatch(int tri, bool any, const group_args &a, hipStream_t s) {
    if (tri == TRI_EXACT)
        return any ? launch_k<K, TRI_EXACT, true, MULTI>(a, s) : launch_k<K, TRI_EXACT, false, MULTI>(a, s);
    return any ? launch_k<K, TRI_WOOP, true, MULTI>(a, s) : launch_k<K, TRI_WOOP, false, MULTI>(a, s);
}

template <bool MULTI>
hipError_t dispatch_lanes(int lanes, int tri, bool any, int need, group_args &a, hipStream_t s) {
    // one wavefront a block, so that its LDS is free when its slowest ray
    // ends; 8 lanes and the hall's stack need of 22: 72 entries a ray, 4.6 KB
    a.soft = lanes == 8 ? 40u : 64u;
    a.cap = a.soft + (uint32_t)need + 2u;
    // groups whose lists are equally long read different LDS banks
    a.cap += (8u - a.cap) & 15u;
    if (lanes == 8) return dispatch<8, MULTI>(tri, any, a, s);
    return dispatch<16, MULTI>(tri, any, a, s);
}

} // namespace

int group_lanes(int bvh, int need, uint32_t n, uint32_t rays8) {
    if (bvh != BVH2 || need > kGroupStackNeed) return 0;
    return n <= kGroupRays16 ? 16 : (n <= rays8 ? 8 : 0);
}

hipError_t launch_trace_group(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                              uint32_t n, const uint32_t *count_ptr, bool any, int lanes, int need, hipStream_t s,
                              ray_gather gather) {
    if (n == 0) return hipSuccess;
    group_args a{sc, rays, hits, occluded, n, count_ptr, nullptr, 0, gather, 0, 0};
    return dispatch_lanes<false>(lanes, sc.tri, any, need, a, s);
}

hipError_t launch_trace_group_batch(const batch_desc *d_table, uint32_t n_desc, uint32_t total, int tri, bool any,
                                    int lanes, int need, hipStream_t s) {
    if (total == 0) return hipSuccess;
    group_args a{};
    a.n = total;
    a.table = d_table;
    a.n_desc = n_desc;
    return dispatch_lanes<true>(lanes, tri, any, need, a, s);
}

} // namespace dev
} // namespace rt
