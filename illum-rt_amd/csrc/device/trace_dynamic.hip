// Postponing persistent trace of binary trees with the traversal stack in
// LDS: the speculative tracers' closest and any hits of one scene, and
// descriptor tables.
//
// The work and its order are trace_persistent.hip's (parked leaves, a vote
// that ends the node loop, refill from the work counters): what differs is
// how a lane's step is written.
//   * Tree and ray bound the stack (the tree's stack need), so it is an LDS
//     column with two sentinels below and no empty test.  Any-hit and table
//     launches hold all of it (at most kDynamicStackNeed entries) and need no
//     overflow test either.  Closest hits of one scene keep kSpillWords words,
//     which leaves room for 7 waves per SIMD: a push on a full column moves
//     the kSpillStep oldest entries to a global column per lane, and a lane
//     that runs into the sentinel fetches them back once per leaf phase.
//   * The two newest entries are read before the node arrives.  A miss, a
//     hit, a parked leaf and a pop are then selects between registers, where
//     the other kernel branches and waits for LDS after the box tests.
//   * All control flow outside the step is wave-uniform.  Closest hits are
//     written when the wavefront leaves to take new rays, with barycentrics
//     computed again there (each leaf phase: 2-3% slower); any-hit results
//     after each leaf phase (8.3 M random rays 5635 us, when it leaves 6496).
//     70 VGPRs (any-hit), 71 (closest) and 74 (closest, table).
//
// Bound, 8.3 M hall rays: L1 lines on incoherent rays (bounce: 1.06 line
// accesses a clock, address units 98% busy, VALU 89% at 44% of the lanes;
// trace_persistent's kernel: VALU 99% at 32%), VALU issue on camera rays (all
// of it at 64% of the lanes, before 54%).
// Measured, trace_persistent's kernel (its fastest stack configuration for
// single scenes) -> this one, us.  Closest hit, dynamic tracer, hall camera /
// bounce / random rays: 921 k 733 -> 657, 1036 -> 956, 1026 -> 950; 2.07 M
// 1118 -> 1018, 1699 -> 1628, 1782 -> 1750; 8.3 M 3103 -> 3023, 5325 -> 5329,
// 6175 -> 6166 (persistent-speculative 2935 -> 2860, 6406 -> 6283, 7089 ->
// 7060); soup 2.07 M 333 -> 305, 393 -> 353, 809 -> 784.  The whole 24 words
// in LDS: 8.3 M random 7480 (6 waves per SIMD); registers capped for 8 waves:
// bounce 5405, 921 k 1036.  Any-hit, dynamic tracer: hall 2.07 M 1160 -> 1075,
// 1885 -> 1690, 1950 -> 1658, 8.3 M 3065 -> 3000, 5770 -> 5350, 6670 -> 5635;
// soup 327 -> 302, 385 -> 339, 793 -> 739.  Descriptor tables, closest hit,
// random rays: 24 scenes x 200 k rays of 5 k triangles 2355 -> 1985
// (speculative), 1765 -> 1615 (dynamic); 8 x 500 k of 90 k 3630 -> 2970, 2575
// -> 2400; 3 x 1.1 M of 250 k 3440 -> 2860, 2545 -> 2400.
#include "kernels.h"
#include "trace_core.h"

namespace rt {
namespace dev {

namespace {

struct dynamic_args {
    scene_desc sc;
    ray_soa rays;
    hit_soa hits;
    uint8_t *occluded;
    uint32_t n;
    const uint32_t *count_ptr;
    uint32_t *counter;
    const batch_desc *table;
    uint32_t n_desc;
    ray_gather gather;
    uint32_t entries;   // LDS words per lane: two sentinels and the stack need, or as much of it as fits
    int32_t *spill;     // columns of the oldest entries, one per lane (closest hits of one scene)
    uint32_t chunks;
    int32_t refill_thr, park;
};

// Closest hits of one scene: LDS words per lane, sentinels included, and the
// entries that move between them and the global column at a time.
constexpr uint32_t kSpillWords = 20;
constexpr int kSpillStep = 4;

} // namespace

template <int TRI, bool ANY, bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ANY ? 7 : MULTI ? 6 : 7)))
void k_trace_dynamic(dynamic_args a) {
    extern __shared__ int32_t lds_words[];
    const uint32_t n = a.count_ptr ? *a.count_ptr : a.n;
    const uint32_t lane = threadIdx.x & 63u;
    int32_t *col = lds_words + (threadIdx.x >> 6) * 64u * a.entries + lane;
    col[0] = kInvalidRef;
    col[64] = kInvalidRef;
    constexpr bool SPILL = !ANY && !MULTI;
    const int top = (int)(64u * a.entries);   // sp when the LDS part is full
    int gs = 0;                               // entries moved to the global column
    uint32_t chunk = blockIdx.x % a.chunks, dry = 0;
    bool exhausted = false, alive = false, finite = true;
    const char *nodes = static_cast<const char *>(a.sc.nodes);
    const tri_rec *tris = a.sc.tris;
    const uint32_t *slot_ids = a.sc.slot_ids;
    bool alpha_on = a.sc.alpha != 0;
    uint32_t desc = 0, ray_id = 0;
    dray r{};
    int32_t cur = kInvalidRef;
    int sp = 128;           // word of the column the next entry goes to
    int32_t p0 = 0, p1 = 0, p2 = 0, p3 = 0;   // parked leaves, p0 the newest
    int pc = 0;
    const int park = ANY ? 1 : a.park;
    float ht = 0;
    uint32_t hslot = 0;
    bool found = false;
    bool exact = false;

    // ---- ended rays: write the result, the lane is idle ----
    auto end_rays = [&]() {
        if (alive && cur == kInvalidRef) {
            hit_soa ho = a.hits;
            uint8_t *occ = a.occluded;
            if (MULTI) {
                ho = a.table[desc].hits;
                occ = a.table[desc].occluded;
            }
            if (ANY) {
                if (occ) occ[ray_id] = found ? 1 : 0;
                if (ho.t)
                    store_hit(ho, ray_id, found ? 4294967295.0f : FLT_MAX, 0.0f, 0.0f, found ? 0xffffffffu : 0u);
            } else if (found) {
                // the hit's barycentrics, by the same arithmetic again: two
                // registers less to carry
                const float4 *p = reinterpret_cast<const float4 *>(tris + hslot);
                float4 r0 = p[0], r1 = p[1], r2 = p[2];
                float t = ht, u = 0.0f, v = 0.0f;
                if (TRI == TRI_EXACT) (void)tri_exact(r0, r1, r2, r, INFINITY, t, u, v);
                else (void)tri_woop(r0, r1, r2, r, INFINITY, t, u, v);
                store_hit(ho, ray_id, t, u, v, TRI == TRI_EXACT ? __float_as_uint(r0.w) : slot_ids[hslot]);
            } else {
                store_hit(ho, ray_id, FLT_MAX, 0.0f, 0.0f, 0u);
            }
            alive = false;
        }
    };

    for (;;) {
        // ---- idle lanes take new rays: one atomic per wavefront ----
        if (!exhausted) {
            const uint64_t idle = wave_mask(!alive);
            const uint32_t want = (uint32_t)__popcll(idle);
            const uint32_t lo = (uint32_t)((uint64_t)n * chunk / a.chunks);
            const uint32_t hi = (uint32_t)((uint64_t)n * (chunk + 1) / a.chunks);
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(a.counter + chunk * kCounterStride, want);
            base = __builtin_amdgcn_readfirstlane(base);
            const uint64_t first = (uint64_t)lo + base;
            if (first + want >= hi) {
                chunk = chunk + 1 == a.chunks ? 0 : chunk + 1;
                if (++dry >= a.chunks) exhausted = true;
            }
            if (!alive) {
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                const uint64_t i64 = first + rank;
                if (i64 < hi) {
                    const uint32_t idx = (uint32_t)i64;
                    ray_id = idx;
                    int32_t root = a.sc.root_ref;
                    bool nan_free = a.sc.nan_free != 0;
                    if (MULTI) {
                        desc = find_desc(a.table, a.n_desc, idx);
                        const batch_desc &bd = a.table[desc];
                        nodes = static_cast<const char *>(bd.scene.nodes);
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
                    finite = nan_free && ray_is_finite(r);
                    cur = root;
                    sp = 128;
                    gs = 0;
                    pc = 0;
                    found = false;
                    ht = ANY ? INFINITY : FLT_MAX;
                    alive = true;
                }
            }
        }
        if (wave_mask(alive) == 0) {
            if (exhausted) break;
            continue;
        }
        exact = wave_mask(alive && !finite) != 0;
        do {
            // ---- inner nodes, until every descending lane has a leaf ----
            for (;;) {
                const bool inner = (uint32_t)cur < (uint32_t)kInvalidRef;
                const bool step = inner || (cur < 0 && pc < park);
                if (wave_mask(step && pc == 0) == 0) break;
                if (step) {
                    const int32_t t0 = col[sp - 64], t1 = col[sp - 128];
                    int32_t c = cur, next = t0;   // what the lane is at after this step, and the entry below it
                    int d = 0;
                    bool both = false, any = false;
                    if (inner) {
                        const float4 *np = reinterpret_cast<const float4 *>(nodes + ((uint32_t)cur << 6));
                        const float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
                        float dl, dr;
                        bool hl, hr;
                        if (exact) {
                            hl = box_exact<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, ht, dl);
                            hr = box_exact<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, ht, dr);
                        } else {
                            hl = box_min3<ANY>(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, r, ht, dl);
                            hr = box_min3<ANY>(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, r, ht, dr);
                        }
                        const int32_t rl = __float_as_int(n3.x), rr = __float_as_int(n3.y);
                        both = hl && hr;
                        any = hl || hr;
                        const bool left = hl && (!hr || dl < dr);
                        const int32_t far_ref = left ? rr : rl;
                        if (both) {
                            if (SPILL && sp == top) {   // rare: the oldest entries go to the global column
                                int32_t *g = a.spill + blockIdx.x * 256u + threadIdx.x;
                                const size_t stride = gridDim.x * 256u;
                                for (int k = 0; k < kSpillStep; ++k) g[(gs + k) * stride] = col[64 * (2 + k)];
                                gs += kSpillStep;
                                for (int k = 128; k < top - 64 * kSpillStep; k += 64) col[k] = col[k + 64 * kSpillStep];
                                sp -= 64 * kSpillStep;
                            }
                            col[sp] = far_ref;
                        }
                        c = any ? (left ? rl : rr) : t0;
                        next = both ? far_ref : (any ? t0 : t1);
                        d = both ? 64 : (any ? 0 : -64);
                    }
                    const bool keep = c < 0 && pc < park;
                    if (!ANY) {
                        p3 = keep ? p2 : p3;
                        p2 = keep ? p1 : p2;
                        p1 = keep ? p0 : p1;
                    }
                    p0 = keep ? c : p0;
                    pc += keep ? 1 : 0;
                    cur = keep ? next : c;
                    sp += d - (keep ? 64 : 0);
                }
            }
            // ---- leaves: the parked ones, oldest first, then those in hand ----
            for (;;) {
                int32_t lf;
                if (pc > 0) {
                    lf = ANY ? p0 : (pc > 2 ? (pc > 3 ? p3 : p2) : (pc > 1 ? p1 : p0));
                    --pc;
                } else if (cur < 0) {
                    lf = cur;
                    sp -= 64;
                    cur = col[sp];
                } else {
                    break;
                }
                const uint32_t slot = leaf_slot(lf), cnt = leaf_count(lf);
                for (uint32_t k = 0; k < cnt; ++k) {
                    const float4 *p = reinterpret_cast<const float4 *>(tris + slot + k);
                    float4 r0 = p[0], r1 = p[1], r2 = p[2];
                    float t, u, v;
                    bool hit = TRI == TRI_EXACT ? tri_exact(r0, r1, r2, r, ht, t, u, v)
                                                : tri_woop(r0, r1, r2, r, ht, t, u, v);
                    if (hit && alpha_on)
                        hit = alpha_opaque(MULTI ? a.table[desc].scene : a.sc,
                                           TRI == TRI_EXACT ? __float_as_uint(r0.w) : slot_ids[slot + k], u, v);
                    if (hit) {
                        found = true;
                        hslot = slot + k;
                        if (!ANY) ht = t;
                    }
                }
                if (ANY && found) {
                    cur = kInvalidRef;
                    pc = 0;
                    break;
                }
            }
            if (SPILL && cur == kInvalidRef && gs > 0) {   // the LDS part is empty: the column's newest entries
                int32_t *g = a.spill + blockIdx.x * 256u + threadIdx.x;
                const size_t stride = gridDim.x * 256u;
                gs -= kSpillStep;
                for (int k = 0; k < kSpillStep; ++k) col[64 * (2 + k)] = g[(gs + k) * stride];
                sp = 64 * (kSpillStep + 1);
                cur = col[sp];
            }
            if (ANY) end_rays();
        } while (exhausted ? wave_mask(cur != kInvalidRef) != 0
                           : (int)__popcll(wave_mask(cur != kInvalidRef)) >= a.refill_thr);
        if (!ANY) end_rays();
        if (exhausted) break;
    }
}

namespace {

// Sentinel words below the stack: a step reads the two newest entries.
constexpr uint32_t kSentinels = 2;

// Blocks of a launch without a caller's grid: what fits the device at once,
// asked once per device and stack size.  Closest hits of a refilled table
// take 4 blocks per CU (16 wavefronts) when more fit: their 64 rays are the
// least alike, and more wavefronts evict each other's nodes (3 x 1.1 M rays
// of 250 k triangles: 6 blocks 2745 us, 5 2620, 4 2395; 24 x 200 k of 5 k
// 1580, 1560, 1615).  Any-hit keeps all: camera rays, 8.3 M, 3012 us with 6
// blocks, 3451 with 4.  (Random any-hit rays are the exception: 8.3 M of the
// hall 6428 us with 7 blocks, 6043 with 5, 2.07 M 1843 and 1774; camera rays pay
// for it, 2810 and 2920.)
//
// One scene and few rays: a grid of 7 blocks per CU is 459 k lanes, so up to a
// million rays most lanes take one or two, the rays of a wavefront are spread
// over the batch by its end, and every further block adds its start and its
// round of empty work counters.  Closest hit, dynamic tracer, 5 / 6 / 7 blocks,
// camera and bounce rays: 500 triangles, 640 k rays 116 / 123 / 133 and 130 / 146 /
// 169; 2.07 M 182 / 188 / 195 and 206 / 208 / 216; 8,192 triangles, 640 k 193 /
// 206 / 220 and 232 / 243 / 265; 2.07 M 312 / 310 / 303 and 364 / 369 / 364;
// 130,000, 800 k 353 / 366 / 373 and 386 / 415 / 429; hall, 1 M 696 / 661 / 658
// and 950 / 938 / 972, 1.3 M 802 / 766 / 750 and 1116 / 1106 / 1117.  (Without
// refill the hall's trees take them all: bounce rays, 1 M, 1039 / 1010 with 6 / 7.)
inline int few_rays_blocks(int need, uint32_t rays, bool refill) {
    if (rays <= 1u << 20) return need <= 14 ? 5 : (refill || need <= 19 ? 6 : 8);
    return rays <= 1u << 21 && need <= 12 ? 5 : 8;
}

template <int TRI, bool ANY, bool MULTI>
hipError_t grid_of(uint32_t entries, const persistent_cfg &cfg, int *blocks) {
    static int cached[64][kDynamicStackNeed + kSentinels + 1] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    int cus = 0, per_cu = cached[dev][entries];
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    if (per_cu == 0) {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_trace_dynamic<TRI, ANY, MULTI>, 256,
                                                         1024u * entries);
        if (e != hipSuccess) return e;
        if (per_cu < 1) per_cu = 1;
        cached[dev][entries] = per_cu;
    }
    if (MULTI && !ANY && cfg.refill && per_cu > 4) per_cu = 4;
    if (!MULTI) per_cu = min(per_cu, few_rays_blocks(cfg.need, cfg.rays, cfg.refill));
    *blocks = cus * per_cu;
    return hipSuccess;
}

template <int TRI, bool ANY, bool MULTI>
hipError_t launch_one(const dynamic_args &a, const persistent_cfg &cfg, hipStream_t s, int *grid_out) {
    int blocks = cfg.blocks;
    if (blocks <= 0) {
        hipError_t e = grid_of<TRI, ANY, MULTI>(a.entries, cfg, &blocks);
        if (e != hipSuccess) return e;
    }
    if (grid_out) {
        *grid_out = blocks;
        return hipSuccess;
    }
    const uint32_t column = ANY || MULTI ? 0u : dynamic_spill_entries(cfg.need);
    if (column && (!cfg.spill || cfg.spill_bytes < persistent_spill_bytes(blocks, column))) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_trace_dynamic<TRI, ANY, MULTI>), dim3(blocks), dim3(256), 1024u * a.entries, s, a);
    return hipGetLastError();
}

hipError_t dispatch(int tri, bool any, bool multi, dynamic_args &a, const persistent_cfg &cfg, hipStream_t s,
                    int *grid_out) {
    a.entries = any || multi ? (uint32_t)cfg.need + kSentinels
                             : min((uint32_t)cfg.need + kSentinels, kSpillWords);
    a.spill = cfg.spill;
    a.chunks = cfg.chunks == 8 ? 8u : 1u;
    a.refill_thr = cfg.refill ? (cfg.refill_thr < 1 ? 1 : (cfg.refill_thr > 64 ? 64 : cfg.refill_thr)) : 1;
    a.park = cfg.park < 1 || cfg.park > kParkClosest ? kParkClosest : cfg.park;
    if (!multi && !any)
        return tri == TRI_EXACT ? launch_one<TRI_EXACT, false, false>(a, cfg, s, grid_out)
                                : launch_one<TRI_WOOP, false, false>(a, cfg, s, grid_out);
    if (!multi)
        return tri == TRI_EXACT ? launch_one<TRI_EXACT, true, false>(a, cfg, s, grid_out)
                                : launch_one<TRI_WOOP, true, false>(a, cfg, s, grid_out);
    if (tri == TRI_EXACT)
        return any ? launch_one<TRI_EXACT, true, true>(a, cfg, s, grid_out)
                   : launch_one<TRI_EXACT, false, true>(a, cfg, s, grid_out);
    return any ? launch_one<TRI_WOOP, true, true>(a, cfg, s, grid_out)
               : launch_one<TRI_WOOP, false, true>(a, cfg, s, grid_out);
}

} // namespace

uint32_t dynamic_spill_entries(int need) {
    const int over = need - (int)(kSpillWords - kSentinels);
    return over > 0 ? (uint32_t)((over + kSpillStep - 1) / kSpillStep * kSpillStep) : 0u;
}

bool dynamic_fits(int bvh, bool any, bool multi, const persistent_cfg &cfg) {
    return bvh == BVH2 && cfg.speculative && !cfg.stats && cfg.need > 0 &&
           (cfg.need <= kDynamicStackNeed || !(any || multi));
}

hipError_t dynamic_grid(int tri, bool any, bool multi, const persistent_cfg &cfg, int *blocks) {
    dynamic_args a{};
    return dispatch(tri, any, multi, a, cfg, nullptr, blocks);
}

hipError_t launch_trace_dynamic(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                                uint32_t n, const uint32_t *count_ptr, uint32_t *counter, bool any,
                                const persistent_cfg &cfg, hipStream_t stream, ray_gather gather) {
    dynamic_args a{};
    a.sc = sc;
    a.rays = rays;
    a.hits = hits;
    a.occluded = occluded;
    a.n = n;
    a.count_ptr = count_ptr;
    a.counter = counter;
    a.gather = gather;
    return dispatch(sc.tri, any, false, a, cfg, stream, nullptr);
}

hipError_t launch_trace_dynamic_batch(const batch_desc *d_table, uint32_t n_desc, uint32_t total, int tri, bool any,
                                      uint32_t *counter, const persistent_cfg &cfg, hipStream_t stream) {
    dynamic_args a{};
    a.n = total;
    a.counter = counter;
    a.table = d_table;
    a.n_desc = n_desc;
    return dispatch(tri, any, true, a, cfg, stream, nullptr);
}

} // namespace dev
} // namespace rt
