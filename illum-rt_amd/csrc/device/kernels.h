// Host-callable launchers of the gfx950 kernels (implemented in the .hip
// files of this directory).  All launches are asynchronous on `stream`.
#pragma once

#include <hip/hip_runtime.h>

#include "../core/layout.h"

#include <cstdint>

namespace rt {
namespace dev {

// The plain kernels hold their stack in LDS (256 bytes a block and entry);
// the host refuses BVHs that need kPlainStackCap or more entries for them.
constexpr int kPlainStackCap = 64;

// Persistent kernels, stack configuration 0: per-lane stack of kRegStack
// entries in VGPRs backed by a ring of kLdsStack entries per lane in LDS and,
// for deeper traversals, a per-lane column of a global spill buffer.
constexpr int kRegStack = 4;
constexpr int kLdsStack = 28;
constexpr int kPersistentWavesPerBlock = 4;
constexpr int kStackConfigs = 5;
// Leaves a closest-hit lane of the speculative persistent tracers parks
// before it stops descending: registers for at most 4; persistent_cfg::park
// picks 1..4 at run time (default 4).
constexpr int kParkClosest = 4;
// Work counters of the persistent kernels: one per chunk, each in its own
// 256-byte line; kCounterBytes of device memory hold all of them.
constexpr uint32_t kMaxChunks = 8;
constexpr uint32_t kCounterStride = 64;
constexpr size_t kCounterBytes = kMaxChunks * kCounterStride * 4;

// Stack entries the persistent kernels hold in VGPRs and LDS for a BVH of
// the given format and stack configuration (0: 4 VGPR + 28 LDS entries,
// 1: 8 + 16, 2: 2 + 20, 3: 0 + 24, 4: 0 + 20 with registers capped for 8
// waves per SIMD on single-scene binary trees).
int persistent_stack_cap(int bvh, int stack = 0);

// Spill entries per lane a persistent launch needs for a tree whose
// traversal can hold `need` stack entries (0 when VGPRs and LDS hold them),
// and the bytes of spill buffer a grid of `blocks` needs for that many.
uint32_t persistent_spill_entries(int bvh, int stack, int need);
size_t persistent_spill_bytes(int blocks, uint32_t entries);

// One entry of a multi-scene batch: a scene and its own ray and hit buffers;
// its rays occupy [first, first + n) of the launch's index space.
struct batch_desc {
    scene_desc scene;
    ray_soa rays;
    hit_soa hits;
    uint8_t *occluded;
    uint32_t first, n;
};

// `need`: the tree's stack need, below kPlainStackCap.  With `stats` non-null
// the counting variant runs and adds the number of inner nodes fetched to stats[0] and of triangle records tested to stats[1].
hipError_t launch_trace_plain(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                              uint32_t n, bool any, int need, hipStream_t stream,
                              unsigned long long *stats = nullptr);

// Rays of a single-scene persistent launch read from records of `stride`
// float4 (at least two) that begin (ox, oy, oz, tmin | dx, dy, dz, tmax)
// instead of planes: ray idx is record perm[idx] (record idx when perm is
// null); hits are still written at idx.  With fixed_t set every ray spans
// [kRayEps, FLT_MAX] and the records' tmin/tmax words are not read.
struct ray_gather {
    const float4 *aos = nullptr;
    const uint32_t *perm = nullptr;
    uint32_t stride = 2;
    uint32_t fixed_t = 0;
};

// Tunables of the persistent kernel.
struct persistent_cfg {
    int speculative;      // leaf postponement
    int refill;           // fetch new rays when active lanes drop below refill_thr
    int refill_thr;       // active-lane threshold for refill (out of 64)
    int blocks;           // grid size; 0 = occupancy-derived default
    unsigned long long *stats = nullptr;   // non-null: counting variant (inner nodes, triangle tests)
    int stack = 0;        // stack configuration 0..kStackConfigs-1, see persistent_stack_cap
    int chunks = 8;       // 1: one work counter; 8: one contiguous chunk of rays per XCD
    int park = kParkClosest;   // parked leaves per closest-hit lane of the speculative tracers (1..4)
    // Global spill buffer: spill_cap entries per lane of the grid
    // (persistent_spill_bytes); spill_cap 0 when the tree fits VGPRs + LDS.
    int32_t *spill = nullptr;
    uint32_t spill_cap = 0;
    size_t spill_bytes = 0;
    int need = 0;         // the trees' stack need; 0: trace_persistent.hip's kernels (see dynamic_fits)
    uint32_t rays = 0xffffffffu;   // rays of the launch, or as many as it can have (sizes the grid of one scene)
};

// `counter` points to kCounterBytes of device memory (cleared by the launch);
// `n` is the number of rays, read from device memory when count_ptr is
// non-null (so a captured graph can trace a batch whose size an earlier
// kernel produced).  The launch fails with hipErrorInvalidValue when
// cfg.spill_cap is set and the spill buffer is smaller than the grid needs.
hipError_t launch_trace_persistent(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits,
                                   uint8_t *occluded, uint32_t n, const uint32_t *count_ptr, uint32_t *counter,
                                   bool any, const persistent_cfg &cfg, hipStream_t stream,
                                   ray_gather gather = ray_gather{});

// The postponing tracers of binary trees, with the stack in LDS
// (trace_dynamic.hip).  Does a launch of this kind take it?  cfg.need set to
// 0 (the caller bounds the spill column, or must not depend on one), launches
// that count fetches, and any-hit and table launches over trees of more than
// kDynamicStackNeed entries keep the kernels of trace_persistent.hip, which
// call these.  dynamic_spill_entries: cfg.spill_cap of a closest-hit launch of
// one scene (0 when the stack fits); the others need no column.
constexpr int kDynamicStackNeed = 32;
// Nodes whose byte offsets fit the kernel's 32-bit offset register (a 64-bit
// address per lane costs two registers); the caller sets cfg.need to 0 for
// larger trees, which only an upload whose leaves share slots can have.
constexpr uint32_t kDynamicNodes = 1u << 26;
bool dynamic_fits(int bvh, bool any, bool multi, const persistent_cfg &cfg);
uint32_t dynamic_spill_entries(int need);
hipError_t dynamic_grid(int tri, bool any, bool multi, const persistent_cfg &cfg, int *blocks);
hipError_t launch_trace_dynamic(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                                uint32_t n, const uint32_t *count_ptr, uint32_t *counter, bool any,
                                const persistent_cfg &cfg, hipStream_t stream, ray_gather gather);
hipError_t launch_trace_dynamic_batch(const batch_desc *d_table, uint32_t n_desc, uint32_t total, int tri, bool any,
                                      uint32_t *counter, const persistent_cfg &cfg, hipStream_t stream);

// One persistent launch over a descriptor table (device memory, sorted by
// `first`, first entry at 0, `total` rays in all).  All scenes must share the
// triangle and BVH formats.
hipError_t launch_trace_batch(const batch_desc *d_table, uint32_t n_desc, uint32_t total, int tri, int bvh, bool any,
                              uint32_t *counter, const persistent_cfg &cfg, hipStream_t stream);

// Grid size (blocks) of the persistent kernel instantiation for these
// settings (`multi`: the descriptor-table variant; only the scene's
// triangle and BVH formats are read): cfg.blocks when positive, else blocks
// resident per CU times the CU count.
hipError_t persistent_grid(const scene_desc &sc, bool any, const persistent_cfg &cfg, int *blocks,
                           bool multi = false);

// Group trace (trace_group.hip): `lanes` lanes per ray, for batches too small
// to fill the chip with one ray per lane.  group_lanes: 16 up to kGroupRays16
// rays, 8 up to kGroupRays8 (kGroupRays8Spec for the closest hits of the
// postponing tracers), else 0, and 0 for 4-wide or very deep trees: the plain
// and persistent kernels serve those.  Callers pass the tree's own limit
// (hiprt_detail::group_rays_of) where that is lower.  Hall, us, camera / bounce
// rays:
//   16 -> 8: 320 x 240 (77k) 124 / 131 against 129 / 139, but 53 / 41 against
//   43 / 44 in the 8,192-triangle scene.
//   8 -> 0: 960 x 540 (518k) 504 / 547, plain 576 / 789; 1280 x 720 (922k)
//   839 / 913, plain 740 / 1128, dynamic 657 / 956 (any hit 748 / 793, plain
//   695 / 1201); 1920 x 1080 (2.07M) 1734 / 1912, plain
//   1181 / 2069, dynamic 1018 / 1628.
// A path tracer's later levels hold ever fewer of its slots: kGroupSlots8.
// Whole frames against the persistent kernel: 1280 x 720 (922k) 4.19 and 4.83
// ms, 320 x 240 x 16 samples (1.23M) 5.41 and 5.82.
// Up to kAppendSlots of them the group trace takes the later levels' records in
// the order they were appended: a group's lanes share one ray, so sorting
// buys less than its six launches a level.  Whole frames of 5 levels, us,
// sorted / not: hall 480 x 270 1045 / 906, 640 x 480 1770 / 1665, 1120 x 630
// (706k) 3340 / 3285, 1280 x 720 (922k) 4170 / 4180, 480 x 270 x 8 samples
// (1.04M) 4555 / 4610; a hall of 74,068 650 / 506, 1070 / 931, 2010 /
// 1878, 2525 / 2395, 2890 / 2660; 2 slots per pixel for 8 samples of 480 x 270
// 7030 / 6060 and 4995 / 3460.
constexpr uint32_t kAppendSlots = 7u << 17;
constexpr int kGroupStackNeed = 64;
constexpr uint32_t kGroupRays16 = 1u << 16;
constexpr uint32_t kGroupRays8 = 1u << 20;
constexpr uint32_t kGroupRays8Spec = 5u << 17;
constexpr uint32_t kGroupSlots8 = 5u << 18;
int group_lanes(int bvh, int need, uint32_t n, uint32_t rays8);
// The hits (or occlusion) of n rays (of *count_ptr, when given, at most n) of
// a binary tree with stack need `need` <= kGroupStackNeed; no device memory
// besides the arguments.  Rays, hits and gather as launch_trace_persistent;
// the results are the plain kernel's, bit for bit.
hipError_t launch_trace_group(const scene_desc &sc, const ray_soa &rays, const hit_soa &hits, uint8_t *occluded,
                              uint32_t n, const uint32_t *count_ptr, bool any, int lanes, int need, hipStream_t s,
                              ray_gather gather = ray_gather{});
// The same over a descriptor table, as launch_trace_batch.
hipError_t launch_trace_group_batch(const batch_desc *d_table, uint32_t n_desc, uint32_t total, int tri, bool any,
                                    int lanes, int need, hipStream_t s);

// Fills `n` uint32 words with `value` (used instead of hipMemsetAsync so the
// clearing can be captured into graphs).
hipError_t launch_fill_u32(uint32_t *p, uint32_t value, uint32_t n, hipStream_t stream);

} // namespace dev
} // namespace rt
