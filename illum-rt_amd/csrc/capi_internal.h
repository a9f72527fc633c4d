// Internal state behind the C ABI's opaque handles, shared by the .hip files
// that implement include/illum_hiprt.h.
#pragma once

#include "../../include/illum_hiprt.h"

#include "core/layout.h"
#include "device/kernels.h"
#include "host/bvh.h"
#include "host/flatten.h"
#include "host/scene.h"

#include <hip/hip_runtime.h>

#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

namespace hiprt_detail {

// Records `msg` as the calling thread's last error and returns `code`.
int fail(int code, const std::string &msg);
inline int ok() { return HIPRT_OK; }

#define HIP_TRY(call)                                                                                          \
    do {                                                                                                       \
        hipError_t e_ = (call);                                                                                \
        if (e_ != hipSuccess)                                                                                  \
            return ::hiprt_detail::fail(HIPRT_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_));     \
    } while (0)

// Owned device allocation, or a view of a part of another one.
struct dbuf {
    void *p = nullptr;
    size_t bytes = 0;
    bool owned = true;
    dbuf() = default;
    dbuf(const dbuf &) = delete;
    dbuf &operator=(const dbuf &) = delete;
    ~dbuf() { release(); }
    void release() {
        if (p && owned) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
        owned = true;
    }
    // The `n` bytes at `at` of an allocation that outlives this buffer.
    void view(void *at, size_t n) {
        release();
        p = at;
        bytes = n;
        owned = false;
    }
    hipError_t alloc(size_t n) {
        release();
        bytes = n;
        return n ? hipMalloc(&p, n) : hipSuccess;
    }
    hipError_t upload(const void *src, size_t n) {
        hipError_t e = alloc(n);
        if (e != hipSuccess || n == 0) return e;
        return hipMemcpy(p, src, n, hipMemcpyHostToDevice);
    }
    template <class T> T *as() const { return static_cast<T *>(p); }
};

} // namespace hiprt_detail

struct hiprt_host_scene_s {
    rt::scene sc;
};

struct hiprt_bvh_s {
    rt::bvh b;
    rt::bvh_stats st;
};

// Per-stream state of a context: launches on one stream are ordered, so
// they can share a work-counter block and a descriptor table; launches on
// different streams get their own.
struct hiprt_stream_state {
    hiprt_detail::dbuf counter;       // work counters of the persistent kernels
    hiprt_detail::dbuf batch_table;   // descriptor table of the last batched trace on the stream
    hiprt_detail::dbuf spill;         // stack spill buffer of the persistent kernels (grown on demand)
    hiprt_detail::dbuf adjoint;       // sort scratch of the adjoint's vertex accumulation (grown on demand)
};

struct hiprt_context_s {
    int device = 0;
    std::mutex lock;                  // guards `streams`
    std::map<void *, std::unique_ptr<hiprt_stream_state>> streams;
    // Device BVH builds: scratch and result words kept for the next build on
    // any stream (a build waits for its own work, so they are idle between
    // builds).  A build that finds them in use allocates its own.
    std::mutex build_lock;
    hiprt_detail::dbuf build_scratch, build_result;
    // The state of `stream` (created on first use, counters zeroed); null on
    // allocation failure.
    hiprt_stream_state *state(void *stream);
};

struct hiprt_scene_s {
    hiprt_context ctx = nullptr;
    rt::flat_scene host;                         // host copy of the uploaded layout (a scene built on the
                                                 // device: its scalars only, see host_nodes)
    uint32_t n_nodes = 0, n_slots = 0;
    rt::node2 root{};                            // inner node 0 as a device build wrote it
    uint32_t group_rays = rt::dev::kGroupRays16; // rays up to which 8 lanes trace one of them (group_rays_of)
    hiprt_detail::dbuf arena;                    // one allocation behind the buffers below (device builds)
    hiprt_detail::dbuf nodes, tris, slot_ids;    // traversal data
    hiprt_detail::dbuf tri_geo, mats;            // shading data (scenes committed from a host scene)
    hiprt_detail::dbuf tri_vidx;                 // vertex indices per triangle (adjoint scatter)
    hiprt_detail::dbuf tri_ns;                   // corner shading normals per triangle (scenes with normals)
    hiprt_detail::dbuf alpha_tri, alpha_tex, alpha_mask;   // opacity data (scenes with textures)
    uint32_t n_tris = 0, n_vert = 0;
    int stack_need = 0;                          // most stack entries any traversal can hold
    hiprt_detail::dbuf light_rec, light_f, light_cdf;   // light list of the direct-lighting steps
    uint32_t n_lights = 0;
    float light_integral = 0.0f;
    hiprt_detail::dbuf refit_ranges, refit_boxes;   // leaf slots below each child; box tree over the slots (refit)
    rt::scene_desc desc{};
    // Stack need as the LDS-stack kernel takes it: 0, which keeps that kernel
    // out, for trees of more nodes than its 32-bit byte offsets reach.
    int lds_need() const { return n_nodes > rt::dev::kDynamicNodes ? 0 : stack_need; }
};

namespace hiprt_detail {

// Checks a flattened tree (children after their parent, leaf slots in range,
// depth and node limits) and computes the most stack entries a traversal can
// hold.  Returns "" when the tree is valid.
std::string check_layout(rt::flat_scene &f, uint32_t &stack_need);

// The scene's inner nodes on the host (references as committed; a scene built
// on the device copies them into `fetched` from device memory).
hipError_t host_nodes(const hiprt_scene_s *s, std::vector<rt::node2> &fetched, const rt::node2 *&nodes2,
                      const rt::node4 *&nodes4);

// Rays of one binary tree up to which the group trace's 8 lanes per ray are the
// faster (the launch's own limit applies too): `inner` and `leaf` sum half the
// surface of its inner nodes' boxes, without the root's, and of its leaves'.
//
// Over the root's surface these are the nodes Sn and leaves Sl that a random
// line meets.  Plain and persistent kernels have a floor, the slowest
// wavefront, and a slope that leaves set; the group trace pays for nodes and
// a fixed part per ray and has next to no floor, so it holds on the longer the
// more of a ray's work is leaves.  570,000 Sl^2 / Sn (1 - 3 / Sn) fits the measured
// crossings over random triangles and both halls.  Sl, Sn, limit; us of camera
// and random rays, closest hit, group / plain:
//   100 triangles     1.9   7.8  155 k  at 200 k 30 / 34, 60 / 54     300 k 41 / 34, 85 / 65
//   500               3.5  17.3  334 k  at 300 k 54 / 57, 113 / 118   500 k 79 / 61, 176 / 172
//   2,000             6.3  32.3  631 k  at 500 k 95 / 105, 233 / 256  800 k 145 / 138, 363 / 333
//   8,192            10.9  58.3  1.11 M at 800 k 174 / 207, 449 / 465  1 M 210 / 283, 550 / 558
//   74,068 (hall)     6.5  53.7  421 k  at 400 k 216 / 321, 239 / 229  640 k 324 / 229, 365 / 306
//   262,144 (hall)   17.6   131  1.31 M at 800 k 660 / 661, 765 / 1006  1 M 809 / 900, 943 / 1157
// A limit on the ray count alone, 1 M, took 481 us for 1 M camera rays of the
// small hall (plain 352) and 147 us for those of 500 triangles (plain 95).
uint32_t group_rays_of(double inner, double leaf, const rt::node2 &root);

// Fills the scene descriptor from the device buffers and the host copy.
void set_desc(hiprt_scene_s *s, uint32_t stack_need);

// The scene's descriptor for one trace: the opacity test on when `alpha`
// is asked for and the scene has opacity data.
rt::scene_desc desc_for(const hiprt_scene_s *sc, bool alpha);

// Gives `cfg` the spill buffer a persistent launch on stream `s` needs for
// trees whose traversal can hold `need` stack entries (none when the
// configuration's VGPR and LDS entries hold them): the stream state's
// buffer, grown once the stream's earlier launches, which may still use the
// old one, have finished.  `multi` selects the descriptor-table kernel;
// lds_need (hiprt_scene_s::lds_need) 0 keeps the LDS-stack kernel out;
// spill_limit > 0 caps the entries per lane (hiprt_tracer_opts::spill_limit).
hipError_t attach_spill(hiprt_stream_state *st, hipStream_t s, const rt::scene_desc &d, bool any, bool multi,
                        int need, int lds_need, rt::dev::persistent_cfg &cfg, int spill_limit = 0);

} // namespace hiprt_detail
