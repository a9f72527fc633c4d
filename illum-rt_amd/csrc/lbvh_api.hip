// C ABI of the device BVH build: triangles in device memory in, a committed
// scene out, without a host-side builder.
#include "capi_internal.h"

#include "device/lbvh_kernels.h"

#include <cstring>
#include <memory>
#include <new>
#include <vector>

using hiprt_detail::dbuf;
using hiprt_detail::fail;
using hiprt_detail::ok;

namespace {
// Build scratch up to this size (about 1.5 million triangles) stays with the
// context for the next build; more is returned after the call.
constexpr size_t kKeptScratchBytes = size_t(256) << 20;
} // namespace

extern "C" {

int hiprt_scene_build(hiprt_context ctx, const float *d_positions, uint32_t n_vert, const uint32_t *d_indices,
                      uint32_t n_tris, const uint32_t *d_materials, const float *materials, uint32_t n_materials,
                      int32_t max_leaf, int32_t tri_format, hiprt_scene *out, float *device_ms, void *stream) {
    if (!ctx || !out) return fail(HIPRT_ERR_ARG, "null argument");
    if ((n_tris && (!d_positions || !d_indices)) || (n_materials && !materials))
        return fail(HIPRT_ERR_ARG, "null array");
    if (max_leaf < 1 || max_leaf > (int32_t)rt::kMaxLeafCount) return fail(HIPRT_ERR_ARG, "max_leaf must be 1..32");
    if (tri_format != HIPRT_TRI_EXACT && tri_format != HIPRT_TRI_WOOP) return fail(HIPRT_ERR_ARG, "unknown tri_format");
    if (n_tris > rt::kMaxLeafSlot) return fail(HIPRT_ERR_ARG, "too many triangles for the 26-bit slot field");
    HIP_TRY(hipSetDevice(ctx->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    std::unique_ptr<hiprt_scene_s> sc(new (std::nothrow) hiprt_scene_s);
    if (!sc) return fail(HIPRT_ERR_ARG, "out of host memory");
    sc->ctx = ctx;
    const uint32_t n = n_tris, m = n > 1 ? n - 1 : 1, n1 = n ? n : 1;
    const size_t scratch_bytes = rt::dev::lbvh_scratch_bytes(n);
    dbuf own, own_result;   // (freed after the lock: theirs is not shared)
    std::unique_lock<std::mutex> mine(ctx->build_lock, std::try_to_lock);
    dbuf &scratch = mine.owns_lock() && scratch_bytes <= kKeptScratchBytes ? ctx->build_scratch : own;
    dbuf &result = mine.owns_lock() ? ctx->build_result : own_result;
    auto need = [](dbuf &b, size_t bytes) {   // (the last build that used it has ended)
        if (b.bytes >= bytes) return hipSuccess;
        hipError_t e = b.alloc(bytes);
        if (e != hipSuccess) b.release();
        return e;
    };
    HIP_TRY(need(scratch, scratch_bytes));
    const uint32_t n_areas = rt::dev::lbvh_area_blocks(n);
    const size_t result_bytes = sizeof(rt::dev::lbvh_result) + n_areas * sizeof(float2);
    HIP_TRY(need(result, result_bytes));
    // on the stack while it is small: a copy into fresh heap memory takes 5-10 us longer
    alignas(16) char near_result[8192];
    std::vector<char> far_result(result_bytes > sizeof near_result ? result_bytes : 0);
    char *host_result = far_result.empty() ? near_result : far_result.data();
    std::vector<float> mats(8 * (n_materials ? n_materials : 1), 0.0f);
    if (n_materials) std::memcpy(mats.data(), materials, 32ull * n_materials);
    // one allocation for the scene: each hipMalloc of this size takes 20-30 us
    {
        struct {
            dbuf &b;
            size_t bytes;
        } part[] = {{sc->nodes, sizeof(rt::node2) * m}, {sc->tris, sizeof(rt::tri_rec) * n1}, {sc->slot_ids, 4ull * n1},
                    {sc->tri_geo, 48ull * n1},          {sc->tri_vidx, 12ull * n1},          {sc->mats, mats.size() * 4}};
        auto align = [](size_t x) { return (x + 255) & ~size_t(255); };
        size_t total = 0;
        for (auto &q : part) total += align(q.bytes);
        HIP_TRY(sc->arena.alloc(total));
        char *at = sc->arena.as<char>();
        for (auto &q : part) {
            q.b.view(at, q.bytes);
            at += align(q.bytes);
        }
    }
    auto *d_result = result.as<rt::dev::lbvh_result>();
    rt::dev::lbvh_in in{d_positions, d_indices, d_materials, n_vert, n, n_materials ? n_materials : 1, max_leaf, tri_format};
    rt::dev::lbvh_out o{sc->nodes.as<rt::node2>(), sc->tris.as<rt::tri_rec>(), sc->slot_ids.as<uint32_t>(),
                        sc->tri_geo.as<float>(),   sc->tri_vidx.as<uint32_t>(), d_result,
                        reinterpret_cast<float2 *>(d_result + 1)};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (device_ms) {
        HIP_TRY(hipEventCreate(&e0));
        HIP_TRY(hipEventCreate(&e1));
        HIP_TRY(hipEventRecord(e0, s));
    }
    hipError_t le = rt::dev::launch_lbvh(in, o, scratch.p, s);
    if (device_ms && le == hipSuccess) le = hipEventRecord(e1, s);
    if (le == hipSuccess) le = hipMemcpyAsync(sc->mats.p, mats.data(), mats.size() * 4, hipMemcpyHostToDevice, s);
    if (le == hipSuccess) le = hipMemcpyAsync(host_result, d_result, result_bytes, hipMemcpyDeviceToHost, s);
    // (waits also after a failed launch: the buffers must be idle when freed)
    hipError_t we = hipStreamSynchronize(s);
    if (le == hipSuccess) le = we;
    if (le == hipSuccess && device_ms) le = hipEventElapsedTime(device_ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (le != hipSuccess) return fail(HIPRT_ERR_HIP, std::string("device BVH build: ") + hipGetErrorString(le));

    const auto &res = *reinterpret_cast<const rt::dev::lbvh_result *>(host_result);
    const uint32_t *counts = res.counts;
    if (counts[2]) return fail(HIPRT_ERR_ARG, std::to_string(counts[2]) + " triangles name a vertex past n_vert");
    if (counts[3]) return fail(HIPRT_ERR_HIP, "device BVH build produced a node off the tree");
    if (counts[0] > m) return fail(HIPRT_ERR_HIP, "device BVH build: node count out of range");
    if (counts[4]) return fail(HIPRT_ERR_ARG, "triangle material id out of range");

    // The emit kernel has made the checks an uploaded tree gets on the host
    // (children after their parent, slot ranges); a binary tree's stack need
    // is its depth, and no box bound is NaN (box_tree.h).  The tree stays on
    // the device: host_nodes fetches it for who needs it.
    rt::flat_scene &h = sc->host;
    h.bvh_kind = rt::BVH2;
    h.tri_kind = tri_format;
    h.root_ref = res.root_ref;
    sc->root = res.root;
    h.depth = counts[1];
    hiprt_detail::set_desc(sc.get(), counts[1]);
    sc->n_nodes = counts[0];
    sc->n_slots = n;
    if (counts[0]) {
        const auto *areas = reinterpret_cast<const float2 *>(host_result + sizeof res);
        double inner = 0, leaf = 0;
        for (uint32_t k = 0; k < n_areas; ++k) {
            inner += areas[k].x;
            leaf += areas[k].y;
        }
        sc->group_rays = hiprt_detail::group_rays_of(inner, leaf, res.root);
    }
    sc->desc.nan_free = 1;
    sc->desc.nested = 1;   // unions; a subtree of empty boxes holds no triangle to hit
    sc->n_tris = n;
    sc->n_vert = n_vert;
    *out = sc.release();
    return ok();
}

} // extern "C"
