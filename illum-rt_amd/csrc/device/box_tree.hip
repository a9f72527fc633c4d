// Upper levels of a box tree (box_tree.h).
#include "box_tree.h"

namespace rt {
namespace dev {

namespace {

// A level of n entries and the ten above it.
__global__ __launch_bounds__(kBoxBlock) void k_box_levels(box6 *level, uint32_t n) {
    const uint32_t i = blockIdx.x * (uint32_t)kBoxBlock + threadIdx.x;
    box_levels(i < n ? level[i] : empty_box6(), level, n);
}

} // namespace

hipError_t launch_box_tree_top(box6 *tree, uint32_t n, hipStream_t stream) {
    for (;;) {
        for (int k = 0; k < 10; ++k) {   // to the last level the blocks have written
            if (n <= 1) return hipSuccess;
            tree += n;
            n = (n + 1) / 2;
        }
        if (n <= 1) return hipSuccess;
        hipLaunchKernelGGL(k_box_levels, dim3((n + kBoxBlock - 1) / kBoxBlock), dim3(kBoxBlock), 0, stream, tree, n);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
}

} // namespace dev
} // namespace rt
