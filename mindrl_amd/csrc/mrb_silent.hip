#include "mrb_silent.h"

#include "mrb_launch.h"
#include "mrb_rows.h"
#include "mrb_tree.h"

namespace mrb {

namespace {

// The silent levels, from the leaves: a thread per eight of those.
__global__ __launch_bounds__(kWG) void k_tree_silent(float* sum, float* mn, uint32_t leaves) {
    static_assert(kSilentLevels == 3, "eight leaves");
    const uint32_t eight = blockIdx.x * kWG + threadIdx.x;
    if (eight >= leaves / 8) return;
    auto levels = [&](float* tree, auto of) {
        const float4 a = *reinterpret_cast<const float4*>(tree + leaves + 8 * eight), b = *reinterpret_cast<const float4*>(tree + leaves + 8 * eight + 4);
        const float4 pairs = make_float4(of(a.x, a.y), of(a.z, a.w), of(b.x, b.y), of(b.z, b.w));
        const float2 fours = make_float2(of(pairs.x, pairs.y), of(pairs.z, pairs.w));
        *reinterpret_cast<float4*>(tree + leaves / 2 + 4 * eight) = pairs;
        *reinterpret_cast<float2*>(tree + leaves / 4 + 2 * eight) = fours;
        tree[leaves / 8 + eight] = of(fours.x, fours.y);
    };
    levels(sum, [](float x, float y) { return x + y; });
    levels(mn, [](float x, float y) { return fminf(x, y); });
}

}  // namespace

hipError_t launch_tree_silent(float* sum, float* mn, int64_t leaves, hipStream_t s) {
    launch_kernel(k_tree_silent, dim3((uint32_t)((leaves / 8 + kWG - 1) / kWG)), dim3(kWG), 0, s, sum, mn, (uint32_t)leaves);
    return hipGetLastError();
}

}  // namespace mrb
