// How the instantiations of k_discounted_return_tiled are launched.
#pragma once
#include "mrb_launch.h"
#include "mrb_returns.h"

namespace mrb {

template <bool kQuad, int kCols, int kMovers, bool kThrough>
void launch_returns(bool back, const float* x, const uint8_t* done, float* end_value, float* out, int64_t timesteps, int64_t batch, int64_t inner,
                    float gamma, hipStream_t s) {
    const dim3 grid((uint32_t)((batch * inner + kCols - 1) / kCols)), threads(64 + kMovers);
    launch_kernel(back ? k_discounted_return_tiled<true, kQuad, kCols, kMovers, kThrough> : k_discounted_return_tiled<false, kQuad, kCols, kMovers, kThrough>, grid,
                  threads, 0, s, x, done, end_value, out, timesteps, batch, inner, gamma);
}

// The kernels of sixteen and thirty-two columns to a workgroup that do not store through the L2 (defined in mrb_returns_streamed.hip).
void launch_returns_streamed(int group, bool quad, bool back, const float* x, const uint8_t* done, float* end_value, float* out, int64_t timesteps,
                             int64_t batch, int64_t inner, float gamma, hipStream_t s);

}  // namespace mrb
