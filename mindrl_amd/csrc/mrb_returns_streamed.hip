// The instantiations of k_discounted_return_tiled for sixteen and thirty-two columns that do not store through the L2.
#include "mrb_returns_launch.h"

namespace mrb {

void launch_returns_streamed(int group, bool quad, bool back, const float* x, const uint8_t* done, float* end_value, float* out, int64_t timesteps,
                             int64_t batch, int64_t inner, float gamma, hipStream_t s) {
    if (group == 16)
        (quad ? launch_returns<true, 16, 256, false> : launch_returns<false, 16, 256, false>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else
        (quad ? launch_returns<true, 32, 256, false> : launch_returns<false, 32, 512, false>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
}

}  // namespace mrb
