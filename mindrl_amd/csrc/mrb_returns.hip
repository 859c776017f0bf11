// Most instantiations of k_discounted_return_tiled and the rule that chooses among them.
#include "mrb_returns_launch.h"

namespace mrb {

// Columns per workgroup. Narrow groups spread the recurrence's waves and the memory traffic over more compute units; wide ones read
// longer pieces of a row, which the memory serves better, and which counts when the call is more than the caches hold. Measured, us for
// 16 / 32 / 64 columns per group: [1000, 4096] 11.8 / 15.4 / 16.1, [1000, 8192] 15.3 / 15.8 / 16.6, [2000, 8192] 43 / 29.5 / 40, [1000, 12000] 31.6 / 26.1 /
// 22.7, [1000, 16384] 43 / 33 / 28.7, [500, 20000] 28.6 / 21.3 / 22.8, [1000, 40000] 67 / 60 / 57. A short time axis moves less, and sixteen stay
// the best or within 0.2 us of it: [100, 8192] 4.6 / 4.5 / 5.2, [100, 16384] 5.8 / 6.0 / 5.8, [64, 20000] 5.8 / 6.6 / 8.4, [100, 30001] 10.5 / 13.1 /
// 10.7. Sixty-four columns take the movers that carry four steps of one column: the other kind's scalar LDS writes meet in the
// same banks there.
hipError_t launch_discounted_return_tiled(bool back, const float* x, const uint8_t* done, float* end_value, float* out,
                                          int64_t timesteps, int64_t batch, int64_t inner, float gamma, hipStream_t s) {
    const int64_t cols = batch * inner;
    const bool quad = inner == 1 && cols >= 4;
    const int group = cols <= 4096 || timesteps < 128 ? 16 : cols <= 8192 ? 32 : 64;
    if (group < 64 && !returns_through(timesteps, cols, group))
        launch_returns_streamed(group, quad, back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else if (group == 16)
        (quad ? launch_returns<true, 16, 256, true> : launch_returns<false, 16, 256, true>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else if (group == 32)
        (quad ? launch_returns<true, 32, 256, true> : launch_returns<false, 32, 512, true>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else
        launch_returns<false, 64, 512, false>(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    return hipGetLastError();
}

}  // namespace mrb
