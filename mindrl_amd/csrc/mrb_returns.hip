// The instantiations of k_discounted_return_tiled and the rule that chooses among them.
#include "mrb_returns.h"

namespace mrb {

namespace {

template <bool kQuad, int kCols, int kMovers>
void launch(bool back, const float* x, const uint8_t* done, float* end_value, float* out, int64_t timesteps, int64_t batch,
            int64_t inner, float gamma, hipStream_t s) {
    const dim3 grid((uint32_t)((batch * inner + kCols - 1) / kCols)), threads(64 + kMovers);
    if (back)
        hipLaunchKernelGGL((k_discounted_return_tiled<true, kQuad, kCols, kMovers>), grid, threads, 0, s, x, done, end_value, out,
                           timesteps, batch, inner, gamma);
    else
        hipLaunchKernelGGL((k_discounted_return_tiled<false, kQuad, kCols, kMovers>), grid, threads, 0, s, x, done, end_value, out,
                           timesteps, batch, inner, gamma);
}

}  // namespace

// Columns per workgroup: sixteen while that fills at most one workgroup per compute unit (4096 columns), thirty-two up
// to 8192, sixty-four beyond. Narrow groups spread the recurrence's waves and the memory traffic over more compute
// units; wide ones read longer pieces of a row, which the memory serves better (3.1, 4.4 and 4.8 TB/s for 16, 32 and
// 64 columns when every compute unit has work). Measured, us for 16 / 32 / 64 columns per group: [1000, 32] 11.9 /
// 13.7 / 17.9, [1000, 4096] 14.5 / 15.8 / 21.8, [1000, 8192] 26.2 / 17.7 / 24.1, [1000, 16384] 48 / 34.5 / 30.6. A short
// time axis keeps thirty-two ([100, 16384]: 7.9 / 6.8 / 7.6). Sixty-four columns take the movers that carry four steps of
// one column: the other kind's scalar LDS writes meet in the same banks there (29 us at [1000, 32]).
hipError_t launch_discounted_return_tiled(bool back, const float* x, const uint8_t* done, float* end_value, float* out,
                                          int64_t timesteps, int64_t batch, int64_t inner, float gamma, hipStream_t s) {
    const int64_t cols = batch * inner;
    const bool quad = inner == 1 && cols >= 4;
    if (cols > 8192 && timesteps >= 128)
        launch<false, 64, 512>(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else if (cols > 4096)
        (quad ? launch<true, 32, 256> : launch<false, 32, 512>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    else
        (quad ? launch<true, 16, 256> : launch<false, 16, 256>)(back, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    return hipGetLastError();
}

}  // namespace mrb
