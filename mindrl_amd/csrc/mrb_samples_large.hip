// Samples of thousands of rows with large fields: the LDS-top kernel for them and its launch.
#include "mrb_launch.h"
#include "mrb_lds_sample.h"

namespace mrb {

namespace {

// (kernels of their own: in the others the code for large fields cost rows of 153 and 521 bytes 2 to 4 %)
template <int kStrata>
__global__ __launch_bounds__(kLdsWG) void k_per_sample_lds_large(const float* __restrict__ sum, const float* __restrict__ uniforms,
                                                              const float* __restrict__ mn, int depth, int lds_levels, int batch,
                                                              float beta, uint64_t seed, uint64_t calls, uint32_t rest, uint32_t large,
                                                              SampleArgs a, IoTable t) {
    sample_lds<kStrata, true>(sum, uniforms, mn, depth, lds_levels, batch, beta, seed, calls, rest, large, a, t);
}

}  // namespace

hipError_t launch_per_sample_lds_large(const SampleArgs& a, const IoTable& t, int64_t nbatch, int strata, int levels, uint32_t rest, uint32_t large,
                                       size_t lds, hipStream_t s) {
    auto* const kernel = strata == 16   ? k_per_sample_lds_large<16>
                         : strata == 32 ? k_per_sample_lds_large<32>
                         : strata == 64 ? k_per_sample_lds_large<64>
                                        : k_per_sample_lds_large<256>;
    launch_kernel(kernel, dim3((uint32_t)((a.batch + strata - 1) / strata), (uint32_t)nbatch), dim3(kLdsWG), lds, s, a.sum, a.uniforms, a.mn,
                  a.depth, levels, (int)a.batch, a.beta, a.seed, a.calls, rest, large, a, t);
    return hipGetLastError();
}

}  // namespace mrb
