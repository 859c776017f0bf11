// Samples of thousands of rows: the LDS-top kernel and its launch.
#include "mrb_launch.h"
#include "mrb_lds_sample.h"

namespace mrb {

namespace {

// (sum .. calls: see sample_lds)
template <int kStrata>
__global__ __launch_bounds__(kLdsWG) void k_per_sample_lds(const float* __restrict__ sum, const float* __restrict__ uniforms,
                                                        const float* __restrict__ mn, int depth, int lds_levels,
                                                        int batch, float beta, uint64_t seed, uint64_t calls, uint32_t rest,
                                                        SampleArgs a, IoTable t) {
    sample_lds<kStrata, false>(sum, uniforms, mn, depth, lds_levels, batch, beta, seed, calls, rest, 0, a, t);
}

}  // namespace

hipError_t launch_per_sample_lds(const SampleArgs& a, const IoTable& t, int64_t nbatch, int strata, int levels, uint32_t rest,
                                 hipStream_t s) {
    const uint32_t ntop = (2u << levels) < 4 ? 4 : (2u << levels);
    const uint64_t bytes = batch_bytes(t);
    uint64_t held = 0;
    for (int f = 0; f < t.nfields; ++f) held += t.row_bytes[f];
    held *= (uint64_t)(a.size >= 0 ? a.size : a.capacity);
    uint32_t large = 0, smaller = rest;
    bool whole = true;
    for (int f = 0; f < t.nfields; ++f) {
        if (!large_field(t, f, strata, nbatch, bytes, held)) continue;
        large |= 1u << f;
        smaller -= t.units[f];
        whole = whole && whole_pieces(t, f);
    }
    const size_t lds = ntop * sizeof(float) + ((size_t)strata + 1) * sizeof(int64_t);
    if (large) return launch_per_sample_lds_large(a, t, nbatch, strata, levels, smaller, large | (stores_through(bytes, kThroughSample, whole) ? 1u << 31 : 0u), lds, s);
    auto* const kernel = strata == 16   ? k_per_sample_lds<16>
                         : strata == 32 ? k_per_sample_lds<32>
                         : strata == 64 ? k_per_sample_lds<64>
                                        : k_per_sample_lds<256>;
    launch_kernel(kernel, dim3((uint32_t)((a.batch + strata - 1) / strata), (uint32_t)nbatch), dim3(kLdsWG), lds, s, a.sum,
                  a.uniforms, a.mn, a.depth, levels, (int)a.batch, a.beta, a.seed, a.calls, rest, a, t);
    return hipGetLastError();
}

}  // namespace mrb
