// Samples of thousands of rows (defined in mrb_samples.hip and mrb_sample_lanes.hip).
#pragma once
#include "mrb_rows.h"

namespace mrb {

// nbatch batches of a.batch strata, `strata` (16, 32, 64 or 256) of them to a workgroup, `levels` of the tree in LDS; rest:
// the granules of a row outside the fields that each thread copies for its own stratum (see kLdsOwn).
hipError_t launch_per_sample_lds(const SampleArgs& a, const IoTable& t, int64_t nbatch, int strata, int levels, uint32_t rest,
                                 hipStream_t s);

// The same where some fields are large (a bit for each, and bit 31 to store through the L2; rest: of the others). launch_per_sample_lds calls it.
hipError_t launch_per_sample_lds_large(const SampleArgs& a, const IoTable& t, int64_t nbatch, int strata, int levels, uint32_t rest, uint32_t large,
                                       size_t lds, hipStream_t s);

// The same by sixteen lanes for each stratum: trees of at least kLanesFewestLevels levels, rows of at most kLanesMostNarrow bytes in
// narrow fields.
constexpr int kLanesFewestLevels = 7;
constexpr uint32_t kLanesMostNarrow = 48;
hipError_t launch_per_sample_lanes(const SampleArgs& a, const WidePlan& plan, int64_t nbatch, hipStream_t s);

}  // namespace mrb
