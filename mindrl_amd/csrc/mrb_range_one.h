// update_priorities of up to 4096 entries, of up to 1024 with a push, in one launch (defined in mrb_range_one.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mrb_rows.h"

namespace mrb {

constexpr int kOneMostEntries = 4096;
constexpr int kOneMostRows = 512;          // pushed with it (2000 rows cost one or two workgroups 2 us)
constexpr uint32_t kOneMostRiders = 128;  // workgroups of its row copy (each is as large as the others: up to 128 KB of LDS)

// The pushed rows of an update and push as one call: `nrows` slots from first_slot on, around the ring's end; their
// priorities, or NULL.
struct RangePush {
    const float* priorities;
    uint32_t first_slot, nrows;
};

// Levels of the runs that a launch for n entries divides a tree of `depth` (8 to 22) levels into.
int range_one_levels(int depth, int64_t n);
// indices and priorities of n entries (1 .. kOneMostEntries; more than 1024 on trees of at most 20 levels) -> the trees and the running max.
hipError_t launch_range_one(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                            int64_t capacity, int depth, float alpha, hipStream_t s);
// The same (of up to 1024 entries) and then a push whose row copy is `put`, in one launch. With priorities the slots must lie in one run.
hipError_t launch_range_one_push(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                                 int64_t capacity, int depth, float alpha, const RangePush& push, const PutArgs& put, hipStream_t s);

}  // namespace mrb
