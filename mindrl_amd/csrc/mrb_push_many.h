// Pushes in one launch of several workgroups (defined in mrb_push_many.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mrb_short.h"

namespace mrb {

constexpr uint32_t kManyMostTiles = 256;  // (their roots lie under two tiles at most)

// A push of n rows to consecutive slots from first_slot on (not around the ring's end), on a tree of more than 8 levels, with
// its row copy (t: the call's table). With priorities, running max included.
hipError_t launch_push_many(const RowTable* table, const ShortIo& io, const IoTable& t, float* sum, float* mn, float* maxp, const float* priorities,
                            int64_t first_slot, int64_t n, int depth, float alpha, hipStream_t s);

}  // namespace mrb
