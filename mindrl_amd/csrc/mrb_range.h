// update_priorities of a few thousand entries as two launches (defined in mrb_range.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mrb {

// Levels that k_tree_range rebuilds on a tree of `depth` levels (at least 8): what is left above is a tree of its own.
int tree_range_levels(int depth);
// indices and priorities of n entries -> leaves and the tree_range_levels(depth) levels above them.
hipError_t launch_tree_range(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                             uint32_t* err, int64_t capacity, int depth, float alpha, hipStream_t s);
// The levels above depth `top`, at most 8.
hipError_t launch_tree_cap(float* sum, float* mn, int top, hipStream_t s);

}  // namespace mrb
