// update_priorities of a few thousand entries by runs of leaves, and the rebuild of very large trees (defined in
// mrb_range.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mrb {

// Levels that k_tree_range rebuilds on a tree of `depth` levels (at least 8): what is left above is a tree of its own.
int tree_range_levels(int depth);
// indices and priorities of n entries -> leaves and the tree_range_levels(depth) levels above them.
hipError_t launch_tree_range(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                             int64_t capacity, int depth, float alpha, hipStream_t s);
// An update driven by its entries on a very large tree, after k_update_stamp: the lowest g0 levels (4 to 6), and `dirty`
// gets the epoch for each run of 2^g_dirty of the nodes at depth - g0 that has a changed one.
hipError_t launch_tree_sparse(const int64_t* indices, const unsigned long long* stamp, const float* powered, float* sum, float* mn,
                              uint32_t* dirty, int64_t n, int64_t capacity, int depth, int g0, int g_dirty, uint32_t epoch,
                              hipStream_t s);
// From depth `top` (17 to 20) to the root: the tiles of 256 nodes whose word in `dirty` carries the epoch.
hipError_t launch_tree_runs(float* sum, float* mn, const uint32_t* dirty, float* maxp, int top, uint32_t epoch, hipStream_t s);

}  // namespace mrb
