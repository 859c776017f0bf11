// Writes the levels of a tree that are not kept up (kSilentLevels, mrb_tree.h), for who wants every node (defined in mrb_silent.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mrb {

hipError_t launch_tree_silent(float* sum, float* mn, int64_t leaves, hipStream_t s);

}  // namespace mrb
