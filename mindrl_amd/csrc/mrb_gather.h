// The gather's body (no kernels here).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mrb.h"
#include "mrb_rows.h"

namespace mrb {

// ---------------------------------------------------------------------------
// Gather: io_f[k] = store_f[slot_k]. slot_k is `fixed_slot` when that is >= 0
// (single-row read), else comes from `indices` or, when that is NULL, from the
// counter-based generator (uniform in [0, count), with replacement). Replaces P.BufferSample / P.BufferGetItem
// (mindspore_rl/core/uniform_replay_buffer.py:83-89,128,139).
// ---------------------------------------------------------------------------
template <typename Rows>
__device__ __forceinline__ void gather_body(const Rows& t, int64_t capacity, int64_t count, const int64_t* __restrict__ indices,
                                            int64_t fixed_slot, uint64_t seed, uint64_t calls, int64_t* __restrict__ out_indices,
                                            uint32_t* __restrict__ err, uint32_t blocks) {
    // blockIdx.y is the field: the table's entries for it are the same for every thread of the launch's row of
    // workgroups and come through scalar registers, requested with the other arguments. (Indexed by a field number
    // each thread works out for itself they were two more dependent trips to memory in a kernel that is a chain of
    // such trips and nothing else.)
    const int f = blockIdx.y;
    const uint32_t units = t.units(f), vl = t.vl(f), row_bytes = t.row_bytes(f), stride_f = t.stride(f);
    const gbyte* const store = as_global((const uint8_t*)t.store(f));
    gbyte* const io = as_global(t.io(f));
    const uint64_t total = t.granules(f);
    const uint64_t step = (uint64_t)blocks * kWG;
    for (uint64_t w = (uint64_t)blockIdx.x * kWG + threadIdx.x; w < total; w += step) {
        uint64_t row;
        uint32_t unit;
        split_work(w, units, row, unit);
        int64_t slot = fixed_slot >= 0 ? fixed_slot : indices ? indices[row] : rng_below(seed, calls, row, count);
        // a fixed slot was range-checked by the host against the ring (it may lie above `count` after a reset)
        if (fixed_slot < 0 && (slot < 0 || slot >= count)) {
            if (f == 0 && unit == 0) atomicOr(err, MRB_DERR_INDEX);
            slot = slot < 0 ? 0 : (count > 0 ? count - 1 : 0);
            if (slot >= capacity) slot = capacity - 1;
        }
        if (out_indices && f == 0 && unit == 0) out_indices[row] = slot;
        const uint32_t off = granule_offset(unit, vl, row_bytes);
        copy_granule(io + row * row_bytes + off, store + (uint64_t)slot * stride_f + off, vl);
    }
}

}  // namespace mrb
