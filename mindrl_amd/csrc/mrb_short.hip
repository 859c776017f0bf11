#include "mrb_short.h"

#include "mrb_gather.h"
#include "mrb_launch.h"

namespace mrb {

namespace {

// (The leading plain parameters are preloaded into scalar registers.)
__global__ __launch_bounds__(kWG) void k_short_gather(const RowTable* __restrict__ table, const int64_t* __restrict__ indices, uint64_t seed,
                                                      uint64_t calls, uint32_t count, uint32_t n, uint32_t blocks, int with_indices, ShortIo io) {
    gather_body(ShortRows{table, io, n, with_indices}, table->capacity, count, indices, -1, seed, calls,
                with_indices ? reinterpret_cast<int64_t*>(io.at(0)) : nullptr, table->err, blocks);
}

// The same for many granules: four to a thread of the large fields, each field its own workgroups. (A kernel of its own: in one with the
// other, whose threads need 18 registers, they had 46, and 16,384 drawn rows of 899 bytes, a granule to a thread, took 10.4 us for 9.8.)
__global__ __launch_bounds__(kWG) void k_short_gather_many(const RowTable* __restrict__ table, const int64_t* __restrict__ indices, uint64_t seed,
                                                           uint64_t calls, uint32_t count, uint32_t n, int flags, ShortIo io) {
    gather_fields(ShortRows{table, io, n, flags & 1}, indices, count, seed, calls, blockIdx.x, flags & 2);
}

__global__ __launch_bounds__(kWG) void k_short_put(const RowTable* __restrict__ table, uint32_t first_slot, uint32_t n, uint32_t blocks,
                                                   ShortIo io) {
    put_fields(table, io, first_slot, n, blockIdx.x, blocks);
}

// Pushes: workgroup (0, 0) does the tree's work, those with a column of at least 1 copy rows of field blockIdx.y.
__global__ __launch_bounds__(kWG) void k_short_push_one(float* __restrict__ sum, float* __restrict__ mn, float* maxp,
                                                        const RowTable* __restrict__ table, const float* priority, uint32_t first_slot,
                                                        int depth, float alpha, uint32_t blocks, ShortIo io) {
    if (__builtin_expect((blockIdx.x | blockIdx.y) != 0, 0)) {  // (the tree workgroup's code comes first)
        if (blockIdx.x) put_field(table, io, blockIdx.y, first_slot, 1, blockIdx.x - 1, blocks, kWG);
        rider_ends();
    }
    if (threadIdx.x >= 64) return;
    CounterTicket none{};
    push_one_walk<false>(sum, mn, maxp, first_slot, 0, (int64_t)1 << depth, depth, alpha, priority, err_before(maxp), threadIdx.x, none, false,
                         false, 0);
}

// plan: depth | units << 8 | threads == kFusedWG << 16 | raise the running max << 17
__global__ __launch_bounds__(kFusedWG) void k_short_push_run(float* sum, float* mn, float* maxp, const float* priorities,
                                                             const RowTable* __restrict__ table, uint32_t first_slot, uint32_t n, uint32_t plan,
                                                             float alpha, uint32_t capacity, uint32_t blocks, ShortIo io) {
    const uint32_t threads = plan >> 16 & 1u ? (uint32_t)kFusedWG : (uint32_t)kWG;
    if (__builtin_expect((blockIdx.x | blockIdx.y) != 0, 0)) {
        if (blockIdx.x) put_field(table, io, blockIdx.y, first_slot, n, blockIdx.x - 1, blocks, threads);
        rider_ends();
    }
    UpdateArgs a{};
    a.priorities = priorities;
    a.n = n;
    a.first_slot = first_slot;
    a.capacity = capacity;
    a.depth = (int)(plan & 255u);
    a.leaves = (int64_t)1 << a.depth;
    a.alpha = alpha;
    a.sum = sum;
    a.mn = mn;
    a.maxp = maxp;
    a.err = err_before(maxp);
    a.fold_max = (int)(plan >> 17 & 1u);
    push_run_body(a, plan >> 8 & 255u, threads);
}

}  // namespace

hipError_t launch_short_gather(const RowTable* table, const ShortIo& io, const IoTable& t, const int64_t* indices, int64_t count, uint64_t seed,
                               uint64_t calls, int64_t n, uint32_t blocks, bool with_indices, hipStream_t s) {
    if (blocks > (indices ? kGatherFew : kGatherFewDrawn)) {
        dim3 grid(0);
        bool whole = true;
        for (int f = 0; f < t.nfields; ++f) {
            grid.x += put_blocks(t.prefix[f + 1] - t.prefix[f], kWG);
            if (t.vec_log2[f] == 4) whole = whole && whole_pieces(t, f);
        }
        launch_kernel(k_short_gather_many, grid, dim3(kWG), 0, s, table, indices, seed, calls, (uint32_t)count, (uint32_t)n,
                      (with_indices ? 1 : 0) | (stores_through(batch_bytes(t), kThroughGather, whole) ? 2 : 0), io);
        return hipGetLastError();
    }
    launch_kernel(k_short_gather, dim3(blocks, (uint32_t)t.nfields), dim3(kWG), 0, s, table, indices, seed, calls, (uint32_t)count, (uint32_t)n,
                  blocks, with_indices ? 1 : 0, io);
    return hipGetLastError();
}

hipError_t launch_short_put(const RowTable* table, const ShortIo& io, const IoTable& t, int64_t first_slot, int64_t n, hipStream_t s) {
    uint32_t blocks;
    const dim3 grid = put_grid(t, 0, blocks);
    launch_kernel(k_short_put, grid, dim3(kWG), 0, s, table, (uint32_t)first_slot, (uint32_t)n, blocks, io);
    return hipGetLastError();
}

hipError_t launch_short_push_one(const RowTable* table, const ShortIo& io, int nfields, float* sum, float* mn, float* maxp, int64_t first_slot,
                                 int depth, float alpha, const float* priority, uint64_t granules, hipStream_t s) {
    const uint32_t blocks = put_blocks(granules, kWG);
    launch_kernel(k_short_push_one, dim3(1 + blocks, (uint32_t)nfields), dim3(kWG), 0, s, sum, mn, maxp, table, priority,
                  (uint32_t)first_slot, depth, alpha, blocks, io);
    return hipGetLastError();
}

hipError_t launch_short_push_run(const RowTable* table, const ShortIo& io, int nfields, const UpdateArgs& a, uint32_t units, uint64_t granules,
                                 uint32_t threads, hipStream_t s) {
    const uint32_t plan = (uint32_t)a.depth | units << 8 | (threads == (uint32_t)kFusedWG ? 1u << 16 : 0u) | (a.fold_max ? 1u << 17 : 0u);
    const uint32_t blocks = put_blocks(granules, threads);
    launch_kernel(k_short_push_run, dim3(1 + blocks, (uint32_t)nfields), dim3(threads), 0, s, a.sum, a.mn, a.maxp, a.priorities, table,
                  (uint32_t)a.first_slot, (uint32_t)a.n, plan, a.alpha, (uint32_t)a.capacity, blocks, io);
    return hipGetLastError();
}

}  // namespace mrb
