#include "mrb_short.h"

#include "mrb_gather.h"

namespace mrb {

namespace {

// (The leading plain parameters are preloaded into scalar registers.)
__global__ __launch_bounds__(kWG) void k_short_gather(const RowTable* __restrict__ table, const int64_t* __restrict__ indices, uint64_t seed,
                                                      uint64_t calls, uint32_t count, uint32_t n, uint32_t blocks, int with_indices, ShortIo io) {
    gather_body(ShortRows{table, io, n, with_indices}, table->capacity, count, indices, -1, seed, calls,
                with_indices ? reinterpret_cast<int64_t*>(io.at(0)) : nullptr, table->err, blocks);
}

// The copy of a ring append, one field's n rows by workgroup `block` of `blocks` with `threads` threads each. (A row of
// workgroups per field: what the table says of it is the same for all its threads and comes in one trip through scalar
// registers.) A thread has up to four granules on their way before it stores the first.
constexpr int kPutTrip = 4;

__device__ __forceinline__ void put_field(const RowTable* __restrict__ table, const ShortIo& io, int f, uint32_t first_slot, uint32_t n,
                                          uint32_t block, uint32_t blocks, uint32_t threads) {
    const ShortRows rows{table, io, n, 0};
    const uint32_t units = rows.units(f), vl = rows.vl(f), row_bytes = rows.row_bytes(f), stride = rows.stride(f);
    gbyte* const store = as_global(rows.store(f));
    const gbyte* const from = as_global((const uint8_t*)rows.io(f));
    const uint64_t ring = (uint64_t)table->capacity, total = (uint64_t)n * units, step = (uint64_t)blocks * threads;
    auto place = [&](uint64_t w, const gbyte*& src) -> gbyte* {
        uint64_t row;
        uint32_t unit;
        split_work(w, units, row, unit);
        uint64_t slot = first_slot + row;
        if (slot >= ring) slot -= ring;
        const uint32_t off = granule_offset(unit, vl, row_bytes);
        src = from + row * row_bytes + off;
        return store + slot * stride + off;
    };
    uint64_t w = (uint64_t)block * threads + threadIdx.x;
    if (vl == 4) {  // (uniform)
        for (; w < total; w += kPutTrip * step) {
            granule_t held[kPutTrip];
            gbyte* to[kPutTrip];
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q) {
                const gbyte* src;
                to[q] = place(w + q * step < total ? w + q * step : w, src);  // (past the end: the thread's first again)
                held[q] = __builtin_nontemporal_load((const g16*)src);
            }
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q) asm volatile("" : "+v"(held[q]));
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q)
                if (w + q * step < total) __builtin_nontemporal_store(held[q], (g16*)to[q]);
        }
        return;
    }
    for (; w < total; w += step) {
        const gbyte* src;
        gbyte* const to = place(w, src);
        copy_granule(to, src, vl);
    }
}

__global__ __launch_bounds__(kWG) void k_short_put(const RowTable* __restrict__ table, uint32_t first_slot, uint32_t n, uint32_t blocks,
                                                   ShortIo io) {
    put_field(table, io, blockIdx.y, first_slot, n, blockIdx.x, blocks, kWG);
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

// Workgroups per field: one granule to a thread where that is all there is to do, four where the launch would be tens of
// thousands of waves (a call of 32 MB: 9.1 us with one, 6.5 with four).
uint32_t put_blocks(uint64_t granules, uint32_t threads) {
    uint64_t blocks = (granules + threads - 1) / threads;
    if (blocks > 512) blocks = (blocks + kPutTrip - 1) / kPutTrip;
    return (uint32_t)(blocks < 16384 ? blocks : 16384);
}

}  // namespace

hipError_t launch_short_gather(const RowTable* table, const ShortIo& io, int nfields, const int64_t* indices, int64_t count, uint64_t seed,
                               uint64_t calls, int64_t n, uint32_t blocks, bool with_indices, hipStream_t s) {
    hipLaunchKernelGGL(k_short_gather, dim3(blocks, (uint32_t)nfields), dim3(kWG), 0, s, table, indices, seed, calls, (uint32_t)count, (uint32_t)n,
                       blocks, with_indices ? 1 : 0, io);
    return hipGetLastError();
}

hipError_t launch_short_put(const RowTable* table, const ShortIo& io, int nfields, int64_t first_slot, int64_t n, uint64_t granules,
                            hipStream_t s) {
    const uint32_t blocks = put_blocks(granules, kWG);
    hipLaunchKernelGGL(k_short_put, dim3(blocks, (uint32_t)nfields), dim3(kWG), 0, s, table, (uint32_t)first_slot, (uint32_t)n, blocks, io);
    return hipGetLastError();
}

hipError_t launch_short_push_one(const RowTable* table, const ShortIo& io, int nfields, float* sum, float* mn, float* maxp, int64_t first_slot,
                                 int depth, float alpha, const float* priority, uint64_t granules, hipStream_t s) {
    const uint32_t blocks = put_blocks(granules, kWG);
    hipLaunchKernelGGL(k_short_push_one, dim3(1 + blocks, (uint32_t)nfields), dim3(kWG), 0, s, sum, mn, maxp, table, priority,
                       (uint32_t)first_slot, depth, alpha, blocks, io);
    return hipGetLastError();
}

hipError_t launch_short_push_run(const RowTable* table, const ShortIo& io, int nfields, const UpdateArgs& a, uint32_t units, uint64_t granules,
                                 uint32_t threads, hipStream_t s) {
    const uint32_t plan = (uint32_t)a.depth | units << 8 | (threads == (uint32_t)kFusedWG ? 1u << 16 : 0u) | (a.fold_max ? 1u << 17 : 0u);
    const uint32_t blocks = put_blocks(granules, threads);
    hipLaunchKernelGGL(k_short_push_run, dim3(1 + blocks, (uint32_t)nfields), dim3(threads), 0, s, a.sum, a.mn, a.maxp, a.priorities, table,
                       (uint32_t)a.first_slot, (uint32_t)a.n, plan, a.alpha, (uint32_t)a.capacity, blocks, io);
    return hipGetLastError();
}

}  // namespace mrb
