// Kernels whose arguments are short (defined in mrb_short.hip): the same bodies as the kernels of mrb_kernels.h with the
// buffer's constant tables read from device memory and the caller's matrices given as distances from the first.
//
// A launch's arguments are written across the bus and the last of them is read back before the launch: up to 112 bytes cost a
// process whose memory is far from the device 2.7 us of host time, 120 to 960 bytes 3.1 to 3.9, more than a kilobyte 4.1 to 4.5.
// By-value field tables are 550 to 1000 bytes, and nearly all of them is the same in every call. On the device a kernel's first
// trip reads what it needs of the table into scalar registers, and the copies have a row of workgroups per field instead of a
// search for each granule's field. Device time per call, us, by value / short: an append of 1 row 2.85 / 2.04, of 1000 rows of
// 133 bytes 3.08 / 2.39, of 57.5 MB (read and written) 15.5 / 11.4; a gather of 256 rows of 162 bytes 3.17 / 2.66, of 8192 rows
// of 133 bytes 4.87 / 4.25; a push of 1 row 2.86 / 2.28, of 64 3.09 / 2.84, of 1000 3.56 / 3.13. Host
// time of one uniform insert and sample 10.0 / 9.2.
//
// By value stay: more than kShortPointers matrices, matrices too far apart at an odd address, device-resident counters, single-row
// reads, copies from another buffer's ring; the sampling kernels and the reservoir's push (3.35 / 3.40 and 2.8 / 2.9 when they
// were tried: their row copies come last, so the table's trip is not hidden); and the gather with a workgroup or a wave to a row, which takes a plan
// that a wave divides its lanes by (within 4 % of each other either way, 24,831-byte rows slower short).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mrb_push.h"
#include "mrb_rows.h"

namespace mrb {

constexpr int kShortPointers = 8;

// The matrices of a call: up to kShortPointers addresses, as distances from the first in units of 1 << shift bytes (what
// torch's allocator gives lies 512 bytes from each other or a multiple of that, and anywhere in the device's address space).
struct ShortIo {
    uint64_t base;
    uint32_t shift;
    int32_t away[kShortPointers - 1];
    __device__ __forceinline__ uint8_t* at(int i) const {
        return reinterpret_cast<uint8_t*>(base + (i ? (uint64_t)((int64_t)away[i - 1] << shift) : 0));
    }
};

// What stays the same of a buffer's arguments from call to call, in device memory.
struct RowTable {
    IoTable t;  // (store, row_bytes, stride, units and vec_log2 of it)
    int64_t capacity;
    uint32_t* err;  // the buffer's flags
};

// The fields of n rows (see FullRows); `first`: the number of the first field's matrix in io.
struct ShortRows {
    const RowTable* r;
    const ShortIo& s;
    uint64_t n;
    int first;
    __device__ __forceinline__ uint32_t units(int f) const { return r->t.units[f]; }
    __device__ __forceinline__ uint32_t vl(int f) const { return r->t.vec_log2[f]; }
    __device__ __forceinline__ uint32_t row_bytes(int f) const { return r->t.row_bytes[f]; }
    __device__ __forceinline__ uint32_t stride(int f) const { return r->t.stride[f]; }
    __device__ __forceinline__ uint8_t* store(int f) const { return r->t.store[f]; }
    __device__ __forceinline__ uint8_t* io(int f) const { return s.at(first + f); }
    __device__ __forceinline__ uint64_t granules(int f) const { return n * r->t.units[f]; }
};

constexpr int kPutTrip = 4;
constexpr uint32_t kPutFew = 512;  // workgroups up to which a thread has one

// Workgroups per field: one granule to a thread where that is all there is to do, four where the launch would be tens of
// thousands of waves (16 MB
// 4.8 us with one, 3.4 with four; 57 MB of odd rows 15.0 / 11.4; 200 MB 44.9 / 35.2; 500 MB 110 / 85, and 92 with a thread's four
// a launch's width apart).
__host__ __device__ inline uint32_t put_blocks(uint64_t granules, uint32_t threads) {
    uint64_t blocks = (granules + threads - 1) / threads;
    if (blocks > kPutFew) blocks = (blocks + kPutTrip - 1) / kPutTrip;
    return (uint32_t)(blocks < 16384 ? blocks : 16384);
}

// The field whose workgroups hold number `block` of those of all fields, one field's behind the other's; `block` is left as the number among
// that field's, which are `blocks`. (The fields' sizes in one trip: with a dependent one for each, and four granules to a
// thread of the small fields too, a gather of 4096 rows of 400 bytes in five fields took 6.0 us, with a granule to a thread 3.3.)
__device__ __forceinline__ int field_of_block(const RowTable* __restrict__ table, uint64_t n, uint32_t& block, uint32_t& blocks) {
    uint32_t units[kShortPointers];
#pragma unroll
    for (int f = 0; f < kShortPointers; ++f) units[f] = table->t.units[f];
    const int nfields = table->t.nfields;
    int at = 0;
    blocks = put_blocks(n * units[0], kWG);
#pragma unroll
    for (int f = 1; f < kShortPointers; ++f)
        if (at == f - 1 && f < nfields && block >= blocks) {
            block -= blocks;
            blocks = put_blocks(n * units[f], kWG);
            at = f;
        }
    return at;
}

// The copy of a ring append, one field's n rows by workgroup `block` of `blocks` with `threads` threads each. (A row of
// workgroups per field: what the table says of it is the same for all its threads and comes in one trip through scalar
// registers.) A thread has up to four granules on their way before it stores the first.

__device__ __forceinline__ void put_field(const RowTable* __restrict__ table, const ShortIo& io, int f, uint32_t first_slot, uint32_t n,
                                          uint32_t block, uint32_t blocks, uint32_t threads) {
    const ShortRows rows{table, io, n, 0};
    const uint32_t units = rows.units(f), vl = rows.vl(f), row_bytes = rows.row_bytes(f), stride = rows.stride(f);
    gbyte* const store = as_global(rows.store(f));
    const gbyte* const from = as_global((const uint8_t*)rows.io(f));
    const uint64_t ring = (uint64_t)table->capacity, total = (uint64_t)n * units;
    // granules of a thread and trip: side by side those of a workgroup, which keeps what is in flight within few pages
    const uint32_t per = total > (uint64_t)kPutFew * threads ? kPutTrip : 1;
    const uint64_t step = (uint64_t)blocks * threads * per;
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
    if (vl == 4 && per > 1) {  // (uniform)
        for (uint64_t w = (uint64_t)block * threads * kPutTrip + threadIdx.x; w < total; w += step) {
            granule_t held[kPutTrip];
            gbyte* to[kPutTrip];
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q) {
                const gbyte* src;
                to[q] = place(w + q * threads < total ? w + q * threads : w, src);  // (past the end: the thread's first again)
                held[q] = __builtin_nontemporal_load((const g16*)src);
            }
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q) asm volatile("" : "+v"(held[q]));
#pragma unroll
            for (int q = 0; q < kPutTrip; ++q)
                if (w + q * threads < total) __builtin_nontemporal_store(held[q], (g16*)to[q]);
        }
        return;
    }
    for (uint64_t w = (uint64_t)block * threads + threadIdx.x; w < total; w += (uint64_t)blocks * threads) {
        const gbyte* src;
        gbyte* const to = place(w, src);
        copy_granule(to, src, vl);
    }
}

// A launch of few workgroups has as many for every field (blockIdx.y). Of one of many those of the small fields would do nothing, and
// 65,536 workgroups that leave at once take 15 us: it has each field's own number of them, one field's behind the other's.
__device__ __forceinline__ void put_fields(const RowTable* __restrict__ table, const ShortIo& io, uint32_t first_slot, uint32_t n,
                                           uint32_t block, uint32_t blocks) {
    if (blocks) {  // uniform
        put_field(table, io, blockIdx.y, first_slot, n, block, blocks, kWG);
        return;
    }
    const int f = field_of_block(table, n, block, blocks);
    put_field(table, io, f, first_slot, n, block, blocks, kWG);
}

// Workgroups of a gather's largest field, a granule to a thread, from which on threads take four of the large fields and every field has its own
// number of workgroups; later for drawn slots, which each granule draws for itself. us, a granule to a thread / four:
//   row         workgroups   given           drawn            row         workgroups   given           drawn
//   1.8 KB        928        5.5 / 5.0       5.6 / 5.6        1.8 KB       1359         6.7 / 6.1       7.1 / 6.8
//   1.1 KB       1008        4.6 / 4.1       5.0 / 5.1        1.1 KB       1476         5.9 / 5.1       6.1 / 6.1
//   1 KB         1024        3.6 / 3.6       4.2 / 4.5        0.6 KB       1500         6.3 / 5.6       6.4 / 6.7
//   1 KB (odd)   1024        4.2 / 4.0       4.5 / 4.9        1 KB         1546         7.2 / 6.8       7.6 / 7.7
//   1.4 KB       1054        5.3 / 5.3       5.7 / 6.0        0.9 KB       1568         6.2 / 5.7       6.5 / 6.3
//   0.9 KB       1148        5.4 / 5.2       5.5 / 5.9        1.3 KB       1898         5.5 / 4.5       6.0 / 5.7
//   0.6 KB       1152        4.0 / 3.8       4.4 / 4.7        1 KB         2048         5.7 / 4.6       6.1 / 6.1
//   0.4 KB       1216        5.9 / 5.7       6.4 / 6.6        0.9 KB       3136         9.6 / 9.2       9.8 / 10.2
//   0.8 KB       1218        6.3 / 6.0       6.6 / 6.7        1.6 KB       3200         8.3 / 6.4       8.8 / 7.8
//   1.3 KB       1296        4.2 / 3.9       4.7 / 4.9        7.5 KB       7504        19.3 / 14.0     20.4 / 13.9
constexpr uint32_t kGatherFew = 1024, kGatherFewDrawn = 1312;

// A gather of many granules, one field's n rows by workgroup `block` of `blocks`: as put_field, with the rows' slots given or drawn (see gather_body).
template <int kPer, bool kThrough = false>
__device__ __forceinline__ void gather_field(const ShortRows& rows, int f, const int64_t* __restrict__ indices, int64_t count, uint64_t seed,
                                             uint64_t calls, uint32_t block, uint32_t blocks) {
    const uint32_t units = rows.units(f), vl = rows.vl(f), row_bytes = rows.row_bytes(f), stride = rows.stride(f);
    const gbyte* const store = as_global((const uint8_t*)rows.store(f));
    gbyte* const to = as_global(rows.io(f));
    int64_t* const out_indices = rows.first && f == 0 ? reinterpret_cast<int64_t*>(rows.s.at(0)) : nullptr;
    const uint64_t total = rows.granules(f);
    for (uint64_t w = (uint64_t)block * kWG * kPer + threadIdx.x; w < total; w += (uint64_t)blocks * kWG * kPer) {
        uint64_t row[kPer];
        uint32_t unit[kPer];
        int64_t slot[kPer];
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            split_work(w + q * kWG < total ? w + q * kWG : w, units, row[q], unit[q]);  // (past the end: the thread's first again)
            slot[q] = indices ? indices[row[q]] : rng_below(seed, calls, row[q], count);
        }
        bool outside = false;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            outside = outside || (f == 0 && unit[q] == 0 && (slot[q] < 0 || slot[q] >= count));  // (one granule of a row: see gather_body)
            slot[q] = slot[q] < 0 ? 0 : slot[q] >= count ? (count > 0 ? count - 1 : 0) : slot[q];
            if (out_indices && unit[q] == 0) out_indices[row[q]] = slot[q];
        }
        if (outside) atomicOr(rows.r->err, MRB_DERR_INDEX);
        if (kPer > 1) {  // (granules of 16 bytes)
            granule_t held[kPer];
#pragma unroll
            for (int q = 0; q < kPer; ++q)
                held[q] = __builtin_nontemporal_load((const g16*)(store + (uint64_t)slot[q] * stride + granule_offset(unit[q], 4, row_bytes)));
#pragma unroll
            for (int q = 0; q < kPer; ++q) asm volatile("" : "+v"(held[q]));
#pragma unroll
            for (int q = 0; q < kPer; ++q)
                if (w + q * kWG < total) store_granule<kThrough>((g16*)(to + row[q] * row_bytes + granule_offset(unit[q], 4, row_bytes)), held[q]);
        } else {
            const uint32_t off = granule_offset(unit[0], vl, row_bytes);
            copy_granule(to + row[0] * row_bytes + off, store + (uint64_t)slot[0] * stride + off, vl);
        }
    }
}
__device__ __forceinline__ void gather_fields(const ShortRows& rows, const int64_t* __restrict__ indices, int64_t count, uint64_t seed, uint64_t calls,
                                              uint32_t block, bool through) {
    uint32_t blocks;
    const int f = field_of_block(rows.r, rows.n, block, blocks);
    const bool many = rows.vl(f) == 4 && rows.granules(f) > (uint64_t)kPutFew * kWG;
    if (many && through) gather_field<kPutTrip, true>(rows, f, indices, count, seed, calls, block, blocks);
    else if (many) gather_field<kPutTrip>(rows, f, indices, count, seed, calls, block, blocks);
    else gather_field<1>(rows, f, indices, count, seed, calls, block, blocks);
}

// `blocks` of such a launch, and its grid behind (in x) `in_front` other workgroups. (t: the call's table.)
inline dim3 put_grid(const IoTable& t, uint32_t in_front, uint32_t& blocks) {
    uint32_t most = 0, all = 0;
    for (int f = 0; f < t.nfields; ++f) {
        const uint32_t b = put_blocks(t.prefix[f + 1] - t.prefix[f], kWG);
        most = b > most ? b : most;
        all += b;
    }
    blocks = most <= kPutFew ? most : 0;
    return blocks ? dim3(in_front + blocks, (uint32_t)t.nfields) : dim3(in_front + all);
}

hipError_t launch_short_gather(const RowTable* table, const ShortIo& io, const IoTable& t, const int64_t* indices, int64_t count, uint64_t seed,
                               uint64_t calls, int64_t n, uint32_t blocks, bool with_indices, hipStream_t s);
hipError_t launch_short_put(const RowTable* table, const ShortIo& io, const IoTable& t, int64_t first_slot, int64_t n, hipStream_t s);
// (granules: the field's with the most)
hipError_t launch_short_push_one(const RowTable* table, const ShortIo& io, int nfields, float* sum, float* mn, float* maxp, int64_t first_slot,
                                 int depth, float alpha, const float* priority, uint64_t granules, hipStream_t s);
hipError_t launch_short_push_run(const RowTable* table, const ShortIo& io, int nfields, const UpdateArgs& a, uint32_t units, uint64_t granules,
                                 uint32_t threads, hipStream_t s);

}  // namespace mrb
