// What the row kernels of several source files share: the field tables, the copies of a row, the arguments of a sample and
// the steps of its descent (no kernels here).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/mrb.h"
#include "mrb_device.h"

namespace mrb {

constexpr int kWG = 256;          // threads per workgroup of the row and sample kernels
constexpr int kLdsWG = kWG + 64;  // the LDS-top sample kernel: kWG strata and a helper wave

// Per-call table of the fields of a row, passed to kernels by value.
// `store` is the field's place in the buffer - row r of the field at store + r * stride: a [capacity, row_bytes]
// matrix of its own, or a column of the packed rows -, `io` the caller's contiguous [n, row_bytes] matrix
// (source of an append, destination of a gather).
struct IoTable {
    int nfields;
    uint8_t* store[MRB_MAX_FIELDS];
    uint8_t* io[MRB_MAX_FIELDS];
    uint32_t row_bytes[MRB_MAX_FIELDS];
    uint32_t stride[MRB_MAX_FIELDS];    // bytes from one row of the field to the next in `store`: row_bytes when every
                                        // field has an array of its own, the packed row's size when rows are packed
    uint32_t units[MRB_MAX_FIELDS];     // copy granules of a row: row_bytes / 2^vec_log2, rounded up
    uint32_t vec_log2[MRB_MAX_FIELDS];  // copy granule: the largest of 16, 8, 4, 2 and 1 bytes that a row holds
    uint64_t prefix[MRB_MAX_FIELDS + 1];  // running sum of n * units over fields
};

// Row pointers reach the kernels inside by-value tables, where the compiler cannot
// see that they point to global memory; the qualified type makes every row access a
// global_load/global_store rather than a flat one.
using gbyte = __attribute__((address_space(1))) uint8_t;
__device__ __forceinline__ gbyte* as_global(uint8_t* p) { return (gbyte*)p; }
__device__ __forceinline__ const gbyte* as_global(const uint8_t* p) { return (const gbyte*)p; }

// A row of a field is copied in granules of 16 bytes (of 8, 4, 2 or 1 where it has fewer), whatever its size and
// alignment: granule u starts at byte u * 16, the last one where it ends with the row, over bytes the one before it
// has too (both bring the same bytes). A granule may lie at any address; the device's loads and stores take that. A row
// of 147 bytes is then 10 granules rather than 147, one of 111 floats 28 rather than 111. Measured, per call: 250
// prioritized rows of 925 bytes 8.3 -> 4.4 us, 8192 uniform rows of 268 bytes in odd fields 10.5 -> 5.3 us.
__device__ __forceinline__ uint32_t granule_offset(uint32_t unit, uint32_t vl, uint32_t row_bytes) {
    const uint32_t at = unit << vl, last = row_bytes - (1u << vl);
    return at < last ? at : last;
}

using granule_t = __attribute__((ext_vector_type(4))) uint32_t;  // one 16-byte copy granule
// the same, and smaller ones, at any address
using granule16_u = __attribute__((ext_vector_type(4), aligned(1))) uint32_t;
using granule8_u = __attribute__((ext_vector_type(2), aligned(1))) uint32_t;
typedef uint32_t granule4_u __attribute__((aligned(1)));
typedef uint16_t granule2_u __attribute__((aligned(1)));
#define MRB_GLOBAL __attribute__((address_space(1)))

// One granule of 1 << vl bytes. Rows are read once and written once, so both
// sides bypass the caches' retention (non-temporal).
__device__ __forceinline__ void copy_granule(gbyte* dst, const gbyte* src, uint32_t vl) {
    switch (vl) {
        case 4: {
            const granule16_u t = __builtin_nontemporal_load((const MRB_GLOBAL granule16_u*)src);
            __builtin_nontemporal_store(t, (MRB_GLOBAL granule16_u*)dst);
            break;
        }
        case 3: {
            const granule8_u t = __builtin_nontemporal_load((const MRB_GLOBAL granule8_u*)src);
            __builtin_nontemporal_store(t, (MRB_GLOBAL granule8_u*)dst);
            break;
        }
        case 2: *(MRB_GLOBAL granule4_u*)dst = *(const MRB_GLOBAL granule4_u*)src; break;
        case 1: *(MRB_GLOBAL granule2_u*)dst = *(const MRB_GLOBAL granule2_u*)src; break;
        default: *dst = *src; break;
    }
}

// One granule of 1 << vl bytes held between its load and its store. vl may differ from lane to lane (where a wave's
// lanes copy different fields: k_res_push, k_per_sample_lds); every size has its own member so that no value of one
// load is merged with another's (a merge would make the compiler wait for the load right away).
struct AnyGranule {
    granule_t q;
    uint64_t d;
    uint32_t w;
    uint16_t h;
    uint8_t b;
    typedef uint64_t u64_u __attribute__((aligned(1)));
    __device__ __forceinline__ void load(const gbyte* src, uint32_t vl) {
        switch (vl) {
            case 4: q = *(const MRB_GLOBAL granule16_u*)src; break;
            case 3: d = *(const MRB_GLOBAL u64_u*)src; break;
            case 2: w = *(const MRB_GLOBAL granule4_u*)src; break;
            case 1: h = *(const MRB_GLOBAL granule2_u*)src; break;
            default: b = *src; break;
        }
    }
    __device__ __forceinline__ void store(gbyte* dst, uint32_t vl) const {
        switch (vl) {
            case 4: *(MRB_GLOBAL granule16_u*)dst = q; break;
            case 3: *(MRB_GLOBAL u64_u*)dst = d; break;
            case 2: *(MRB_GLOBAL granule4_u*)dst = w; break;
            case 1: *(MRB_GLOBAL granule2_u*)dst = h; break;
            default: *dst = b; break;
        }
    }
};

// A call's fields as the gather looks at them: of a by-value table, or (ShortRows, mrb_short.h) of one in device memory.
struct FullRows {
    const IoTable& t;
    __device__ __forceinline__ uint32_t units(int f) const { return t.units[f]; }
    __device__ __forceinline__ uint32_t vl(int f) const { return t.vec_log2[f]; }
    __device__ __forceinline__ uint32_t row_bytes(int f) const { return t.row_bytes[f]; }
    __device__ __forceinline__ uint32_t stride(int f) const { return t.stride[f]; }
    __device__ __forceinline__ uint8_t* store(int f) const { return t.store[f]; }
    __device__ __forceinline__ uint8_t* io(int f) const { return t.io[f]; }
    __device__ __forceinline__ uint64_t granules(int f) const { return t.prefix[f + 1] - t.prefix[f]; }
};

__device__ __forceinline__ int field_of(const IoTable& t, uint64_t w) {
    int f = 0;
    while (f + 1 < t.nfields && w >= t.prefix[f + 1]) ++f;
    return f;
}

__device__ __forceinline__ void split_work(uint64_t local, uint32_t units, uint64_t& row, uint32_t& unit) {
    if (local <= 0xffffffffull) {
        const uint32_t l32 = (uint32_t)local;
        const uint32_t r = l32 / units;
        row = r;
        unit = l32 - r * units;
    } else {
        row = local / units;
        unit = (uint32_t)(local - row * units);
    }
}

// ---------------------------------------------------------------------------
// Ring append: rows [0, nrows) of each io matrix go to slots
// (first_slot + row) mod capacity. Replaces P.BufferAppend
// (mindspore_rl/core/uniform_replay_buffer.py:82,114) and the row copy of
// PriorityReplayBufferPush (mindspore_rl/core/priority_replay_buffer.py:67-69).
// The host guarantees nrows <= capacity, so no two rows share a slot.
// ---------------------------------------------------------------------------
// src_capacity > 0: the source is itself a ring of that many rows and row r is read from its
// slot (src_first + r) mod src_capacity (buffer-to-buffer copy); 0: the source is contiguous.
struct PutArgs {
    IoTable t;
    int64_t capacity, first_slot, src_capacity, src_first;
    uint32_t blocks;  // workgroups doing this copy when it rides along in another kernel's launch (0: none)
    uint32_t threads; // of each. (From the host: a kernel that asks for its launch's size gets 256 bytes more of arguments,
                      // and a launch of more than 1 KB of them costs the host half a microsecond more than one of less.)
    // first_slot < 0: the buffer's counters live on the device (see Counters below), the rows go to
    // (pushes mod capacity) onwards, and src_first - unused then, the source is never a ring - holds the
    // counters' address
};

// A prioritized buffer's counters as device memory, for callers that record their loop into a HIP
// graph: kernels then take the ring position, the number of stored rows and the generator's call
// counter from here, and a one-thread kernel advances them after each call, so that every replay
// continues where the one before stopped.
// Kernels are told through a negative first slot / row count in their arguments and find the counters
// behind the buffer's error word (one allocation: 16 bytes of flags, then the counters), so that the
// arguments of the ordinary case are what they were.
// ([3] counts the reports of a launch that moves the counters on; [4] is the ring position, pushes mod capacity, kept
// beside the count so that no kernel divides)
constexpr int kCntPushes = 0, kCntSize = 1, kCntCalls = 2, kCntPos = 4, kCntWords = 5;

__device__ __forceinline__ const int64_t* counters_behind(const uint32_t* err) {
    return reinterpret_cast<const int64_t*>(err + 4);
}
// A prioritized buffer's running max lives in the same allocation, kMaxpBehindErr bytes behind the error word: a
// kernel that has its address among its preloaded arguments finds the counters without reading another argument.
constexpr int kMaxpBehindErr = 64;
__device__ __forceinline__ int64_t* counters_before(float* maxp) {
    return reinterpret_cast<int64_t*>(reinterpret_cast<char*>(maxp) - kMaxpBehindErr + 16);
}
__device__ __forceinline__ uint32_t* err_before(float* maxp) {
    return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(maxp) - kMaxpBehindErr);
}
__device__ __forceinline__ int64_t ring_position(const int64_t* counters, int64_t capacity) {
    return counters[kCntPos];
}
// The counters after a push of `pushed` rows (at most `capacity`), stored.
__device__ __forceinline__ void counters_store_advanced(int64_t* counters, int64_t pushes, int64_t size, int64_t pos,
                                                        int64_t pushed, int64_t capacity) {
    counters[kCntPushes] = pushes + pushed;
    size += pushed;
    counters[kCntSize] = size < capacity ? size : capacity;
    pos += pushed;
    counters[kCntPos] = pos < capacity ? pos : pos - capacity;
}

// The generator's call counter for a sample kernel: the argument, or - when the counters live on the device (a
// negative row count tells) and the generator supplies the draws - the device's counter plus the argument (the
// number of the batch among those the call launches one by one).
__device__ __forceinline__ uint64_t generator_calls(const float* uniforms, uint64_t calls, int64_t size, const uint32_t* err) {
    if (uniforms || size >= 0) return calls;
    return (uint64_t)counters_behind(err)[kCntCalls] + calls;
}

// The counters as a wave found them, and what its report returned (see counters_report).
struct CounterTicket {
    int64_t pushes, size, pos;
    uint32_t before;  // reports ahead of this wave's
};
// (atomic loads: vector loads past the compute unit's caches, which wait for nothing but themselves)
__device__ __forceinline__ CounterTicket counters_take(const uint32_t* err) {
    const int64_t* counters = counters_behind(err);
    CounterTicket t;
    t.pushes = __hip_atomic_load(counters + kCntPushes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t.size = __hip_atomic_load(counters + kCntSize, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t.pos = __hip_atomic_load(counters + kCntPos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t.before = 0;
    return t;
}
__device__ __forceinline__ int64_t ticket_position(const CounterTicket& t, int64_t capacity) { return t.pos; }

// A push moves the device-resident counters on in its own last launch. Where that launch is also the one whose
// workgroups read the ring position (`readers` of them: the tree workgroup and the row copy's), every such
// workgroup reports here when it is done, and the last one to report advances the counters: no workgroup waits
// for another, and none can read a position already moved on. readers <= 1: the caller is the only reader left.
// Called by every thread of the workgroup (it contains a barrier); the counters' fourth word counts the reports.
// `known`: the counters as thread 0 took them when the kernel started (nobody changes them before this advance);
// without it thread 0 requests them here, ahead of the barrier and the report.
__device__ __forceinline__ void counters_push_done(uint32_t* err, int64_t pushed, int64_t capacity, uint32_t readers,
                                                   const CounterTicket* known = nullptr) {
    if (pushed <= 0) return;  // uniform over the launch
    CounterTicket t{};
    if (threadIdx.x == 0) t = known ? *known : counters_take(err);
    __syncthreads();  // every wave's reads of the position are behind it
    if (threadIdx.x != 0) return;
    int64_t* counters = reinterpret_cast<int64_t*>(err + 4);
    if (readers > 1) {
        unsigned int* arrived = reinterpret_cast<unsigned int*>(counters + 3);
        if (atomicAdd(arrived, 1u) != readers - 1) return;
        atomicExch(arrived, 0u);
    }
    counters_store_advanced(counters, t.pushes, t.size, t.pos, pushed, capacity);
}

// The same for the one-launch pushes whose tree work is a single wave (k_push_one, k_tree_wg_push,
// k_tree_paths_push), wave by wave and EARLY: what must precede the advance is every wave's READ of the
// counters, not its work. A wave takes the counters (counters_take: loads only), reports as soon as the values
// are there (counters_report: one atomic whose operand depends on the loaded values, so that it cannot be issued
// before they arrive; its result is not awaited here) and goes on with its work; when that is done it looks at
// what the atomic returned (counters_settle) and, if it was the last of the `readers` waves to report, stores the
// advanced counters, computed from the values it took - no load, and no round trip to L2 at the kernel's end.
// All three are called by whole waves; lane 0 acts. readers <= 1: the calling wave is the only reader.
__device__ __forceinline__ void counters_report(CounterTicket& t, uint32_t* err, uint32_t readers, uint32_t lane) {
    if (readers <= 1 || lane != 0) return;
    unsigned int* arrived = reinterpret_cast<unsigned int*>(reinterpret_cast<int64_t*>(err + 4) + 3);
    // (both counters are non-negative: the operand is 1)
    t.before = atomicAdd(arrived, 1u + (unsigned int)((uint64_t)(t.pushes | t.size | t.pos) >> 63));
}
__device__ __forceinline__ void counters_settle(const CounterTicket& t, uint32_t* err, int64_t pushed, int64_t capacity,
                                                uint32_t readers, uint32_t lane) {
    if (lane != 0) return;
    int64_t* counters = reinterpret_cast<int64_t*>(err + 4);
    if (readers > 1) {
        if (t.before != readers - 1) return;
        atomicExch(reinterpret_cast<unsigned int*>(counters + 3), 0u);
    }
    counters_store_advanced(counters, t.pushes, t.size, t.pos, pushed, capacity);
}

// How a workgroup that carries a row copy in another kernel's launch ends. The compiler lays such a kernel out as
// if the tree workgroup's code could follow the copy, and without the explicit wait it makes the tree workgroup
// wait, early on, for loads that only the copy ever issues (its first requests then go out one after the other
// instead of together: a third of a microsecond on a one-workgroup call).
__device__ __forceinline__ void rider_ends() {
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_endpgm();
}

// The copy itself, by workgroup `block` of `nblocks` (grid-stride over the granules). known_first >= 0: the
// first slot, already read from the device's counters by the caller.
__device__ __forceinline__ void rows_put_part(const PutArgs& p, uint32_t block, uint32_t nblocks, int64_t known_first = -1) {
    const IoTable& t = p.t;
    const uint64_t total = t.prefix[t.nfields];
    const uint64_t stride = (uint64_t)nblocks * p.threads;
    const int64_t first_slot = known_first >= 0  ? known_first
                               : p.first_slot >= 0 ? p.first_slot
                                                   : ring_position(reinterpret_cast<const int64_t*>(p.src_first), p.capacity);
    for (uint64_t w = (uint64_t)block * p.threads + threadIdx.x; w < total; w += stride) {
        const int f = field_of(t, w);
        uint64_t row;
        uint32_t unit;
        split_work(w - t.prefix[f], t.units[f], row, unit);
        int64_t slot = first_slot + (int64_t)row;
        if (slot >= p.capacity) slot -= p.capacity;
        uint64_t src_row = row;
        if (p.src_capacity > 0) {
            int64_t q = p.src_first + (int64_t)row;
            if (q >= p.src_capacity) q -= p.src_capacity;
            src_row = (uint64_t)q;
        }
        const uint32_t vl = t.vec_log2[f];
        const uint32_t off = granule_offset(unit, vl, t.row_bytes[f]);
        // (a source that is itself a ring is another buffer's storage, laid out like this one's)
        copy_granule(as_global(t.store[f]) + (uint64_t)slot * t.stride[f] + off,
                     as_global(t.io[f]) + src_row * (p.src_capacity > 0 ? t.stride[f] : t.row_bytes[f]) + off, vl);
    }
}

// Arguments of a PER sample (the wide-row kernel takes what its tree walk needs as plain leading
// parameters instead).
struct SampleArgs {
    const float* sum;       // sum tree, heap order
    const float* uniforms;  // f32[batch] or NULL -> generator
    int64_t batch;
    int depth;              // log2(leaves)
    float beta;
    uint64_t seed, calls;
    int64_t leaves;
    int64_t capacity;
    int64_t size;           // rows stored; negative: read from the device (see Counters)
    const float* mn;        // min tree, heap order
    int64_t* out_idx;
    float* out_w;
    uint32_t* err;
};

__device__ __forceinline__ void sample_flags(const SampleArgs& a, float total, int64_t idx, int64_t size) {
    if (!(total > 0.0f) || total > 3.0e38f) atomicOr(a.err, MRB_DERR_TOTAL);
    if (idx >= size) atomicOr(a.err, MRB_DERR_UNFILLED);
}

// ---------------------------------------------------------------------------
// Wide rows (at least one field of 1 KB or more): k_per_sample_wide (PER sample)
// and k_rows_gather_wide (gather at given / drawn / fixed slots).
//
// A row's fields are of two kinds: "wide" fields, whose rows have at least
// 16 bytes and are copied in 16-byte granules, and "narrow" fields (the
// others: scalars and short vectors), copied byte by byte. The granules
// (bytes) of each kind are numbered consecutively over the fields. `split` workgroups share a row (one unless a
// row has more than 2048 wide granules); workgroup `part` copies wide granules
// [part * share, (part + 1) * share), the row's first workgroup also the
// narrow ones. A workgroup is one "walker" wave and four copy waves:
//   walker   finds the row's slot - for a sample by walking the sum tree with
//            group_request / group_walk (one dependent load per 10 levels; the
//            first group sits under the root, so it is requested together with
//            the total and the uniform draw) - using nothing but kernel
//            arguments preloaded into scalar registers, and publishes it
//            through LDS. Afterwards it copies the narrow fields, computes the
//            importance weight (the two powers in two lanes of one instruction
//            stream) and writes index and weight, off the copy waves' path.
//   copy     meanwhile every copy thread works out where its up to kInF
//            granules lie within a row (field, offset, destination) from the
//            field table, and the first copy wave stages in LDS what the
//            walker needs afterwards (narrow-field table, output pointers,
//            the minimum priority). After the barrier one multiply-add per
//            granule gives the source address; all loads are issued before
//            the first store: a row costs one memory round trip, not one per
//            field.
// Everything read from the kernel-argument segment costs a memory round trip
// of its own when a kernel starts (nothing is cached across launches), which
// is why the walker touches none of it before the barrier and the copy waves
// fetch the table in one round.
// Sampling reads its rows non-temporally so that they do not push the tree
// out of the caches; the gathered batch is stored with ordinary stores (it is
// what the caller reads next).
// ---------------------------------------------------------------------------
struct WideField {  // one table entry, 32 bytes
    const uint8_t* src;  // the field's place in the buffer: row r at src + r * ss
    uint8_t* dst;        // the caller's [batch, row_bytes] matrix
    uint32_t rb;         // row_bytes
    uint32_t first;      // wide field: number of its first granule among the wide ones; narrow: of its first byte
    uint32_t ss;         // bytes from one row to the next in the buffer (row_bytes, or the packed row's size)
    uint32_t pad;
};
struct WidePlan {
    int split;              // workgroups per row
    uint32_t share;         // wide granules per workgroup
    uint32_t wide_items;    // wide granules per row
    uint32_t narrow_items;  // bytes of narrow fields per row
    int nwide, nnarrow;     // fields of each kind
    uint32_t nbatch;        // host side only: batches in the launch
    uint32_t through;       // whether the batch is stored through the L2 (see store_granule)
    WideField f[MRB_MAX_FIELDS];  // the wide fields first, then the narrow ones
};

// What the walker of a sample needs after the descent.
struct SampleTail {
    const float* mn;  // min tree, heap order
    int64_t* out_idx;
    float* out_w;
    uint32_t* err;
    int64_t size;  // rows stored; negative: read from the device (see Counters)
    float beta;
};

constexpr int kCopyWaves = 4;
constexpr int kCopyThreads = 64 * kCopyWaves;
constexpr int kWideWG = 64 + kCopyThreads + 64;  // the walker wave, four copy waves and, for rows with narrow
                                                  // fields, a wave that carries those (launched only then)
constexpr int kMaxInFlight = 8;             // most granules a copy thread holds between its loads and its stores
constexpr int kFastWide = 2;                // wide fields whose table entries are fetched unconditionally, in one round

using g16 = MRB_GLOBAL granule16_u;

// A granule of a batch, or (kThrough) of a large one: stored through the die's L2 into memory at once. What lies changed in the eight
// dies' caches (4 MB each) when a kernel ends is written out then, with nothing else going on; a large batch's stores had better be on
// their way while rows are still being read. The memory's own cache keeps them either way, as it does not behind non-temporal stores
// (220 MB sampled and read 128 us, 124 so, 149 with those). us, L2 / through, by MB of the batch:
//                                       14            16            20             24             32             48             64             220
//   sample, 28 KB rows               9.3 /  9.2    9.7 / 10.0    10.8 / 10.4    12.5 / 11.8    15.0 / 14.3    21.6 / 19.9    26.9 / 24.5    88.0 / 84.0
//   uniform gather, 28 KB            9.0 /  8.9    9.0 /  9.5    10.2 / 10.0    11.6 / 11.2    14.3 / 13.5    19.8 / 18.1    25.2 / 23.1
//   uniform gather, 7.5 KB           8.7 /  8.7    9.4 /  9.3    10.7 / 10.8    12.3 / 12.2    15.3 / 14.5    21.1 / 19.6    26.4 / 25.0
//   uniform gather, 4 KB             7.9 /  8.2    8.5 /  8.6    10.2 / 10.1    11.6 / 11.4    13.8 / 13.2    19.3 / 18.0    24.7 / 22.8
//   uniform gather, 2.4 KB           8.3 /  8.7    9.3 /  9.4    10.9 / 10.7    12.5 / 12.0    15.5 / 15.5
// But a batch is read next, and what the dies' caches (32 MB together) hold of a gather's is found there, so the line of gathers lies where
// about as many readers gain as lose. The call and a reader behind it, us, L2 / through (a product with 64 or 256 columns, a copy into bf16):
//   MB                                                    22              26              34              40              48              64
//   gather, 2.4 KB, f32 x 64                         32.1 / 36.9     31.6 / 37.6     32.8 / 34.4     46.1 / 45.5     49.9 / 48.6     52.2 / 51.5
//   gather, 2.4 KB, bf16 x 256                       38.4 / 42.0     39.3 / 42.7     41.1 / 42.4     46.7 / 48.3     49.6 / 50.7     56.6 / 55.1
//   gather, 4 KB, f32 x 64                           29.5 / 34.0     29.4 / 34.7     36.9 / 38.2     38.0 / 38.9     40.1 / 40.8     45.8 / 45.5
//   gather, 7.5 KB, f32 x 64                         33.7 / 37.8     33.5 / 39.0     40.0 / 43.9     41.9 / 43.8     44.6 / 45.8     63.0 / 62.4
//   gather, 1 KB, bf16 x 256                         29.1 / 32.2     30.8 / 33.0     35.3 / 37.6     37.4 / 38.6     44.6 / 45.0     50.7 / 49.8
//   gather, 28 KB, u8 to bf16                        51.9 / 51.0     59.2 / 58.4     73.5 / 72.6     85.4 / 83.8    100.4 / 98.6    130.3 / 128.0
//   sample, 28 KB, u8 to bf16                        52.4 / 51.0     59.1 / 57.9     74.1 / 73.1     87.5 / 85.9    102.0 / 100.6   132.2 / 129.7
//   sample, 28 KB, bf16 x 256                        66.3 / 66.1     67.3 / 67.4     75.0 / 74.9     79.0 / 77.6     82.4 / 81.0     96.6 / 94.6
//   sample, 1 KB (k_per_sample_lds_large), f32 x 64  35.3 / 34.2     30.0 / 29.5     50.9 / 49.9     52.8 / 51.9     47.4 / 45.7     53.0 / 51.0
// (A sample with a mere maximum of each row behind it, 24 MB 26.7 / 27.3, 32 MB 28.5 / 28.7, 48 MB 35.3 / 33.9.)
// And where a wave's store ends in the middle of 64 bytes, the rest of them comes later, from another wave: what is more than
// the memory's cache (256 MB, of which the batch's readers and the rows take their part) is then written to memory in pieces. us, L2 / through:
//                                                   128 MB          180 MB          256 MB           360 MB          460 MB          920 MB
//   sample, 28,224 bytes                                                                            136 / 129       169 / 161       332 / 313
//   sample, 28,192                                                                                  142 / 139       171 / 194       334 / 397
//   sample, 40,000 (two workgroups, 20,000 each)                                                    155 / 152       192 / 205       385 / 415
//   sample, 28,225, and a copy behind it            93 /  92       144 / 143       224 / 235
//   gather, 7488 (k_short_gather_many)                                                              136 / 129       174 / 165       350 / 333
//   gather, 7500                                                                                    153 / 146       187 / 210       385 / 438
//   gather, 1500, and a copy behind it              85 /  83       136 / 133       217 / 226
//   gather, 2432 (k_rows_gather_rows)                                                               137 / 128       176 / 165       346 / 323
//   gather, 2400                                                                                    153 / 145       183 / 194       358 / 395
// So such batches are stored so up to 160 MB, others without an end (measured up to 1.8 GB: sample, 28,224 bytes 690 / 659).
// Not stored so is what k_rows_gather, k_short_gather, k_per_sample_rows, k_per_sample_lds and k_per_sample_lanes copy (the last one's lanes store
// pieces of many rows at once and are slower so at every size: 7.5 KB 32.2 / 35.8 with 64 MB).
template <bool kThrough>
__device__ __forceinline__ void store_granule(g16* to, granule_t v) {
    if (kThrough) store_through((void*)to, v);
    else *to = v;
}
constexpr uint64_t kThroughSample = 20ull << 20, kThroughGather = 40ull << 20;  // bytes of a batch from which on it is stored so
constexpr uint64_t kThroughBroken = 160ull << 20;                                // and up to which, where waves' stores end within 64 bytes
inline uint64_t batch_bytes(const IoTable& t) {
    uint64_t bytes = 0;
    for (int f = 0; f < t.nfields; ++f) bytes += (t.prefix[f + 1] - t.prefix[f]) << t.vec_log2[f];
    return bytes;
}
// Whether a wave's stores are whole pieces of 64 bytes: of the rows, or parts of rows, that a plan's workgroups or waves write, or of a field
// whose granules are numbered over all rows.
inline bool whole_pieces(const WidePlan& plan) {
    bool whole = plan.split == 1 || plan.share % 4 == 0;
    for (int q = 0; q < plan.nwide; ++q) whole = whole && (((uint64_t)plan.f[q].dst | plan.f[q].rb) & 63) == 0;
    return whole;
}
inline bool whole_pieces(const IoTable& t, int f) { return ((uint64_t)t.io[f] & 63) == 0 && t.row_bytes[f] % 16 == 0; }
inline bool stores_through(uint64_t bytes, uint64_t from, bool whole) { return bytes > from && (whole || bytes <= kThroughBroken); }

constexpr int kNarrowInF = 2;  // narrow bytes a thread of the first copy wave holds beside its wide granules

__device__ __forceinline__ uint32_t lane_u32(uint32_t x, int src_lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, src_lane);
}
__device__ __forceinline__ uint64_t lane_u64(uint64_t x, int src_lane) {
    return ((uint64_t)lane_u32((uint32_t)(x >> 32), src_lane) << 32) | lane_u32((uint32_t)x, src_lane);
}

// The narrow fields of a row, copied byte by byte by a wave of their own in the row's first
// workgroup (the sixth; a copy wave that also carried them would hold its wide stores back until
// the narrow loads have arrived: 0.06 us per launch of 512 Atari-shaped rows): lane l takes bytes l,
// l + 64, ... of the narrow fields' bytes, numbered consecutively over the fields. Narrow fields are small (scalars such as action, reward, done); byte
// granularity keeps their copy free of branches on a granule size.
struct NarrowWork {
    const gbyte* base[kNarrowInF];
    gbyte* dst[kNarrowInF];
    uint32_t rb[kNarrowInF];  // the byte's field: bytes from one row to the next in the buffer
    uint32_t live;  // bit j: position j holds a byte
    // the table entry of field `lane` (lanes 0 .. MRB_MAX_FIELDS - 1), kept for bytes past the first ones
    uint64_t e_src, e_dst;
    uint32_t e_rb, e_first, e_ss;

    // Each lane finds the fields of its bytes from the table's entries. Up to kNarrowFast narrow fields (the
    // usual few scalars) are read with wave-uniform indices - scalar loads, issued together, from lines of the
    // kernel-argument segment that the copy waves' own reads bring into the scalar cache. More fields than that:
    // lane q fetches entry q with one vector load (a round trip of its own through memory, which holds back the
    // workgroup's barrier when nothing else, such as a tree descent, takes as long) and the entries are read from
    // the lanes. Rows with more than 64 * kNarrowInF narrow bytes keep the per-lane copy for store().
    static constexpr int kNarrowFast = 4;
    __device__ __forceinline__ void take(const WidePlan& plan, int64_t k, uint32_t lane, uint64_t src_q, uint64_t dst_q,
                                         uint32_t rb_q, uint32_t first_q, uint32_t ss_q) {
#pragma unroll
        for (int j = 0; j < kNarrowInF; ++j) {
            const uint32_t rel = ((live >> j) & 1u ? lane + 64 * j : 0u) - first_q;  // wraps for bytes of earlier fields
            if (rel < rb_q) {
                base[j] = (const gbyte*)(src_q + rel);
                dst[j] = (gbyte*)(dst_q + rel);
                rb[j] = ss_q;
            }
        }
    }
    __device__ __forceinline__ void prepare(const WidePlan& plan, int64_t k, uint32_t lane) {
        live = 0;
#pragma unroll
        for (int j = 0; j < kNarrowInF; ++j) {
            base[j] = nullptr;
            dst[j] = nullptr;
            rb[j] = 0;
            if (lane + 64 * j < plan.narrow_items) live |= 1u << j;
        }
        e_src = e_dst = 0;
        e_rb = e_first = e_ss = 0;
        if (plan.nnarrow <= kNarrowFast && plan.narrow_items <= 64u * kNarrowInF) {  // wave-uniform
            WideField e[kNarrowFast];
#pragma unroll
            for (int i = 0; i < kNarrowFast; ++i) e[i] = plan.f[plan.nwide + (i < plan.nnarrow ? i : 0)];
#pragma unroll
            for (int i = 0; i < kNarrowFast; ++i)
                if (i < plan.nnarrow)
                    take(plan, k, lane, (uint64_t)e[i].src, (uint64_t)e[i].dst + (uint64_t)k * e[i].rb, e[i].rb, e[i].first, e[i].ss);
            return;
        }
        const WideField e = plan.f[lane < MRB_MAX_FIELDS ? lane : 0];
        e_src = (uint64_t)e.src;
        e_dst = (uint64_t)e.dst + (uint64_t)k * e.rb;
        e_rb = e.rb;
        e_first = e.first;
        e_ss = e.ss;
        for (int q = plan.nwide; q < plan.nwide + plan.nnarrow; ++q)
            take(plan, k, lane, lane_u64(e_src, q), lane_u64(e_dst, q), lane_u32(e_rb, q), lane_u32(e_first, q), lane_u32(e_ss, q));
    }
    __device__ __forceinline__ void load(uint32_t slot, uint8_t (&held)[kNarrowInF]) const {
#pragma unroll
        for (int j = 0; j < kNarrowInF; ++j) held[j] = *(base[j] + (uint64_t)slot * rb[j]);
    }
    __device__ __forceinline__ void store(uint32_t slot, const uint8_t (&held)[kNarrowInF], const WidePlan& plan, uint32_t lane) const {
#pragma unroll
        for (int j = 0; j < kNarrowInF; ++j)
            if (live & (1u << j)) *dst[j] = held[j];
        if (plan.narrow_items > 64u * kNarrowInF) {  // wave-uniform; rows with many narrow bytes
            for (int q = plan.nwide; q < plan.nwide + plan.nnarrow; ++q) {
                const uint64_t src_q = lane_u64(e_src, q) + (uint64_t)slot * lane_u32(e_ss, q), dst_q = lane_u64(e_dst, q);
                const uint32_t rb_q = lane_u32(e_rb, q), first_q = lane_u32(e_first, q);
                // bytes of this field numbered 64 * kNarrowInF or more among the narrow bytes
                uint32_t rel = (first_q >= 64u * kNarrowInF ? 0u : 64u * kNarrowInF - first_q) + lane;
                for (; rel < rb_q; rel += 64) *((gbyte*)dst_q + rel) = *((const gbyte*)src_q + rel);
            }
        }
    }
};

// Copy thread `tid` (0 .. kCopyThreads - 1) of workgroup `part` of row k: up to kInF wide granules.
// A thread without a granule in some position re-reads the workgroup's first granule (a valid
// address) and skips the store, so that the loads are unconditional and all in flight together.
// kOneWide: the row has a single wide field (e.g. an image observation beside a few scalars); all
// addresses are then a wave-uniform row base plus a 32-bit offset, which costs a tenth of the
// general path's address arithmetic - work that would otherwise compete with the walker for
// the SIMD's issue slots.
// kThreads: the threads that share a workgroup's granules (the four copy waves; one wave in k_per_sample_rows).
template <int kInF, bool kOneWide, int kThreads = kCopyThreads>
struct CopyWork {
    const gbyte* base[kOneWide ? 1 : kInF];  // general: field storage + offset of the granule within a row
    g16* dst[kOneWide ? 1 : kInF];
    uint32_t rb[kOneWide ? 1 : kInF];        // general: bytes from one row to the next in the buffer
    uint32_t off[kOneWide ? kInF : 1];       // one wide field: byte offset of the granule within a row
    const uint8_t* src0;                     // one wide field: storage, destination row, storage row stride (wave-uniform)
    uint8_t* dst0;
    uint32_t rb0;
    uint32_t live;  // bit j: position j holds a granule of this workgroup

    __device__ __forceinline__ void prepare(const WidePlan& plan, int64_t k, uint32_t part, uint32_t tid) {
        const uint32_t lo = part * plan.share;
        const uint32_t hi = min(plan.wide_items, lo + plan.share);
        uint32_t it[kInF];
        live = 0;
#pragma unroll
        for (int j = 0; j < kInF; ++j) {
            it[j] = lo + j * kThreads + tid;
            if (it[j] < hi) live |= 1u << j;
            else it[j] = lo;
        }
        if (lo >= hi || tid >= (uint32_t)kThreads) live = 0;  // (a wave past the copy waves carries narrow fields only)
        if (kOneWide) {
            const WideField e = plan.f[0];
            src0 = e.src;
            rb0 = e.ss;
            dst0 = e.dst + (uint64_t)k * e.rb;
#pragma unroll
            for (int j = 0; j < kInF; ++j) off[j] = granule_offset(it[j], 4, e.rb);
            return;
        }
#pragma unroll
        for (int j = 0; j < (kOneWide ? 1 : kInF); ++j) {
            base[j] = nullptr;
            dst[j] = nullptr;
            rb[j] = 0;
        }
        auto take = [&](int q) {
            const WideField e = plan.f[q];
            const uint32_t units = q < plan.nwide ? (e.rb + 15) >> 4 : 0u;
            const gbyte* s = as_global(e.src);
            gbyte* d = as_global(e.dst) + (uint64_t)k * e.rb;
#pragma unroll
            for (int j = 0; j < (kOneWide ? 1 : kInF); ++j) {
                const uint32_t rel = it[j] - e.first;  // wraps for granules of earlier fields
                if (rel < units) {
                    const uint32_t at = granule_offset(rel, 4, e.rb);
                    base[j] = s + at;
                    dst[j] = (g16*)(d + at);
                    rb[j] = e.ss;
                }
            }
        };
        // the first entries unconditionally: their (wave-uniform) loads go out together at once
#pragma unroll
        for (int q = 0; q < kFastWide; ++q) take(q);
        for (int q = kFastWide; q < plan.nwide; ++q) take(q);
    }

    // `narrow`: this thread carries narrow bytes (the wave after the copy waves, in the row's first workgroup)
    __device__ __forceinline__ void run(uint32_t slot, const WidePlan& plan, bool narrow, const NarrowWork& nw, uint32_t lane) const {
        uint8_t nheld[kNarrowInF];
        granule_t held[kInF];
        if (narrow) nw.load(slot, nheld);
        if (live) {
            if (kOneWide) {
                const gbyte* row = as_global(src0) + (uint64_t)slot * rb0;  // wave-uniform
#pragma unroll
                for (int j = 0; j < kInF; ++j) held[j] = __builtin_nontemporal_load((const g16*)(row + off[j]));
            } else {
#pragma unroll
                for (int j = 0; j < kInF; ++j)
                    held[j] = __builtin_nontemporal_load((const g16*)(base[j < (kOneWide ? 1 : kInF) ? j : 0] + (uint64_t)slot * rb[j < (kOneWide ? 1 : kInF) ? j : 0]));
            }
            // every load is issued before the first store (the compiler would otherwise move a load
            // next to its conditional store, behind the other stores' waits)
#pragma unroll
            for (int j = 0; j < kInF; ++j) asm volatile("" : "+v"(held[j]));
            auto store = [&](auto through) {
#pragma unroll
                for (int j = 0; j < kInF; ++j)
                    if (live & (1u << j)) {
                        if (kOneWide) store_granule<decltype(through)::value>((g16*)(as_global(dst0) + off[j]), held[j]);
                        else store_granule<decltype(through)::value>(dst[j < (kOneWide ? 1 : kInF) ? j : 0], held[j]);
                    }
            };
            if (plan.through) store(std::true_type{});  // uniform
            else store(std::false_type{});
        }
        if (narrow) nw.store(slot, nheld, plan, lane);
    }
};

// Three levels of the descent from the eight nodes three levels under a node (lo: the first four, hi: the last
// four): which of them the mass falls into, what is left of the mass inside it, and its value. The sums of the
// two levels between are the single additions the tree was built with.
__device__ __forceinline__ uint32_t walk8(const float4 lo, const float4 hi, float& mass, float& picked) {
    const float a0 = lo.x + lo.y, a1 = lo.z + lo.w, a2 = hi.x + hi.y;
    const float b0 = a0 + a1;
    uint32_t p = 0;
    if (!(mass <= b0)) {
        mass -= b0;
        p = 4;
    }
    const float left1 = p ? a2 : a0;
    if (!(mass <= left1)) {
        mass -= left1;
        p += 2;
    }
    const float n0 = p == 0 ? lo.x : p == 2 ? lo.z : p == 4 ? hi.x : hi.z;
    const float n1 = p == 0 ? lo.y : p == 2 ? lo.w : p == 4 ? hi.y : hi.w;
    if (!(mass <= n0)) {
        mass -= n0;
        p += 1;
        picked = n1;
    } else {
        picked = n0;
    }
    return p;
}

// Two levels, and one, of the same descent.
__device__ __forceinline__ uint32_t walk4(const float4 v, float& mass, float& picked) {
    const float left = v.x + v.y;
    uint32_t p = 0;
    if (!(mass <= left)) {
        mass -= left;
        p = 2;
    }
    const float n0 = p ? v.z : v.x, n1 = p ? v.w : v.y;
    if (!(mass <= n0)) {
        mass -= n0;
        p += 1;
        picked = n1;
    } else {
        picked = n0;
    }
    return p;
}
__device__ __forceinline__ uint32_t walk2(const float2 pair, float& mass, float& picked) {
    if (mass <= pair.x) {
        picked = pair.x;
        return 0;
    }
    mass -= pair.x;
    picked = pair.y;
    return 1;
}

// One dependent load of the thread-per-stratum descent: the 2^g descendants of `node` g levels down (g <= 5: at most
// one cache line), the levels between rebuilt with the additions the tree was built with. Returns the node the
// mass falls into, g levels down; `mass` becomes what is left of it inside that node, `picked` the node's value.
__device__ __forceinline__ uint32_t descend_group(const float* __restrict__ sum, uint32_t node, int g, float& mass, float& picked) {
    if (g == 5) {
        const f32x4* src = reinterpret_cast<const f32x4*>(sum + ((uint64_t)node << 5));
        const f32x4 t0 = src[0], t1 = src[1], t2 = src[2], t3 = src[3], t4 = src[4], t5 = src[5], t6 = src[6], t7 = src[7];
        const f32x16 lo = __builtin_shufflevector(__builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7),
                                                  __builtin_shufflevector(t2, t3, 0, 1, 2, 3, 4, 5, 6, 7), 0, 1,
                                                  2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
        const f32x16 hi = __builtin_shufflevector(__builtin_shufflevector(t4, t5, 0, 1, 2, 3, 4, 5, 6, 7),
                                                  __builtin_shufflevector(t6, t7, 0, 1, 2, 3, 4, 5, 6, 7), 0, 1,
                                                  2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
        node = (node << 5) + walk32(lo, hi, mass, picked);
    } else if (g == 4) {
        const f32x4* src = reinterpret_cast<const f32x4*>(sum + ((uint64_t)node << 4));
        const f32x4 t0 = src[0], t1 = src[1], t2 = src[2], t3 = src[3];
        const f32x16 v = __builtin_shufflevector(__builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7),
                                                 __builtin_shufflevector(t2, t3, 0, 1, 2, 3, 4, 5, 6, 7), 0, 1,
                                                 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
        node = (node << 4) + walk16(v, mass, picked);
    } else if (g == 3) {
        const float4* src = reinterpret_cast<const float4*>(sum + ((uint64_t)node << 3));
        const float4 lo = src[0], hi = src[1];
        node = (node << 3) + walk8(lo, hi, mass, picked);
    } else if (g == 2) {
        const float4 v = *reinterpret_cast<const float4*>(sum + ((uint64_t)node << 2));
        const float left = v.x + v.y;
        uint32_t p = 0;
        if (!(mass <= left)) {
            mass -= left;
            p = 2;
        }
        const float n0 = p ? v.z : v.x, n1 = p ? v.w : v.y;
        if (!(mass <= n0)) {
            mass -= n0;
            p += 1;
            picked = n1;
        } else {
            picked = n0;
        }
        node = (node << 2) + p;
    } else {
        const float2 pair = *reinterpret_cast<const float2*>(sum + 2 * (uint64_t)node);
        if (mass <= pair.x) {
            node = 2 * node;
            picked = pair.x;
        } else {
            mass -= pair.x;
            node = 2 * node + 1;
            picked = pair.y;
        }
    }
    return node;
}

constexpr int kLdsOwn = 4;  // leading fields whose row is one granule: every thread copies its own stratum's

}  // namespace mrb
