// libmrb.so — C ABI (include/mrb.h) over the HIP kernels in mrb_kernels.h.
// Host side: handle registry, ring/tree bookkeeping, argument checks, launches.
// Nothing in this file computes a result on the CPU; without a HIP device every
// entry point that touches a buffer fails with MRB_EHIP.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "mrb_kernels.h"
#include "mrb_launch.h"
#include "mrb_meet.h"
#include "mrb_push_many.h"
#include "mrb_range.h"
#include "mrb_range_one.h"
#include "mrb_returns.h"
#include "mrb_samples.h"
#include "mrb_short.h"
#include "mrb_silent.h"
#include "../../include/mrb_more.h"

namespace {

using namespace mrb;

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIP_TRY(expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) return fail(MRB_EHIP, "%s: %s", #expr, hipGetErrorString(e_));    \
    } while (0)

#define LAUNCH_CHECK(name)                                                                     \
    do {                                                                                       \
        hipError_t e_ = hipGetLastError();                                                     \
        if (e_ != hipSuccess) return fail(MRB_EHIP, "launch %s: %s", name, hipGetErrorString(e_)); \
    } while (0)

// Page-locked memory that host rows pass through (mrb_stage): four segments taken in turn.
constexpr int kStageSegments = 4;
constexpr int64_t kStageSegment = 512 << 10;
struct Stage {
    char* memory = nullptr;
    int segment = 0;   // the one in use,
    int64_t at = 0;    // and its first free byte
    hipStream_t stream = nullptr;  // whose work reads it (a call on another stream goes on to the next segment)
    hipEvent_t left[kStageSegments] = {};    // recorded on the stream when a segment was left
    bool was_left[kStageSegments] = {};
    ~Stage() {
        for (auto e : left)
            if (e) (void)hipEventDestroy(e);
        if (memory) (void)hipHostFree(memory);
    }
};

// Row storage. By default a structure of arrays, field i = [capacity, bytes_i] (reference layout:
// mindspore_rl/core/uniform_replay_buffer.py:26-47). With the library option "packed_rows" narrow rows are kept
// packed instead: one [capacity, row_stride] allocation, field i at byte offset_i of every row (each field
// aligned as its size allows), so that a sampled row's fields share cache lines instead of costing one
// 128-byte line per field. Either way row r of field i starts at data[i] + r * stride[i].
struct RowStore {
    int64_t capacity = 0;
    int nfields = 0;
    int64_t bytes[MRB_MAX_FIELDS] = {};
    int64_t stride[MRB_MAX_FIELDS] = {};
    uint8_t* data[MRB_MAX_FIELDS] = {};
    uint8_t* packed_base = nullptr;  // packed rows: the one allocation (data[i] point into it)
    uint32_t align_log2[MRB_MAX_FIELDS] = {};  // log2 of what a row's size is a multiple of, at most 16: the alignment asked
                                              // of the caller's matrices, and a field's in a packed row
    uint32_t vec_log2[MRB_MAX_FIELDS] = {};    // copy granule and granules of a row (see granule_offset)
    uint32_t units[MRB_MAX_FIELDS] = {};
    int64_t row_split = 0;  // option "row_split": least number of workgroups per row in the wide-row kernel (0 = auto)
    int64_t row_wave = 0;   // option "row_wave": the wave-per-row sample kernel, 0 = for launches of many rows, 1 = whenever
                            // the rows fit it, 2 = never
    Stage stage;
    RowTable* table = nullptr;  // on the device: what launches with short arguments find there

    ~RowStore() {
        if (table) (void)hipFree(table);
        if (packed_base) {
            (void)hipFree(packed_base);
            return;
        }
        for (int i = 0; i < nfields; ++i)
            if (data[i]) (void)hipFree(data[i]);
    }
};

// Library-wide default of the option "packed_rows" (mrb_set_option with handle 0): buffers created afterwards
// keep their rows packed when a packed row takes at most this many bytes; 0 = every field an array of its own.
std::atomic<int64_t> g_packed_rows{0};

// What a buffer's launches with short arguments find on the device.
RowTable row_table(const RowStore& r) {
    RowTable t{};
    t.t.nfields = r.nfields;
    for (int i = 0; i < r.nfields; ++i) {
        t.t.store[i] = r.data[i];
        t.t.row_bytes[i] = (uint32_t)r.bytes[i];
        t.t.stride[i] = (uint32_t)r.stride[i];
        t.t.units[i] = r.units[i];
        t.t.vec_log2[i] = r.vec_log2[i];
        t.t.prefix[i + 1] = t.t.prefix[i] + r.units[i];
    }
    t.capacity = r.capacity;
    return t;
}

// A call's matrices as kernels with short arguments take them; false where these cannot say where they are.
bool short_io(const void* const* at, int n, ShortIo& io) {
    if (n > kShortPointers) return false;
    io.base = reinterpret_cast<uint64_t>(at[0]);
    uint64_t any = 1ull << 12;
    for (int i = 1; i < n; ++i) any |= reinterpret_cast<uint64_t>(at[i]) - io.base;
    io.shift = (uint32_t)__builtin_ctzll(any);
    for (int i = 1; i < n; ++i) {
        const int64_t away = static_cast<int64_t>(reinterpret_cast<uint64_t>(at[i]) - io.base) >> io.shift;
        if (away != (int32_t)away) return false;
        io.away[i - 1] = (int32_t)away;
    }
    return true;
}
bool short_io(const IoTable& t, ShortIo& io) { return short_io(reinterpret_cast<const void* const*>(t.io), t.nfields, io); }
// The same with one or two matrices in front.
bool short_io(const void* first, const void* second, const IoTable& t, ShortIo& io) {
    const void* at[MRB_MAX_FIELDS + 2];
    int n = 0;
    at[n++] = first;
    if (second) at[n++] = second;
    for (int i = 0; i < t.nfields; ++i) at[n++] = t.io[i];
    return short_io(at, n, io);
}

// `flags`: `behind` zeroed bytes behind the table, in one allocation with it and filled by the copy that fills it.
int rows_alloc(RowStore& r, int64_t capacity, int nfields, const int64_t* field_bytes, size_t behind, uint32_t** flags) {
    if (capacity <= 0 || capacity > (1ll << 30)) return fail(MRB_EINVAL, "capacity %lld outside [1, 2^30]", (long long)capacity);
    if (nfields <= 0 || nfields > MRB_MAX_FIELDS) return fail(MRB_EINVAL, "nfields %d outside [1, %d]", nfields, MRB_MAX_FIELDS);
    if (!field_bytes) return fail(MRB_EINVAL, "field_bytes is NULL");
    for (int i = 0; i < nfields; ++i)
        if (field_bytes[i] <= 0 || field_bytes[i] > (1ll << 30))
            return fail(MRB_EINVAL, "field_bytes[%d] = %lld outside [1, 2^30]", i, (long long)field_bytes[i]);
    r.capacity = capacity;
    int64_t offset[MRB_MAX_FIELDS], end = 0, widest = 1;
    for (int i = 0; i < nfields; ++i) {
        r.bytes[i] = field_bytes[i];
        uint32_t vl = 4;
        while (vl > 0 && (field_bytes[i] & ((1ll << vl) - 1))) --vl;
        r.align_log2[i] = vl;
        uint32_t copy = 4;
        while ((1ll << copy) > field_bytes[i]) --copy;
        r.vec_log2[i] = copy;
        r.units[i] = (uint32_t)((field_bytes[i] + (1ll << copy) - 1) >> copy);
        // where the field would lie in a packed row: at the next multiple of its own alignment
        const int64_t g = 1ll << vl;
        offset[i] = (end + g - 1) / g * g;
        end = offset[i] + field_bytes[i];
        if (g > widest) widest = g;
    }
    const int64_t packed_row = (end + widest - 1) / widest * widest;  // rows start at multiples of the widest granule
    if (nfields > 1 && packed_row <= g_packed_rows.load()) {
        const size_t total = (size_t)capacity * (size_t)packed_row;
        HIP_TRY(hipMalloc(reinterpret_cast<void**>(&r.packed_base), total));
        HIP_TRY(hipMemset(r.packed_base, 0, total));
        for (int i = 0; i < nfields; ++i) {
            r.data[i] = r.packed_base + offset[i];
            r.stride[i] = packed_row;
        }
        r.nfields = nfields;
    } else {
        for (int i = 0; i < nfields; ++i) {
            const size_t total = (size_t)capacity * (size_t)field_bytes[i];
            HIP_TRY(hipMalloc(reinterpret_cast<void**>(&r.data[i]), total));
            r.nfields = i + 1;  // so the destructor frees what exists
            r.stride[i] = field_bytes[i];
            HIP_TRY(hipMemset(r.data[i], 0, total));
        }
    }
    constexpr size_t kTableBytes = (sizeof(RowTable) + 255) / 256 * 256;
    std::vector<char> fill(kTableBytes + behind, 0);
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&r.table), fill.size()));
    *flags = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(r.table) + kTableBytes);
    RowTable table = row_table(r);
    table.err = *flags;
    memcpy(fill.data(), &table, sizeof(table));
    HIP_TRY(hipMemcpy(r.table, fill.data(), fill.size(), hipMemcpyHostToDevice));
    return MRB_OK;
}

// Builds the per-call field table. `io` pointers must be aligned as each field's row size allows.
int make_table(const RowStore& r, const void* const* io, int64_t n, IoTable& t) {
    if (!io) return fail(MRB_EINVAL, "field pointer array is NULL");
    t.nfields = r.nfields;
    t.prefix[0] = 0;
    for (int i = 0; i < r.nfields; ++i) {
        if (!io[i]) return fail(MRB_EINVAL, "field %d pointer is NULL", i);
        if (reinterpret_cast<uintptr_t>(io[i]) & ((1u << r.align_log2[i]) - 1))
            return fail(MRB_EINVAL, "field %d pointer %p is not %u-byte aligned", i, io[i], 1u << r.align_log2[i]);
        t.store[i] = r.data[i];
        t.io[i] = const_cast<uint8_t*>(static_cast<const uint8_t*>(io[i]));
        t.row_bytes[i] = (uint32_t)r.bytes[i];
        t.stride[i] = (uint32_t)r.stride[i];
        t.units[i] = r.units[i];
        t.vec_log2[i] = r.vec_log2[i];
        t.prefix[i + 1] = t.prefix[i] + (uint64_t)n * r.units[i];
    }
    return MRB_OK;
}

uint32_t grid_for(uint64_t work, uint32_t per_thread = 1) {
    uint64_t g = (work + (uint64_t)kWG * per_thread - 1) / ((uint64_t)kWG * per_thread);
    if (g < 1) g = 1;
    if (g > 16384) g = 16384;
    return (uint32_t)g;
}

// One thread per entry, no grid-stride loop (n < 2^32, so the grid fits).
uint32_t grid_exact(uint64_t n) { return (uint32_t)((n + kWG - 1) / kWG); }

// Describes the append of rows [skip, skip + n) of the caller's matrices at ring position first_slot.
int put_args(const RowStore& r, const void* const* src, int64_t skip, int64_t n, int64_t first_slot, PutArgs& p) {
    const void* shifted[MRB_MAX_FIELDS];
    if (!src) return fail(MRB_EINVAL, "field pointer array is NULL");
    for (int i = 0; i < r.nfields; ++i) {
        if (!src[i]) return fail(MRB_EINVAL, "field %d pointer is NULL", i);
        shifted[i] = static_cast<const uint8_t*>(src[i]) + skip * r.bytes[i];
    }
    int rc = make_table(r, shifted, n, p.t);
    if (rc) return rc;
    p.capacity = r.capacity;
    p.first_slot = first_slot;
    p.src_capacity = 0;
    p.src_first = 0;
    p.blocks = grid_for(p.t.prefix[p.t.nfields]);
    p.threads = kWG;
    return MRB_OK;
}

// Granules of the field that has the most.
uint64_t most_granules(const IoTable& t) {
    uint64_t most = 0;
    for (int f = 0; f < t.nfields; ++f) most = std::max<uint64_t>(most, t.prefix[f + 1] - t.prefix[f]);
    return most;
}

int rows_put(const RowStore& r, const void* const* src, int64_t skip, int64_t n, int64_t first_slot, hipStream_t s) {
    PutArgs p{};
    int rc = put_args(r, src, skip, n, first_slot, p);
    if (rc) return rc;
    if (ShortIo io{}; short_io(p.t, io)) {
        const hipError_t e = launch_short_put(r.table, io, p.t, first_slot, n, s);
        return e == hipSuccess ? MRB_OK : fail(MRB_EHIP, "launch k_short_put: %s", hipGetErrorString(e));
    }
    launch_kernel(k_rows_put, dim3(p.blocks), dim3(kWG), 0, s, p);
    LAUNCH_CHECK("k_rows_put");
    return MRB_OK;
}

int64_t widest_field(const RowStore& r) {
    int64_t m = 0;
    for (int i = 0; i < r.nfields; ++i)
        if (r.bytes[i] > m) m = r.bytes[i];
    return m;
}

// Describes n rows of `r` for the wide-row kernels: one workgroup per row unless a row holds more than
// kMaxInFlight * kCopyThreads (2048) wide granules, or the buffer's "row_split" option asks for more.
// Returns the number of granules a copy thread holds (2 or 8) or 0 on error.
int wide_plan(const RowStore& r, const IoTable& t, int64_t n, WidePlan& plan, dim3& grid) {
    const uint32_t nbatch = plan.nbatch;
    plan = WidePlan{};
    plan.nbatch = nbatch;
    for (int i = 0; i < r.nfields; ++i) plan.nwide += r.vec_log2[i] == 4;
    plan.nnarrow = r.nfields - plan.nwide;
    int w = 0, m = plan.nwide;
    for (int i = 0; i < r.nfields; ++i) {
        const bool wide = r.vec_log2[i] == 4;
        const int q = wide ? w++ : m++;
        plan.f[q].src = t.store[i];
        plan.f[q].dst = t.io[i];
        plan.f[q].rb = t.row_bytes[i];
        plan.f[q].ss = t.stride[i];
        uint32_t& items = wide ? plan.wide_items : plan.narrow_items;
        plan.f[q].first = items;
        items += wide ? r.units[i] : t.row_bytes[i];
    }
    const uint32_t per_wg = (uint32_t)kMaxInFlight * kCopyThreads;
    uint32_t split = (plan.wide_items + per_wg - 1) / per_wg;
    if (r.row_split > (int64_t)split) split = (uint32_t)r.row_split;
    if (split < 1) split = 1;
    plan.split = (int)split;
    plan.share = (plan.wide_items + split - 1) / split;
    if (n > 0x7fffffffll || split > 65535u) {
        fail(MRB_EINVAL, "%lld rows of %u workgroups each exceed one launch", (long long)n, split);
        return 0;
    }
    grid = dim3((uint32_t)n, split);
    const uint32_t per_thread = (plan.share + kCopyThreads - 1) / kCopyThreads;  // <= kMaxInFlight
    return per_thread <= 2 ? 2 : 8;
}

// The descent plan of a tree of `depth` levels as the wide-row sample kernel takes it: bits 0-3 the
// number of node groups (one dependent load each), then 5 bits per group with its levels (<= 10).
uint32_t pack_groups(int depth) {
    const int count = (depth + kGroupMaxLevels - 1) / kGroupMaxLevels;
    uint32_t packed = (uint32_t)count;
    for (int i = 0; i < count; ++i) packed |= (uint32_t)(depth / count + (i < depth % count ? 1 : 0)) << (4 + 5 * i);
    return packed;
}
// The same with what else the sample kernels' `groups` word carries: bit 19 tells that the generator's call counter
// is on the device (the walk then reads it there; the flag is among the preloaded arguments, the counter's address
// is not), bits 20-31 the number of batches in the launch minus one.
uint32_t groups_word(const SampleArgs& a, int64_t nbatch) {
    return pack_groups(a.depth) | ((uint32_t)(nbatch - 1) << 20) | ((!a.uniforms && a.size < 0) ? 1u << 19 : 0u);
}

// Threads of a wide-row workgroup: the walker wave, the copy waves and, where rows have narrow fields, their wave.
inline uint32_t wide_threads(const WidePlan& plan) { return plan.narrow_items ? (uint32_t)kWideWG : (uint32_t)kWideWG - 64u; }

template <int kInF, bool kTen, bool kOneWide>
void launch_sample_wide(dim3 grid, const SampleArgs& a, const WidePlan& plan, hipStream_t s) {
    const SampleTail tail{a.mn, a.out_idx, a.out_w, a.err, a.size, a.beta};
    launch_kernel((k_per_sample_wide<kInF, kTen, kOneWide>), grid, dim3(wide_threads(plan)), 0, s, a.sum, a.uniforms, a.depth,
                  groups_word(a, plan.nbatch), (int)a.batch, (uint32_t)a.capacity, a.seed, a.calls, tail, plan);
}

template <int kInF>
void launch_sample_wide_as(dim3 grid, const SampleArgs& a, const WidePlan& plan, hipStream_t s) {
    const bool ten = a.depth > 0 && a.depth % kGroupMaxLevels == 0;  // every node group takes 10 levels
    const bool one = plan.nwide == 1;
    if (ten) one ? launch_sample_wide<kInF, true, true>(grid, a, plan, s) : launch_sample_wide<kInF, true, false>(grid, a, plan, s);
    else one ? launch_sample_wide<kInF, false, true>(grid, a, plan, s) : launch_sample_wide<kInF, false, false>(grid, a, plan, s);
}

// A sample call's optional second layer: field `row_field` of the row whose slot number the sampled row holds
// in its 8-byte field `slot_field` goes to `out` ([batch, row bytes]).
struct NextRows {
    int slot_field = -1, row_field = -1;
    void* out = nullptr;
};

constexpr int64_t kRowWaveMinRows = 2048;  // fewest rows of a launch that go to the wave-per-row sample and gather kernels

template <int kInF, bool kTen, bool kOneWide>
void launch_sample_next(dim3 grid, const SampleArgs& a, const WidePlan& plan, const NextPlan& nx, hipStream_t s) {
    const SampleTail tail{a.mn, a.out_idx, a.out_w, a.err, a.size, a.beta};
    launch_kernel((k_per_sample_next<kInF, kTen, kOneWide>), grid, dim3(wide_threads(plan)), 0, s, a.sum, a.uniforms, a.depth,
                  groups_word(a, 1), (int)a.batch, (uint32_t)a.capacity, a.seed, a.calls, tail, plan, nx);
}

template <int kInF>
void launch_sample_next_as(dim3 grid, const SampleArgs& a, const WidePlan& plan, const NextPlan& nx, hipStream_t s) {
    const bool ten = a.depth > 0 && a.depth % kGroupMaxLevels == 0;
    const bool one = plan.nwide == 1;
    if (ten) one ? launch_sample_next<kInF, true, true>(grid, a, plan, nx, s) : launch_sample_next<kInF, true, false>(grid, a, plan, nx, s);
    else one ? launch_sample_next<kInF, false, true>(grid, a, plan, nx, s) : launch_sample_next<kInF, false, false>(grid, a, plan, nx, s);
}

int sample_wide(const RowStore& r, const SampleArgs& a, const IoTable& t, int64_t nbatch, hipStream_t s,
                const NextRows* next = nullptr) {
    WidePlan plan;
    dim3 grid;
    plan.nbatch = (uint32_t)nbatch;
    const int inflight = wide_plan(r, t, nbatch * a.batch, plan, grid);
    if (inflight == 0) return MRB_EINVAL;
    plan.through = stores_through(batch_bytes(t), kThroughSample, whole_pieces(plan));
    if (next) {
        // the second layer of workgroups: one wide field, split like a row of its own
        NextPlan nx{};
        const int f = next->row_field;
        nx.slot_field = r.data[next->slot_field];
        nx.plan.nwide = 1;
        nx.plan.nbatch = 1;
        nx.plan.f[0].src = r.data[f];
        nx.plan.f[0].dst = static_cast<uint8_t*>(next->out);
        nx.plan.f[0].rb = (uint32_t)r.bytes[f];
        nx.plan.f[0].ss = (uint32_t)r.stride[f];
        nx.slot_stride = (uint32_t)r.stride[next->slot_field];
        nx.plan.wide_items = r.units[f];
        const uint32_t per_wg = (uint32_t)kMaxInFlight * kCopyThreads;
        const uint32_t split = (nx.plan.wide_items + per_wg - 1) / per_wg;
        nx.plan.split = (int)split;
        nx.plan.share = (nx.plan.wide_items + split - 1) / split;
        plan.through = nx.plan.through =
            stores_through(batch_bytes(t) + (uint64_t)a.batch * r.bytes[f], kThroughSample, whole_pieces(plan) && whole_pieces(nx.plan));
        if (split > 65535u) return fail(MRB_EINVAL, "field %d is too wide for one launch", f);
        if (split > grid.y) grid.y = split;
        grid.z = 2;
        const uint32_t per_thread = (nx.plan.share + kCopyThreads - 1) / kCopyThreads;
        if (inflight == 2 && per_thread <= 2) launch_sample_next_as<2>(grid, a, plan, nx, s);
        else launch_sample_next_as<8>(grid, a, plan, nx, s);
        LAUNCH_CHECK("k_per_sample_next");
        return MRB_OK;
    }
    // Many rows of up to 4 KB in 16-byte fields and 49 to 256 narrow bytes (with fewer, sixteen lanes to a stratum have taken them):
    // a wave per row (k_per_sample_rows) instead of a workgroup per row. One wave does in a row what six do side by side, so a launch
    // of few rows takes longer that way and a launch of many less, for a sixth of the waves to dispatch (rows of 521 bytes, wave /
    // workgroup: 1024 6.4 / 5.5 us, 4096 9.2 / 15.6, 16,384 26 / 54). (`row_split` asks for the workgroup kernel.)
    const int64_t nrows = nbatch * a.batch;
    if (r.row_split == 0 && r.row_wave != 2 && plan.split == 1 && plan.wide_items <= (uint32_t)kRowWaveInF * 64u &&
        plan.narrow_items <= 256u && (nrows >= kRowWaveMinRows || r.row_wave == 1)) {
        const SampleTail tail{a.mn, a.out_idx, a.out_w, a.err, a.size, a.beta};
        const uint32_t blocks = (uint32_t)((nrows + kRowWaveWG / 64 - 1) / (kRowWaveWG / 64));
        const uint32_t packed = groups_word(a, plan.nbatch);
        if (a.depth > 0 && a.depth % kGroupMaxLevels == 0)
            launch_kernel((k_per_sample_rows<true>), dim3(blocks), dim3(kRowWaveWG), 0, s, a.sum, a.uniforms, a.depth, packed,
                          (int)a.batch, (uint32_t)a.capacity, a.seed, a.calls, nrows, tail, plan);
        else
            launch_kernel((k_per_sample_rows<false>), dim3(blocks), dim3(kRowWaveWG), 0, s, a.sum, a.uniforms, a.depth, packed,
                          (int)a.batch, (uint32_t)a.capacity, a.seed, a.calls, nrows, tail, plan);
        LAUNCH_CHECK("k_per_sample_rows");
        return MRB_OK;
    }
    // Fewer rows of that size: the workgroup kernel with two copy waves instead of four (k_per_sample_light).
    if (r.row_split == 0 && plan.split == 1 && plan.wide_items <= 2u * 64u * kLightCopyWaves && a.depth != 22) {
        const SampleTail tail{a.mn, a.out_idx, a.out_w, a.err, a.size, a.beta};
        const uint32_t packed = groups_word(a, plan.nbatch);
        const dim3 threads(plan.narrow_items ? (uint32_t)kLightWG : (uint32_t)kLightWG - 64u);
        const bool ten = a.depth > 0 && a.depth % kGroupMaxLevels == 0, one = plan.nwide == 1;
#define MRB_LAUNCH_LIGHT(T, O)                                                                                         \
    launch_kernel((k_per_sample_light<T, O>), grid, threads, 0, s, a.sum, a.uniforms, a.depth, packed, (int)a.batch, \
                  (uint32_t)a.capacity, a.seed, a.calls, tail, plan)
        if (ten) { if (one) MRB_LAUNCH_LIGHT(true, true); else MRB_LAUNCH_LIGHT(true, false); }
        else { if (one) MRB_LAUNCH_LIGHT(false, true); else MRB_LAUNCH_LIGHT(false, false); }
#undef MRB_LAUNCH_LIGHT
        LAUNCH_CHECK("k_per_sample_light");
        return MRB_OK;
    }
    if (inflight == 2) launch_sample_wide_as<2>(grid, a, plan, s);
    else launch_sample_wide_as<8>(grid, a, plan, s);
    LAUNCH_CHECK("k_per_sample_wide");
    return MRB_OK;
}

template <int kInF>
void launch_gather_wide(dim3 grid, const int64_t* indices, int mode, int64_t count, int64_t fixed_slot, uint64_t seed,
                        uint64_t calls, int64_t* out_indices, uint32_t* err, const WidePlan& plan, hipStream_t s) {
    if (plan.nwide == 1)
        launch_kernel((k_rows_gather_wide<kInF, true>), grid, dim3(wide_threads(plan)), 0, s, indices, mode, count, fixed_slot, seed,
                      calls, out_indices, err, plan);
    else
        launch_kernel((k_rows_gather_wide<kInF, false>), grid, dim3(wide_threads(plan)), 0, s, indices, mode, count, fixed_slot, seed,
                      calls, out_indices, err, plan);
}

// Gather of n rows whose slots are given (indices), drawn from the generator (indices NULL,
// fixed_slot < 0) or one fixed slot: by a kernel that numbers a field's granules over all rows, or one that
// gives a row a workgroup or a wave.
int gather_rows(const RowStore& r, const int64_t* indices, int64_t fixed_slot, int64_t count, uint64_t seed,
                uint64_t calls, int64_t n, int64_t* out_indices, void* const* dst_fields, uint32_t* err,
                hipStream_t s) {
    IoTable t;
    int rc = make_table(r, dst_fields, n, t);
    if (rc) return rc;
    ShortIo io{};
    const bool brief = fixed_slot < 0 && n <= 0xffffffffll && (out_indices ? short_io(out_indices, nullptr, t, io) : short_io(t, io));
    const uint64_t most = most_granules(t);
    // The flat kernel is the faster one but for some hundred rows of 4 KB and more, which are too few granules for four to a thread and
    // go by a workgroup per row, and for more than 29 MB of rows that fill most of a wave, which go by a wave per row. us, that / flat
    // (given slots in brackets):
    //   workgroup per row    32 rows      120,000 granules       200,000                500,000 to 900,000      more
    //     5 KB                            3.5 / 3.3 (3.0 / 3.1)  3.9 / 3.9 (3.2 / 3.7)
    //     7.5 KB             3.1 / 2.8    3.4 / 3.3 (2.9 / 3.0)  3.8 / 3.8 (3.1 / 3.7)  5.3 / 5.5               4096 rows 15.0 / 13.9
    //     12 KB                           3.7 / 2.9 (3.2 / 2.8)  4.1 / 3.5 (3.5 / 3.4)  7.1 / 7.6 (5.9 / 6.0)   2048 rows 12.0 / 11.5
    //     28 KB              3.7 / 2.7    3.9 / 2.9 (3.2 / 2.8)  4.1 / 3.4 (3.4 / 3.4)  7.4 / 7.6 (5.7 / 6.3)   2048 rows 22.9 / 22.5
    //   wave per row         2048 rows    8192                       12,000                     16,384
    //     1 KB               4.9 / 3.5     7.7 /  6.2                10.2 /  7.5                12.3 /  9.2
    //     2 KB (odd)                      11.5 /  9.1                15.5 / 12.1                19.3 / 16.3
    //     2.4 KB             5.4 / 4.7    10.8 / 10.2                14.1 / 14.1 (13.9 / 14.2)  17.4 / 18.0
    //     2.8 KB (odd)                    13.2 / 12.3                17.2 / 17.2 (17.1 / 16.8)  21.6 / 20.4
    //     3.2 KB             5.7 / 5.1    12.4 / 11.7                15.8 / 15.9 (15.6 / 16.2)  20.5 / 20.8
    //     3.6 KB                          13.0 / 12.9 (12.5 / 13.2)  17.1 / 18.1                22.5 / 23.4
    //     4 KB               6.2 / 6.0    13.5 / 14.2 (13.6 / 14.5)  18.3 / 19.1                24.2 / 24.7
    // And row_split asks for a workgroup per row, as row_wave = 2 does, and row_wave = 1 for a wave per row; what a brief launch's arguments do
    // not hold goes to the kernels that take a plan.
    int64_t granules = 0, narrow = 0;  // of a row: in fields of 16 bytes and more, and the bytes of the others
    for (int f = 0; f < r.nfields; ++f) {
        if (r.vec_log2[f] == 4) granules += r.units[f];
        else narrow += r.bytes[f];
    }
    const bool by_workgroup = widest_field(r) >= 4096 && most >= 200000 && most <= 1u << 20;
    const bool by_wave = granules >= 144 && granules <= kRowWaveInF * 64 && narrow <= 256 && n * granules >= 1800000;
    if (widest_field(r) >= 1024 && n <= (1ll << 24) && (by_workgroup || by_wave || !brief || r.row_split != 0 || r.row_wave != 0)) {
        const int mode = fixed_slot >= 0 ? kFromFixedSlot : (indices ? kFromIndices : kFromGenerator);
        WidePlan plan;
        dim3 grid;
        plan.nbatch = 1;
        const int inflight = wide_plan(r, t, n, plan, grid);
        plan.through = stores_through(batch_bytes(t), kThroughGather, whole_pieces(plan));
        // Thousands of rows of up to 4 KB: a wave per row (3 KB, us, workgroup / wave: 1024 rows 6.2 / 6.7, 2048 7.5 / 6.8,
        // 8192 20.7 / 13.6; 1 KB: 2048 5.2 / 5.5, 4096 7.4 / 5.9).
        if (r.row_split == 0 && plan.split == 1 && plan.wide_items <= (uint32_t)kRowWaveInF * 64u && plan.narrow_items <= 256u &&
            inflight != 0 && n >= kRowWaveMinRows && r.row_wave != 2) {
            launch_kernel(k_rows_gather_rows, dim3((uint32_t)((n + kRowWaveWG / 64 - 1) / (kRowWaveWG / 64))), dim3(kRowWaveWG),
                          0, s, indices, mode, count, fixed_slot, seed, calls, n, out_indices, err, plan);
            LAUNCH_CHECK("k_rows_gather_rows");
            return MRB_OK;
        }
        switch (inflight) {
            case 0: return MRB_EINVAL;
            case 2: launch_gather_wide<2>(grid, indices, mode, count, fixed_slot, seed, calls, out_indices, err, plan, s); break;
            default: launch_gather_wide<8>(grid, indices, mode, count, fixed_slot, seed, calls, out_indices, err, plan, s); break;
        }
        LAUNCH_CHECK("k_rows_gather_wide");
        return MRB_OK;
    }
    // a row of workgroups per field, as many as the field with the most granules needs
    const uint32_t blocks = grid_for(most);
    if (brief) {
        const hipError_t e = launch_short_gather(r.table, io, t, indices, count, seed, calls, n, blocks, out_indices != nullptr, s);
        return e == hipSuccess ? MRB_OK : fail(MRB_EHIP, "launch k_short_gather: %s", hipGetErrorString(e));
    }
    launch_kernel(k_rows_gather, dim3(blocks, (uint32_t)t.nfields), dim3(kWG), 0, s, indices, fixed_slot, seed, calls,
                  count, out_indices, err, r.capacity, blocks, t);
    LAUNCH_CHECK("k_rows_gather");
    return MRB_OK;
}

// ---- the allocation-free entry point's scratch (mrb_per_update_noalloc) -------------------------
// Device memory that exists from the moment the library is loaded: callers that must not allocate
// (HIP graph capture, serving loops, harnesses that forbid hipMalloc) get the update_priorities
// scratch from here. Every device holds its own copy at its own address; `scratch` itself is only
// the host-side name of the symbol and is never passed to a kernel.
constexpr int64_t kNoAllocMaxEntries = 1 << 18;  // 1 MiB per device
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

}  // namespace

static __device__ __align__(256) float scratch[1 << 18];

namespace {

// Address of the current device's copy of `scratch`, looked up once per device.
int static_scratch(float** out) {
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(MRB_EINVAL, "device %d outside [0, %d)", dev, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        float* p = nullptr;
        HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return MRB_OK;
}

struct Urb {
    RowStore rows;
    int64_t count = 0, head = 0;
    uint64_t seed = 0, calls = 0;
    uint32_t* err = nullptr;       // (behind rows.table) 16 bytes of flags, then the device copy of the counters (kUrb* in mrb_kernels.h)
    int64_t* counters = nullptr;   // = err + 16 bytes
    int64_t* slots = nullptr;      // device array of kUrbDrawMax slots: drawn there when the counters live on the device
    int64_t device_counters = 0;   // option "device_counters"
    ~Urb() {
        if (slots) (void)hipFree(slots);
    }
};

// count / head after appending n rows (write position chosen once per call: `count` while the
// buffer has never wrapped, else `head`).
void urb_advance(Urb& b, int64_t n) {
    const int64_t cap = b.rows.capacity;
    if (b.count < cap && b.head == 0) {
        const int64_t room = cap - b.count;
        if (n <= room) {
            b.count += n;
        } else {
            b.count = cap;
            b.head = (n - room) % cap;
        }
    } else {
        b.head = (b.head + n) % cap;
        b.count = b.count + n < cap ? b.count + n : cap;
    }
}

struct Per {
    RowStore rows;
    int64_t leaves = 1;
    int depth = 0;
    int64_t size = 0, pushes = 0;
    float alpha = 1.0f;
    float* sum = nullptr;
    float* mn = nullptr;
    unsigned long long* stamp = nullptr;
    float* maxp = nullptr;
    // sparse plan for very large trees (see k_tree_sparse): lowest s_g0 levels per entry, then s_rounds rounds, of which
    // the last one is k_tree_runs
    int s_g0 = 0, s_rounds = 0;
    int s_lo[kMaxRounds] = {}, s_g[kMaxRounds] = {};
    uint32_t* s_dirty[kMaxRounds] = {};
    // scratch of update_priorities (p^alpha of the call's entries): sized at create; a call with more
    // entries gets a larger array and the old one is kept until destroy (work may still be queued on it)
    float* powered = nullptr;
    int64_t powered_cap = 0;
    std::vector<float*> retired;
    uint32_t* err = nullptr;
    uint32_t* dirty[kMaxRounds] = {};
    int nrounds = 0;
    int lo[kMaxRounds] = {};
    int g[kMaxRounds] = {};
    int top_depth = 0;
    uint64_t epoch = 0;
    uint64_t seed = 0, calls = 0;
    int device = 0;           // the HIP device the buffer lives on
    int64_t sample_path = 0;  // option "sample_path": 0 = choose by row size, 1 = wide-row kernel, 2 = LDS-top kernel
    int64_t lds_levels = 0;   // option "lds_levels": tree levels staged in LDS by the LDS-top kernel (0 = auto)
    int64_t fused = 1;        // option "fused_rebuild": small updates and pushes rebuild the tree in one launch
    int64_t* counters = nullptr;   // device copy of pushes / size / calls (Counters in mrb_kernels.h)
    int64_t device_counters = 0;   // option "device_counters": kernels read the counters from the device
    ~Per() {
        if (sum) (void)hipFree(sum);
        if (mn) (void)hipFree(mn);
        if (stamp) (void)hipFree(stamp);
        if (powered) (void)hipFree(powered);
        for (auto* d : retired) (void)hipFree(d);
        for (auto* d : s_dirty)
            if (d) (void)hipFree(d);
        for (auto* d : dirty)
            if (d) (void)hipFree(d);
    }
};

struct Res {
    RowStore rows;
    int64_t size = 0, total = 0;
    uint64_t seed = 0, calls = 0, epoch = 0;
    unsigned long long* stamp = nullptr;
    uint32_t* err = nullptr;
    ~Res() {
        if (stamp) (void)hipFree(stamp);
    }
};

std::mutex g_mu;
int64_t g_next = 1;
std::unordered_map<int64_t, std::shared_ptr<Urb>> g_urb;
std::unordered_map<int64_t, std::shared_ptr<Per>> g_per;
std::unordered_map<int64_t, std::shared_ptr<Res>> g_res;

std::shared_ptr<Urb> find_urb(int64_t h) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_urb.find(h);
    return it == g_urb.end() ? nullptr : it->second;
}
std::shared_ptr<Per> find_per(int64_t h) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_per.find(h);
    return it == g_per.end() ? nullptr : it->second;
}

std::shared_ptr<Res> find_res(int64_t h) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_res.find(h);
    return it == g_res.end() ? nullptr : it->second;
}
#define GET_RES(b, h)                                                              \
    auto b = find_res(h);                                                          \
    if (!b) return fail(MRB_EHANDLE, "unknown reservoir buffer handle %lld", (long long)(h))
#define GET_URB(b, h)                                                              \
    auto b = find_urb(h);                                                          \
    if (!b) return fail(MRB_EHANDLE, "unknown uniform buffer handle %lld", (long long)(h))
#define GET_PER(b, h)                                                              \
    auto b = find_per(h);                                                          \
    if (!b) return fail(MRB_EHANDLE, "unknown priority buffer handle %lld", (long long)(h))

int read_and_clear_flags(uint32_t* d_err, uint32_t* flags, hipStream_t s) {
    uint32_t v = 0;
    HIP_TRY(hipMemcpyAsync(&v, d_err, sizeof(v), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (v) {
        HIP_TRY(hipMemsetAsync(d_err, 0, sizeof(v), s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    if (flags) *flags = v;
    return MRB_OK;
}

// Leaf tiles that n consecutive slots of the ring can meet wherever they start: ceil(n / 256) + 1 for the
// misalignment, one more where the slots wrap around the ring's end; never more than the ring's tiles.
uint32_t push_units(const UpdateArgs& a) {
    const uint64_t ring_tiles = ((uint64_t)a.capacity + kBlockNodes - 1) / kBlockNodes;
    const uint64_t units = ((uint64_t)a.n + kBlockNodes - 1) / kBlockNodes + 2;
    return (uint32_t)(units < ring_tiles ? units : ring_tiles);
}

// A push whose tree work is ONE launch and that also moves the device's counters on (a.advance != 0): every
// workgroup that rides along reports to one counter when it has read the ring position (see counters_push_done),
// which is worth it for a few dozen workgroups only - a larger copy then gets a launch of its own, ahead.
constexpr uint32_t kRideWithCounters = 64;
int ride_alone_if_large(const UpdateArgs& a, PutArgs& put, hipStream_t s) {
    if (a.advance && put.blocks > kRideWithCounters) {
        launch_kernel(k_rows_put, dim3(put.blocks), dim3(kWG), 0, s, put);
        LAUNCH_CHECK("k_rows_put");
        put.blocks = 0;
    }
    return MRB_OK;
}

// A push under at most 16 leaf tiles on a tree with levels above them is one launch of one workgroup, a wave per
// leaf tile (k_push_run; k_tree_fused where an update precedes it in the call): the number of those tiles, 0 where it
// is not taken. (More than one tile per wave does not pay: the 16 waves of a workgroup share one compute unit's issue
// slots, and a second tile costs a wave as much as the launch it would save; four cost twice as much.)
uint32_t run_units(const Per& b, const UpdateArgs& a) {
    if (a.depth <= kRoundLevels || !b.fused || a.indices) return 0;
    uint64_t units;
    if (a.first_slot < 0) {
        units = push_units(a);  // the slots' start is only known on the device
    } else {
        const uint64_t ring_tiles = ((uint64_t)a.capacity + kBlockNodes - 1) / kBlockNodes;
        const int64_t end = a.first_slot + a.n, first = a.first_slot / kBlockNodes;
        units = end <= a.capacity ? (uint64_t)((end - 1) / kBlockNodes - first + 1)
                                  : ring_tiles - first + (uint64_t)((end - a.capacity - 1) / kBlockNodes + 1);
        if (units > ring_tiles) units = ring_tiles;
    }
    return units <= (uint64_t)kRunWaves ? (uint32_t)units : 0u;
}

// Rebuilds the tree above the leaves that `a` writes: one launch per round, then the top. A push hands
// its row copy over (`ride`): it is done by extra workgroups of the first launch.
int tree_rebuild(Per& b, UpdateArgs a, hipStream_t s, const PutArgs* ride = nullptr) {
    PutArgs none{};  // blocks == 0: no copy rides along
    if (const uint32_t units = run_units(b, a)) {
        PutArgs put = ride ? *ride : none;
        if (int rc = ride_alone_if_large(a, put, s)) return rc;
        if (a.full_top) {
            // (the update's launch before this one has carried the row copy)
            a.readers = 1;
            launch_kernel(k_tree_fused, dim3(1), dim3(kFusedWG), 0, s, a, (uint32_t)(a.first_slot / kBlockNodes), units);
            LAUNCH_CHECK("k_tree_fused");
            return MRB_OK;
        }
        const uint32_t threads = units <= kWG / 64 ? (uint32_t)kWG : (uint32_t)kFusedWG;
        put.blocks = (put.blocks * kWG + threads - 1) / threads;  // the ride-along copy was sized for workgroups of kWG
        put.threads = threads;
        if (ShortIo io{}; put.blocks && a.first_slot >= 0 && a.advance == 0 && a.fold_max != 1 && short_io(put.t, io)) {
            const hipError_t e = launch_short_push_run(b.rows.table, io, put.t.nfields, a, units, most_granules(put.t), threads, s);
            return e == hipSuccess ? MRB_OK : fail(MRB_EHIP, "launch k_short_push_run: %s", hipGetErrorString(e));
        }
        a.readers = 1 + put.blocks;  // (a.advance != 0: this one launch also moves the device's counters on)
        launch_kernel(k_push_run, dim3(1 + put.blocks), dim3(threads), 0, s, a, units, put);
        LAUNCH_CHECK("k_push_run");
        return MRB_OK;
    }
    // A push of at most 1024 rows into a tree of at most 16 levels is one launch: the single workgroup of
    // k_tree_top starts at the leaf level and skips the tiles outside the slot range (such a call is
    // launch-bound, not work-bound). Measured on 16,384 leaves: 6.3 us instead of 8.0. Updates keep their
    // leaf round: their waves scan the entries, which one workgroup does more slowly (11.5 vs 9.8 us).
    if (a.nrounds > 0 && !a.indices && a.n <= 1024 && a.depth <= 16) {
        a.nrounds = 0;
        a.top_depth = a.depth;
    }
    for (int r = 0; r < a.nrounds; ++r) {
        uint32_t tiles = (1u << a.lo[r]) / kBlockNodes;
        uint32_t tile_base = 0;
        if (r == 0 && !a.indices && a.first_slot < 0) {
            // a push whose first slot only the device knows: enough waves for every tile the slots can meet;
            // the kernel places them (tile_base carries their number)
            tiles = push_units(a);
            tile_base = tiles;
        } else if (r == 0 && !a.indices && a.first_slot + a.n <= a.capacity) {
            // a push that does not wrap: only the leaf tiles under its slot range need a wave
            tile_base = (uint32_t)(a.first_slot / kBlockNodes);
            tiles = (uint32_t)((a.first_slot + a.n - 1) / kBlockNodes) - tile_base + 1;
        }
        const PutArgs& put = (r == 0 && ride) ? *ride : none;
        if (r == 0 && a.inline_election) tiles = (a.n > kPairedAbove ? 2u : 1u) * (uint32_t)a.n;  // one or two waves per entry (see k_tree_update)
        a.tile_blocks = (tiles + 3) / 4;
        launch_kernel(k_tree_update, dim3(a.tile_blocks + put.blocks), dim3(kWG), 0, s, a.indices, a.priorities, a.sum, a.mn,
                      a.n, a.capacity, r | a.lo[r] << 8 | a.g[r] << 16, a.alpha, a, tile_base, put);
        LAUNCH_CHECK("k_tree_update");
    }
    PutArgs put = (a.nrounds == 0 && ride) ? *ride : none;
    if (int rc = ride_alone_if_large(a, put, s)) return rc;
    put.threads = kTopWG;
    // the top is the call's last launch: it moves the device's counters on (a.advance != 0); only when it is also
    // the first do its workgroups read the ring position
    a.readers = a.nrounds == 0 ? 1 + put.blocks : 0;
    launch_kernel(k_tree_top, dim3(1 + put.blocks), dim3(kTopWG), 0, s, a, put);
    LAUNCH_CHECK("k_tree_top");
    return MRB_OK;
}

// Zero-fills `bytes` (a multiple of 4) of device memory with a kernel.
void fill_zero(void* p, size_t bytes, hipStream_t s) {
    const uint64_t n = bytes / sizeof(float);
    launch_kernel(k_fill_f32, dim3(grid_for(n)), dim3(kWG), 0, s, static_cast<float*>(p), 0.0f, n);
}

// A push whose leaf tiles are rebuilt by several workgroups, or whose powers one shares out over its threads (k_push_many): with
// priorities always; without, one tile (us, k_push_run / this: 3.6 / 3.3), more than k_push_run takes, or on more than 16 levels
// twelve and more: up to there, and on trees with one tile above the leaf tiles, the roots' meeting costs more than sharing the
// tiles out saves (1024 / 2048 / 2560 / 3072 / 3584 rows of 37 bytes, 14 levels 3.1 / 3.4 / 3.4 / 3.6 / 3.6 against 3.8 / 3.8 / 3.8 / 3.8 / 3.9, 16
// levels 3.2 / 3.4 / 3.5 / 3.6 / 3.7 against 4.0 each, 17 levels 3.9 / 4.4 / 4.5 / 4.9 / 5.0 against 4.5 / 4.6 / 4.6 / 4.6 / 4.6, 20 levels
// 4.1 / 4.6 / 4.8 / 5.1 / 5.2 against 4.8 / 4.9 / 4.9 / 4.9 / 4.9). Or a copy of more than kManyCopy workgroups, which waits for
// k_push_run's large ones (300 rows of 28 KB 9.3 / 4.9, 1000 18.2 / 10.9).
constexpr int64_t kManyLeastTiles = 12;
constexpr int kManyLeastDepth = 17;
constexpr uint32_t kManyCopy = 1024;
bool takes_push_many(const Per& b, int64_t first, int64_t n, bool with_priorities, uint32_t copy_blocks) {
    if (b.device_counters || !b.fused || b.depth <= kRoundLevels || first + n > b.rows.capacity) return false;
    const int64_t tiles = (first + n - 1) / kBlockNodes - first / kBlockNodes + 1;
    if (tiles > kManyMostTiles) return false;
    return with_priorities || tiles == 1 || tiles > kRunWaves || (tiles >= kManyLeastTiles && b.depth >= kManyLeastDepth) ||
           copy_blocks > kManyCopy;
}

// Starts a new tree-update epoch. Epochs tag stamps and dirty words so that
// neither needs clearing between calls; when the 32-bit tag would wrap, both
// are cleared once.
int next_epoch(Per& b, hipStream_t s) {
    b.epoch += 1;
    if ((uint32_t)b.epoch == 0) {
        // cleared by a fill kernel, not a memset node: a caller may be capturing this stream (0.0f is all-zero bits)
        fill_zero(b.stamp, sizeof(unsigned long long) * (size_t)b.leaves, s);
        for (int r = 0; r < b.nrounds; ++r) fill_zero(b.dirty[r], sizeof(uint32_t) * ((size_t)1 << (b.lo[r] - b.g[r])), s);
        for (int r = 0; r < b.s_rounds; ++r)
            fill_zero(b.s_dirty[r], sizeof(uint32_t) * ((size_t)1 << (b.s_lo[r] - b.s_g[r])), s);
        LAUNCH_CHECK("k_fill_f32");
        b.epoch += 1;
    }
    return MRB_OK;
}

UpdateArgs update_args(Per& b) {
    UpdateArgs a{};
    a.capacity = b.rows.capacity;
    a.leaves = b.leaves;
    a.depth = b.depth;
    a.alpha = b.alpha;
    a.epoch = (uint32_t)b.epoch;
    a.stamp = b.stamp;
    a.sum = b.sum;
    a.mn = b.mn;
    a.maxp = b.maxp;
    a.maxp_next = b.maxp + 1;
    a.err = b.err;
    a.nrounds = b.nrounds;
    for (int r = 0; r < kMaxRounds; ++r) {
        a.dirty[r] = b.dirty[r];
        a.lo[r] = b.lo[r];
        a.g[r] = b.g[r];
    }
    a.top_depth = b.top_depth;
    return a;
}

// Most entries of an update that elect the last writer of each leaf among themselves (a wave per entry scans
// the call's entries); larger calls take the stamp pass (2048 entries on 2^21 leaves 14.0 us against 14.7 with the pass, at twice
// the waves and four times the comparisons: not taken).
constexpr int64_t kElectMax = 1024;

// Whether an update of few entries goes by runs of leaves in k_range_one, whose workgroups read the priorities with the indices and
// leave where they have no entry, rather than in k_tree_range. us, k_range_one / k_tree_range:
//   levels   entries   random         one by one
//   20       1024       6.7 /  7.3     6.1 /  7.3
//   20       1500       7.8 /  7.5     7.5 /  7.7
//   20       3000       8.5 /  8.2     8.6 /  9.0
//   20       4096       8.8 /  8.5    10.6 / 11.1    (the line of 4096 is where these two take turns)
//   21        512       6.4 /  7.2     5.6 /  6.7
//   21       1024       7.4 /  7.6     6.3 /  7.4
//   22       1024       7.4 /  7.9     6.7 /  7.9
// Trees of fewer than 8 levels have no whole tile, those of more than 22 more than 256 runs.
bool takes_range_one(const Per& b, int64_t n) {
    return b.fused && n <= (b.depth <= 20 ? kOneMostEntries : kElectMax) && b.depth >= 8 && b.depth <= 22;
}

// Whether an update of more entries goes by runs of leaves (launch_tree_range). us, by stamps and tiles / by runs, slots at random; in the
// order that a sample returns them; one after the other:
//   levels   entries    random          sample's        one by one
//   12         8192      9.2 /  9.4                      7.9 /  7.2
//   12       16,384     10.5 / 13.7                      8.1 /  9.6
//   14         8192     10.1 /  8.7      9.2 /  6.6      9.2 /  6.7
//   14       12,000     10.2 / 10.6      9.3 /  7.5      9.2 /  7.7
//   14       16,384     10.3 / 11.5      9.2 /  8.1      9.3 /  7.8
//   14       32,768     10.9 / 16.7                      9.2 / 10.6
//   18       12,000     10.1 / 10.2      9.5 /  8.5      9.1 /  8.6
//   18       16,384     10.3 / 10.9      9.7 /  9.0      9.3 /  9.3
//   20         8192     11.4 /  9.6     11.1 /  8.6      9.9 / 11.6
//   20       16,384     11.9 / 12.2     11.4 / 10.1      9.9 / 13.1
//   20       32,768     12.9 / 16.9                      9.9 / 15.6
// (The line of 16,384 is the sample's order's.) Trees of more than 22 levels have more than one tile above the runs. On 21 levels and more
// what its entries drive is the other way: see takes_sparse.
bool takes_range(const Per& b, int64_t n) {
    if (!b.fused || b.depth < 12 || b.depth > 22) return false;
    return !takes_range_one(b, n) && n <= (b.depth >= 21 ? 3072 : b.depth == 12 ? 8192 : 16384);
}

// Whether the entries drive the lowest levels of an update (launch_tree_sparse), with more than the 1024 that elect among themselves.
// The other ways look at every entry in every workgroup (by runs of leaves: up to 3072 entries on 21 and 22 levels) or at every tile
// of the tree. us per call, the other way / by entries, slots at random; in the order that a sample returns them; one after the
// other; half of them and all of them the same:
//   levels  entries    random         sample's       one by one     half           all
//   21        2,048     8.1 /  9.3     7.8 /  9.1     9.1 /  8.8     9.1 /  9.3     8.8 /  8.1    by runs
//   21        3,073     8.7 /  9.5     8.2 /  9.2    10.8 /  8.8    10.4 /  9.4    10.1 /  8.3    by runs
//   21        4,096     9.3 /  9.6     8.8 /  9.3    11.7 /  9.0    11.8 /  9.6    11.3 /  8.5    by runs
//   21        8,192    10.3 / 10.0     9.4 /  9.6    15.7 /  8.9    15.1 / 10.8    14.8 /  9.1    by runs
//   21       16,384    13.6 / 11.0    11.5 / 10.1    18.4 /  9.0    24.1 / 13.0    24.0 / 10.5    by runs
//   22        2,048     8.6 /  9.3     8.3 /  9.1     9.6 /  8.7     9.2 /  9.0     9.1 /  8.0    by runs
//   22        3,073     9.3 /  9.5     8.9 /  9.3    11.5 /  9.0    10.4 /  9.4    10.2 /  8.2    by runs
//   22        8,192    11.8 / 10.0    11.0 /  9.8    16.4 /  9.0    15.8 / 10.9    15.3 /  9.1    by runs
// and by tiles / by entries, at random, one after the other:
//   21       32,768    17.5 / 13.2                   11.6 /  9.5
//   21       65,536    20.3 / 16.9                   11.6 / 10.3
//   21      131,072    24.9 / 23.6                   12.3 / 11.6
//   22       32,768    26.6 / 13.6                   14.5 /  9.5
//   22      131,072    35.4 / 25.1                   15.5 / 11.7
//   22      200,000    39.8 / 34.3                   16.1 / 14.6
//   23      131,072      49 / 27 and 19.2 / 11.7;   262,144   58 / 44 and 20.6 / 16.3;   524,288   73 / 76 and 23.3 / 24.7
//   24      131,072      72 / 31 and 26.9 / 12.0;   262,144   90 / 53 and 27.4 / 16.6;   524,288  109 / 94 and 30.3 / 25.1
//   25      262,144     151 / 73 and 43.8 / 19.7;   524,288  192 / 127 and 46.7 / 30.9;  1,048,576  237 / 220 and 52.3 / 50.1
//   26      524,288     290 / 240 and 77.6 / 47.8;  1,048,576   372 / 438;   deeper trees were not measured
// (The lines of 21, 22 and 24 levels lie at half of what the entries could take: they were drawn when an entry's block was ten pieces of
// lines instead of four.)
bool takes_sparse(const Per& b, int64_t n) {
    const int share = b.depth == 22 || b.depth == 23 ? 5 : b.depth <= 25 ? 6 : b.depth == 26 ? 7 : 8;
    return b.s_g0 > 0 && n > kElectMax && n <= b.leaves >> share;
}

// Where one workgroup's update alone (k_tree_wg) is faster than that. us, k_tree_wg / by runs:
//   levels   1 entry      16           64           96           128
//   10       3.5 / 3.2    3.5 / 3.4    3.5 / 3.4    3.6 / 3.4    3.6 / 3.4
//   11       3.8 / 3.2    3.8 / 3.9    3.8 / 4.0    3.9 / 4.0    3.9 / 4.0    (left to the runs with 10 levels)
//   12       4.1 / 4.4    4.2 / 4.7    4.3 / 4.7    4.6 / 4.7    4.7 / 4.7
//   13       4.1 / 4.6                 4.4 / 4.7    4.6 / 4.7    4.8 / 4.7
//   14       4.1 / 4.5                 4.4 / 4.7    4.7 / 4.7    4.9 / 4.8
bool takes_wg_rather(const Per& b, int64_t n) { return b.depth >= 12 && b.depth <= kWgMaxDepth && n <= 96; }

// update_priorities on buffer b with `powered` (device f32[n]) as the scratch that holds the entries'
// p^alpha between the stamp pass and the leaf writes. Allocates nothing.
int per_update(Per& pb, const int64_t* indices, const float* priorities, int64_t n, float* powered, hipStream_t s) {
    Per* b = &pb;
    if (b->device_counters && n > kElectMax)
        return fail(MRB_ESTATE, "with device_counters an update takes at most 1024 entries (larger ones elect their "
                                "entries with tags the host counts, which a graph replay would repeat)");
    if (n > kElectMax) {
        // the stamp pass tags leaves with an epoch the HOST counts: a recording would freeze it, and replays would
        // elect entries against stale tags. Refused while the stream is being captured (a host-side query).
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(s, &st));
        if (st != hipStreamCaptureStatusNone)
            return fail(MRB_ESTATE, "an update of more than %lld entries cannot be recorded into a HIP graph (its "
                                    "election tags are counted on the host); split it into calls of at most %lld",
                        (long long)kElectMax, (long long)kElectMax);
    }
    if (takes_range_one(*b, n) && !takes_wg_rather(*b, n)) {
        const hipError_t e = launch_range_one(indices, priorities, n, b->sum, b->mn, b->maxp, b->rows.capacity, b->depth, b->alpha, s);
        return e == hipSuccess ? MRB_OK : fail(MRB_EHIP, "launch k_range_one: %s", hipGetErrorString(e));
    }
    if (takes_range(*b, n)) {
        const hipError_t e = launch_tree_range(indices, priorities, n, b->sum, b->mn, b->maxp, b->rows.capacity, b->depth, b->alpha, s);
        if (e != hipSuccess) return fail(MRB_EHIP, "launch k_tree_range: %s", hipGetErrorString(e));
        return MRB_OK;
    }
    int rc = next_epoch(*b, s);
    if (rc) return rc;
    UpdateArgs a = update_args(*b);
    a.powered = powered;
    a.indices = indices;
    a.priorities = priorities;
    a.n = n;
    const bool sparse = takes_sparse(*b, n);
    if (sparse) {
        a.sparse_g0 = b->s_g0;
        a.nrounds = b->s_rounds;
        for (int r = 0; r < kMaxRounds; ++r) {
            a.dirty[r] = b->s_dirty[r];
            a.lo[r] = b->s_lo[r];
            a.g[r] = b->s_g[r];
        }
    }
    // Up to a few hundred entries on a small tree: one workgroup, a thread per entry, walks the paths in one launch (k_tree_wg).
    if (!sparse && b->fused && n <= kWgBestEntries && b->depth >= 2 && b->depth <= kWgMaxDepth) {
        // (65 to 128 entries: 1024 threads, eight per entry - the kernel's one-step path below the staged top)
        const uint32_t threads = n > 64 && n <= 128 ? 1024u : n <= kWgMinThreads ? (uint32_t)kWgMinThreads : (uint32_t)((n + 63) / 64 * 64);
        launch_kernel(k_tree_wg, dim3(1), dim3(threads), 0, s, a.indices, a.priorities, a.sum, a.mn, a.maxp, (int)a.n,
                      a.depth | (int)threads << 8, (int)a.capacity, a.alpha);
        LAUNCH_CHECK("k_tree_wg");
        return MRB_OK;
    }
    // At most 64 entries on a very deep tree: one wave walks the entries' paths, leaves to root, in one launch (k_tree_paths).
    if (!sparse && b->fused && n <= kPathEntries && b->depth <= kPathMaxDepth) {
        launch_kernel(k_tree_paths, dim3(1), dim3(64), 0, s, a);
        LAUNCH_CHECK("k_tree_paths");
        return MRB_OK;
    }
    // A small call on a tree of at least four leaves needs no stamp pass: the leaf-level waves scan the
    // entries themselves (one launch less).
    if (!sparse && n <= kElectMax && b->depth >= 2) {
        a.inline_election = 1;
        return tree_rebuild(*b, a, s);
    }
    launch_kernel(k_update_stamp, dim3(grid_exact((uint64_t)n)), dim3(kWG), 0, s, a.indices, a.priorities, a.stamp, a.powered, a.maxp,
                  (uint32_t)a.n, (uint32_t)a.capacity, a.epoch, a.alpha, !sparse && a.nrounds ? a.dirty[0] : nullptr, a.g[0]);
    LAUNCH_CHECK("k_update_stamp");
    if (!sparse) return tree_rebuild(*b, a, s);
    const auto checked = [](hipError_t e, const char* name) {
        return e == hipSuccess ? MRB_OK : fail(MRB_EHIP, "launch %s: %s", name, hipGetErrorString(e));
    };
    rc = checked(launch_tree_sparse(a.indices, a.stamp, a.powered, a.sum, a.mn, a.dirty[0], n, a.capacity, a.depth, a.sparse_g0,
                                    a.g[0], a.epoch, s), "k_tree_sparse");
    if (rc) return rc;
    const int last = b->s_rounds - 1;
    for (int r = 0; r < last; ++r) {
        const uint32_t tiles = (1u << b->s_lo[r]) / kBlockNodes;
        a.tile_blocks = (tiles + 3) / 4;
        launch_kernel(k_tree_update, dim3(a.tile_blocks), dim3(kWG), 0, s, a.indices, a.priorities, a.sum, a.mn, a.n,
                      a.capacity, r | a.lo[r] << 8 | a.g[r] << 16, a.alpha, a, 0u, PutArgs{});
        LAUNCH_CHECK("k_tree_update");
    }
    return checked(launch_tree_runs(a.sum, a.mn, a.dirty[last], a.maxp, a.lo[last], a.epoch, s), "k_tree_runs");
}


// Device-resident counters: host -> device (when the option is switched on, after a load) and back (state
// queries, when it is switched off). Both wait for the device.
int counters_to_device(Per& b) {
    const int64_t v[kCntWords] = {b.pushes, b.size, (int64_t)b.calls, 0, b.pushes % b.rows.capacity};
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(b.counters, v, sizeof(v), hipMemcpyHostToDevice));
    return MRB_OK;
}
int counters_from_device(Per& b) {
    int64_t v[kCntWords];
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(v, b.counters, sizeof(v), hipMemcpyDeviceToHost));
    b.pushes = v[kCntPushes], b.size = v[kCntSize], b.calls = (uint64_t)v[kCntCalls];
    return MRB_OK;
}
int counters_to_device(Urb& b) {
    const int64_t cap = b.rows.capacity;
    const int64_t v[kCntWords] = {0, b.count, (int64_t)b.calls, b.head, b.count < cap && b.head == 0 ? b.count : b.head};
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(b.counters, v, sizeof(v), hipMemcpyHostToDevice));
    return MRB_OK;
}
int counters_from_device(Urb& b) {
    int64_t v[kCntWords];
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(v, b.counters, sizeof(v), hipMemcpyDeviceToHost));
    b.count = v[kUrbCount], b.head = v[kUrbHead], b.calls = (uint64_t)v[kUrbCalls];
    return MRB_OK;
}
int counters_advance(Urb& b, int64_t rows, int64_t calls, hipStream_t s) {
    launch_kernel(k_urb_advance, dim3(1), dim3(64), 0, s, b.counters, rows, b.rows.capacity, calls);
    LAUNCH_CHECK("k_urb_advance");
    return MRB_OK;
}
int counters_advance(Per& b, int64_t pushed, int64_t calls, hipStream_t s) {
    launch_kernel(k_counters_advance, dim3(1), dim3(64), 0, s, b.counters, pushed, b.rows.capacity, calls);
    LAUNCH_CHECK("k_counters_advance");
    return MRB_OK;
}

// Rows of a workgroup of k_res_push for a call of `nrows` rows of `per_row` granules, 0 where the two launches with stamps
// are taken. Every workgroup draws the later rows' slots, nrows^2 / rows draws in all: at most 2^20 of them (more rows to
// a workgroup beyond that, up to 64), and a thread copies a few granules only. Small rows share a workgroup. (A call of
// more rows than the buffer holds meets too many of its own slots for the lists.)
// Measured at the rule's ends, us per call, two launches / one: 8192 rows of 96 bytes 7.4 / 6.7, 4096 rows of 4 KB 7.95 /
// 7.7, 1448 rows of 28 KB 11.2 / 10.1; beyond them the draws, or the copy by too few workgroups, take what the launch gave.
constexpr int64_t kResMaxGranules = 4096;  // of a workgroup
int res_rows_per_workgroup(int64_t nrows, int64_t per_row, int64_t capacity) {
    if (nrows > kResMaxRows * 128 || nrows > capacity) return 0;
    int64_t rows = 1;
    while (rows < 16 && 2 * rows * per_row <= kResWG / 2) rows *= 2;
    while (nrows * nrows / rows > 1 << 20) rows *= 2;
    return rows <= kResMaxRows && rows * per_row <= kResMaxGranules ? (int)rows : 0;
}

// The rows of a call by a launch that elects the last row of each slot (where rows can meet: `elect`) and one that copies.
int res_push_by_stamps(Res& b, const IoTable& t, int64_t nrows, bool elect, hipStream_t s) {
    const int64_t cap = b.rows.capacity;
    if (elect) {
        b.epoch += 1;
        if ((uint32_t)b.epoch == 0) {
            // by a fill kernel, not a memset node: the caller may be capturing this stream
            fill_zero(b.stamp, (size_t)cap * sizeof(unsigned long long), s);
            LAUNCH_CHECK("k_fill_f32");
            b.epoch += 1;
        }
        launch_kernel(k_res_elect, dim3(grid_exact((uint64_t)nrows)), dim3(kWG), 0, s, b.stamp, b.total, nrows,
                      cap, b.seed, (uint32_t)b.epoch);
        LAUNCH_CHECK("k_res_elect");
    }
    launch_kernel(k_res_put, dim3(grid_for(t.prefix[t.nfields])), dim3(kWG), 0, s, t,
                  elect ? b.stamp : nullptr, b.total, cap, b.seed, (uint32_t)b.epoch);
    LAUNCH_CHECK("k_res_put");
    return MRB_OK;
}

}  // namespace

extern "C" {

const char* mrb_last_error(void) { return g_err; }
int mrb_backend(void) { return 1; }
int mrb_version(void) { return MRB_ABI_VERSION; }

int mrb_set_option(int64_t h, const char* name, int64_t value) {
    if (!name) return fail(MRB_EINVAL, "option name is NULL");
    if (h == 0) {
        // library-wide defaults, taken by buffers created afterwards
        if (strcmp(name, "packed_rows")) return fail(MRB_EINVAL, "'%s' is not a library-wide option (handle 0)", name);
        if (value < 0 || value > 4096) return fail(MRB_EINVAL, "packed_rows must be in [0, 4096] bytes");
        g_packed_rows.store(value);
        return MRB_OK;
    }
    RowStore* rows = nullptr;
    std::shared_ptr<Per> per = find_per(h);
    std::shared_ptr<Urb> urb = per ? nullptr : find_urb(h);
    std::shared_ptr<Res> res = (per || urb) ? nullptr : find_res(h);
    if (per) rows = &per->rows;
    if (urb) rows = &urb->rows;
    if (res) rows = &res->rows;
    if (!rows) return fail(MRB_EHANDLE, "unknown buffer handle %lld", (long long)h);
    if (!strcmp(name, "row_split")) {
        if (value < 0 || value > 64) return fail(MRB_EINVAL, "row_split must be in [0, 64]");
        rows->row_split = value;
    } else if (!strcmp(name, "row_wave")) {
        if (value < 0 || value > 2) return fail(MRB_EINVAL, "row_wave must be 0, 1 or 2");
        rows->row_wave = value;
    } else if (!strcmp(name, "sample_path")) {
        if (!per) return fail(MRB_EINVAL, "sample_path is an option of prioritized buffers");
        if (value < 0 || value > 2) return fail(MRB_EINVAL, "sample_path must be 0, 1 or 2");
        per->sample_path = value;
    } else if (!strcmp(name, "lds_levels")) {
        if (!per) return fail(MRB_EINVAL, "lds_levels is an option of prioritized buffers");
        if (value < 0 || value > 12) return fail(MRB_EINVAL, "lds_levels must be in [0, 12]");
        per->lds_levels = value;
    } else if (!strcmp(name, "device_counters")) {
        if (!per && !urb) return fail(MRB_EINVAL, "device_counters is an option of prioritized and uniform buffers");
        if (value < 0 || value > 1) return fail(MRB_EINVAL, "device_counters must be 0 or 1");
        if (per && value != per->device_counters) {
            const int rc = value ? counters_to_device(*per) : counters_from_device(*per);
            if (rc) return rc;
            per->device_counters = value;
        }
        if (urb && value != urb->device_counters) {
            const int rc = value ? counters_to_device(*urb) : counters_from_device(*urb);
            if (rc) return rc;
            urb->device_counters = value;
        }
    } else if (!strcmp(name, "fused_rebuild")) {
        if (!per) return fail(MRB_EINVAL, "fused_rebuild is an option of prioritized buffers");
        if (value < 0 || value > 1) return fail(MRB_EINVAL, "fused_rebuild must be 0 or 1");
        per->fused = value;
    } else {
        return fail(MRB_EINVAL, "unknown option '%s'", name);
    }
    return MRB_OK;
}

int mrb_field_layout(int64_t h, int field, void** dev_ptr, int64_t* row_stride) {
    const RowStore* rows = nullptr;
    std::shared_ptr<Per> per = find_per(h);
    std::shared_ptr<Urb> urb = per ? nullptr : find_urb(h);
    std::shared_ptr<Res> res = (per || urb) ? nullptr : find_res(h);
    if (per) rows = &per->rows;
    if (urb) rows = &urb->rows;
    if (res) rows = &res->rows;
    if (!rows) return fail(MRB_EHANDLE, "unknown buffer handle %lld", (long long)h);
    if (field < 0 || field >= rows->nfields) return fail(MRB_EINVAL, "bad field %d", field);
    if (dev_ptr) *dev_ptr = rows->data[field];
    if (row_stride) *row_stride = rows->stride[field];
    return MRB_OK;
}

/* ---------------------------------------------------------------- uniform */

int mrb_urb_create(int64_t capacity, int nfields, const int64_t* field_bytes, int64_t* out_handle) {
    if (!out_handle) return fail(MRB_EINVAL, "out_handle is NULL");
    if (capacity > 0x7fffffffll) return fail(MRB_EINVAL, "capacity %lld does not fit the int32 count", (long long)capacity);
    auto b = std::make_shared<Urb>();
    int rc = rows_alloc(b->rows, capacity, nfields, field_bytes, 16 + kCntWords * sizeof(int64_t), &b->err);
    if (rc) return rc;
    b->counters = reinterpret_cast<int64_t*>(b->err + 4);
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->slots), kUrbDrawMax * sizeof(int64_t)));
    HIP_TRY(hipDeviceSynchronize());  // the zero-fills ran on the null stream; the caller's stream may not wait for it
    std::lock_guard<std::mutex> lk(g_mu);
    *out_handle = g_next++;
    g_urb[*out_handle] = b;
    return MRB_OK;
}

int mrb_urb_append(int64_t h, const void* const* src_fields, int64_t nrows, void* stream) {
    GET_URB(b, h);
    if (nrows <= 0) return fail(MRB_EINVAL, "nrows %lld must be positive", (long long)nrows);
    const int64_t cap = b->rows.capacity;
    // Write position: `count` while the buffer has never wrapped, else `head` (the oldest row).
    const bool growing = b->count < cap && b->head == 0;
    const int64_t w = growing ? b->count : b->head;
    // More rows than slots: only the last `cap` survive, at the positions a row-by-row append leaves them.
    const int64_t skip = nrows > cap ? nrows - cap : 0;
    const int64_t first = (w + skip) % cap;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (b->device_counters) {
        // the write position is read on the device, and advanced there after the copy
        if (nrows > cap) return fail(MRB_ESTATE, "with device_counters an append takes at most capacity (%lld) rows", (long long)cap);
        PutArgs p{};
        int rc = put_args(b->rows, src_fields, 0, nrows, 0, p);
        if (rc) return rc;
        p.first_slot = -1;
        p.src_first = reinterpret_cast<int64_t>(b->counters);
        launch_kernel(k_rows_put, dim3(p.blocks), dim3(kWG), 0, s, p);
        LAUNCH_CHECK("k_rows_put");
        urb_advance(*b, nrows);
        return counters_advance(*b, nrows, 0, s);
    }
    int rc = rows_put(b->rows, src_fields, skip, nrows - skip, first, s);
    if (rc) return rc;
    urb_advance(*b, nrows);
    return MRB_OK;
}

/* Appends to `h` the `n` rows of uniform buffer `src` at logical positions first .. first + n - 1
 * (0 = oldest), in one launch. */
int mrb_urb_append_from(int64_t h, int64_t src, int64_t first_logical, int64_t n, void* stream) {
    GET_URB(b, h);
    auto from = find_urb(src);
    if (!from) return fail(MRB_EHANDLE, "unknown uniform buffer handle %lld", (long long)src);
    if (from.get() == b.get()) return fail(MRB_EINVAL, "source and destination are the same buffer");
    if (b->device_counters || from->device_counters)
        return fail(MRB_ESTATE, "a buffer-to-buffer append needs both buffers' counters on the host (device_counters 0)");
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (first_logical < 0) first_logical += from->count;
    if (first_logical < 0 || first_logical + n > from->count)
        return fail(MRB_EINVAL, "rows [%lld, %lld) outside the %lld stored rows", (long long)first_logical,
                    (long long)(first_logical + n), (long long)from->count);
    if (from->rows.nfields != b->rows.nfields) return fail(MRB_EINVAL, "buffers differ in their fields");
    for (int i = 0; i < b->rows.nfields; ++i)
        if (from->rows.bytes[i] != b->rows.bytes[i] || from->rows.stride[i] != b->rows.stride[i])
            return fail(MRB_EINVAL, "buffers differ in field %d (size or row layout)", i);
    const int64_t cap = b->rows.capacity;
    // source slot of the first row: logical -> physical as in get_item
    const int64_t t0 = from->count - from->head;
    const int64_t src_first = first_logical < t0 ? first_logical + from->head : first_logical - t0;
    const bool growing = b->count < cap && b->head == 0;
    const int64_t w = growing ? b->count : b->head;
    const int64_t skip = n > cap ? n - cap : 0;
    PutArgs p{};
    const void* io[MRB_MAX_FIELDS];
    for (int i = 0; i < b->rows.nfields; ++i) io[i] = from->rows.data[i];
    int rc = make_table(b->rows, io, n - skip, p.t);
    if (rc) return rc;
    p.capacity = cap;
    p.first_slot = (w + skip) % cap;
    p.src_capacity = from->rows.capacity;
    p.src_first = (src_first + skip) % from->rows.capacity;
    p.blocks = grid_for(p.t.prefix[p.t.nfields]);
    p.threads = kWG;
    launch_kernel(k_rows_put, dim3(p.blocks), dim3(kWG), 0, static_cast<hipStream_t>(stream), p);
    LAUNCH_CHECK("k_rows_put");
    urb_advance(*b, n);
    return MRB_OK;
}

static int urb_gather_impl(Urb& b, const int64_t* indices, int64_t fixed_slot, int64_t n, int64_t* out_indices,
                           void* const* dst_fields, hipStream_t s) {
    return gather_rows(b.rows, indices, fixed_slot, b.count, b.seed, b.calls, n, out_indices, dst_fields, b.err, s);
}

int mrb_urb_get_item(int64_t h, int64_t logical_index, void* const* dst_fields, void* stream) {
    GET_URB(b, h);
    int64_t i = logical_index;
    if (i < 0) i += b->count;
    if (i < 0 || i >= b->count)
        return fail(MRB_EINVAL, "index %lld outside the %lld stored rows", (long long)logical_index, (long long)b->count);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (b->device_counters) {
        // count and head are read on the device: the slot is worked out there and the gather takes it as a given index
        launch_kernel(k_urb_slots, dim3(1), dim3(kWG), 0, s, b->slots, b->seed, b->counters, (int64_t)1, logical_index, 1,
                      b->err);
        LAUNCH_CHECK("k_urb_slots");
        return gather_rows(b->rows, b->slots, -1, b->rows.capacity, b->seed, b->calls, 1, nullptr, dst_fields, b->err, s);
    }
    const int64_t t = b->count - b->head;
    const int64_t slot = i < t ? i + b->head : i - t;
    return urb_gather_impl(*b, nullptr, slot, 1, nullptr, dst_fields, s);
}

int mrb_urb_gather(int64_t h, const int64_t* indices, int64_t n, void* const* dst_fields, void* stream) {
    GET_URB(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (!indices) return fail(MRB_EINVAL, "indices is NULL");
    if (b->count <= 0) return fail(MRB_ESTATE, "gather from an empty buffer");
    if (b->device_counters)  // the row count is on the device: slots are checked against the capacity only
        return gather_rows(b->rows, indices, -1, b->rows.capacity, b->seed, b->calls, n, nullptr, dst_fields, b->err,
                           static_cast<hipStream_t>(stream));
    return urb_gather_impl(*b, indices, -1, n, nullptr, dst_fields, static_cast<hipStream_t>(stream));
}

int mrb_urb_sample(int64_t h, int64_t n, int64_t* out_indices, void* const* dst_fields, void* stream) {
    GET_URB(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (n > b->count)
        return fail(MRB_ESTATE, "sample size %lld exceeds the %lld stored rows", (long long)n, (long long)b->count);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (b->device_counters) {
        // count and the generator's call counter are read on the device: the slots are drawn there, the gather
        // takes them as given indices, and the call counter moves on there
        if (n > kUrbDrawMax)
            return fail(MRB_ESTATE, "with device_counters a sample takes at most %lld rows", (long long)kUrbDrawMax);
        launch_kernel(k_urb_slots, dim3(grid_exact((uint64_t)n)), dim3(kWG), 0, s, b->slots, b->seed, b->counters, n,
                      (int64_t)0, 0, b->err);
        LAUNCH_CHECK("k_urb_slots");
        int rc = gather_rows(b->rows, b->slots, -1, b->rows.capacity, b->seed, b->calls, n, out_indices, dst_fields, b->err, s);
        if (rc) return rc;
        b->calls += 1;
        return counters_advance(*b, 0, 1, s);
    }
    int rc = urb_gather_impl(*b, nullptr, -1, n, out_indices, dst_fields, s);
    if (rc) return rc;
    b->calls += 1;
    return MRB_OK;
}

int mrb_urb_seed(int64_t h, uint64_t seed) {
    GET_URB(b, h);
    if (b->device_counters) {
        const int rc = counters_from_device(*b);
        if (rc) return rc;
    }
    b->seed = seed;
    b->calls = 0;
    return b->device_counters ? counters_to_device(*b) : MRB_OK;
}

int mrb_urb_state(int64_t h, int32_t* count, int32_t* head) {
    GET_URB(b, h);
    if (b->device_counters) {  // the device's counters are the current ones (a graph replay advances only them)
        const int rc = counters_from_device(*b);
        if (rc) return rc;
    }
    if (count) *count = (int32_t)b->count;
    if (head) *head = (int32_t)b->head;
    return MRB_OK;
}

int mrb_urb_reset(int64_t h) {
    GET_URB(b, h);
    if (b->device_counters) {  // no stream to order it on: the counters come back, are reset and go out again
        int rc = counters_from_device(*b);
        if (rc) return rc;
        b->count = 0;
        return counters_to_device(*b);
    }
    b->count = 0;
    return MRB_OK;
}

int mrb_urb_check(int64_t h, uint32_t* flags, void* stream) {
    GET_URB(b, h);
    return read_and_clear_flags(b->err, flags, static_cast<hipStream_t>(stream));
}

int mrb_urb_field_ptr(int64_t h, int field, void** dev_ptr) {
    GET_URB(b, h);
    if (field < 0 || field >= b->rows.nfields || !dev_ptr) return fail(MRB_EINVAL, "bad field %d", field);
    *dev_ptr = b->rows.data[field];
    return MRB_OK;
}

int mrb_urb_destroy(int64_t h) {
    std::shared_ptr<Urb> b;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_urb.find(h);
        if (it == g_urb.end()) return fail(MRB_EHANDLE, "unknown uniform buffer handle %lld", (long long)h);
        b = it->second;
        g_urb.erase(it);
    }
    HIP_TRY(hipDeviceSynchronize());
    return MRB_OK;
}

/* ------------------------------------------------------------ prioritized */

int mrb_per_create(int64_t capacity, float alpha, int nfields, const int64_t* field_bytes, uint64_t seed,
                   int64_t* out_handle) {
    if (!out_handle) return fail(MRB_EINVAL, "out_handle is NULL");
    if (!(alpha >= 0.0f) || alpha > 16.0f) return fail(MRB_EINVAL, "alpha %g outside [0, 16]", (double)alpha);
    auto b = std::make_shared<Per>();
    int rc = rows_alloc(b->rows, capacity, nfields, field_bytes, kMaxpBehindErr + kMeetBehindMaxp + sizeof(Meet), &b->err);
    if (rc) return rc;
    while (b->leaves < capacity) {
        b->leaves <<= 1;
        b->depth += 1;
    }
    b->alpha = alpha;
    b->seed = seed;
    // Rebuild plan: a tree of at most 12 levels is one workgroup's work (the top). A taller one gets as few
    // rounds (launches of a wave per 256-node tile) below its top as possible, and every round takes the full
    // 8 levels, which leaves the top - one workgroup, the end of every call's chain of launches - as low as
    // it can be: up to 8 levels it is one tile and one pass, beyond that tiles, a barrier and a second pass.
    b->top_depth = b->depth < kTopMaxDepth ? b->depth : kTopMaxDepth;
    if (const int rest = b->depth - b->top_depth; rest > 0) {
        // (21 levels: a top one level deeper, 32 tiles, saves a whole round, i.e. a launch)
        b->nrounds = rest == kRoundLevels + 1 ? 1 : (rest + kRoundLevels - 1) / kRoundLevels;
        b->top_depth = b->depth - kRoundLevels * b->nrounds;
    }
    for (int r = 0, lo = b->depth; r < b->nrounds; ++r) {
        b->lo[r] = lo;
        b->g[r] = kRoundLevels;
        lo -= kRoundLevels;
    }
    const size_t nodes = 2 * (size_t)b->leaves;
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->sum), nodes * sizeof(float)));
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->mn), nodes * sizeof(float)));
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->stamp), (size_t)b->leaves * sizeof(unsigned long long)));
    // one allocation, behind the row table: the error word (16 bytes), the device copy of the counters (kernels find them behind the error
    // word), and kMaxpBehindErr bytes in the running max (16 bytes; a kernel that is given its address finds the
    // counters in front of it: counters_before)
    static_assert(16 + kCntWords * sizeof(int64_t) <= kMaxpBehindErr, "the counters end before the running max");
    // (and, behind it, what the workgroups of an update meet over: Meet)
    b->counters = reinterpret_cast<int64_t*>(b->err + 4);
    b->maxp = reinterpret_cast<float*>(reinterpret_cast<char*>(b->err) + kMaxpBehindErr);
    // update_priorities scratch, sized once: a call rarely names more entries than there are rows
    b->powered_cap = capacity < 4096 ? 4096 : (capacity > (1ll << 20) ? (1ll << 20) : capacity);
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->powered), (size_t)b->powered_cap * sizeof(float)));
    HIP_TRY(hipGetDevice(&b->device));
    float* unused = nullptr;
    rc = static_scratch(&unused);  // set-up of the allocation-free entry point for this device
    if (rc) return rc;
    HIP_TRY(hipMemset(b->sum, 0, nodes * sizeof(float)));
    HIP_TRY(hipMemset(b->stamp, 0, (size_t)b->leaves * sizeof(unsigned long long)));
    for (int r = 0; r < b->nrounds; ++r) {
        const size_t nblocks = (size_t)1 << (b->lo[r] - b->g[r]);
        HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->dirty[r]), nblocks * sizeof(uint32_t)));
        HIP_TRY(hipMemset(b->dirty[r], 0, nblocks * sizeof(uint32_t)));
    }
    if (b->depth >= 21) {
        // sparse plan: with thousands of leaf tiles a call with few entries is better driven by its entries (takes_sparse)
        b->s_g0 = b->depth - 20 < 4 ? 4 : (b->depth - 20 > 6 ? 6 : b->depth - 20);
        // k_tree_runs takes at most 20 levels; deeper trees go through a round of tiles first (at least two levels, so
        // that a lane's four nodes share a block)
        const int d2 = b->depth - b->s_g0, g = d2 <= 20 ? 0 : d2 - 20 < 2 ? 2 : d2 - 20;
        if (g) {
            b->s_lo[b->s_rounds] = d2;
            b->s_g[b->s_rounds++] = g;
        }
        b->s_lo[b->s_rounds] = d2 - g;
        b->s_g[b->s_rounds++] = kRoundLevels;
        for (int r = 0; r < b->s_rounds; ++r) {
            const size_t nblocks = (size_t)1 << (b->s_lo[r] - b->s_g[r]);
            HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->s_dirty[r]), nblocks * sizeof(uint32_t)));
            HIP_TRY(hipMemset(b->s_dirty[r], 0, nblocks * sizeof(uint32_t)));
        }
    }
    launch_kernel(k_fill_f32, dim3(grid_for(nodes)), dim3(kWG), 0, nullptr, b->mn, FLT_MAX, (uint64_t)nodes);
    LAUNCH_CHECK("k_fill_f32");
    const float one_then_zero[4] = {1.0f, 0.0f, 0.0f, 0.0f};  // the running max; the max a push in progress has seen
    HIP_TRY(hipMemcpy(b->maxp, one_then_zero, sizeof(one_then_zero), hipMemcpyHostToDevice));
    HIP_TRY(hipDeviceSynchronize());
    std::lock_guard<std::mutex> lk(g_mu);
    *out_handle = g_next++;
    g_per[*out_handle] = b;
    return MRB_OK;
}

// The push behind mrb_per_push and mrb_per_update_push. `after_update`: an update_priorities of this very call
// precedes the push on the stream and changed nodes anywhere in the tree, so a one-launch push rebuilds the
// whole top (see UpdateArgs::full_top); `lead`, if given, is that update's leaf round, still to be launched:
// the push's row copy rides along in it and the push's own tree work follows as the last launch.
struct LeadRound {
    UpdateArgs a;
};

static int per_push(Per* b, const void* const* src_fields, int64_t nrows, const float* opt_priorities, hipStream_t s,
                    const LeadRound* lead = nullptr) {
    if (nrows <= 0) return fail(MRB_EINVAL, "nrows %lld must be positive", (long long)nrows);
    if (nrows > 0x7fffffffll) return fail(MRB_EINVAL, "nrows %lld exceeds 2^31 - 1 rows per call", (long long)nrows);
    const int64_t cap = b->rows.capacity;
    if (b->device_counters && nrows > cap)
        return fail(MRB_ESTATE, "with device_counters a push takes at most capacity (%lld) rows", (long long)cap);
    const int64_t skip = nrows > cap ? nrows - cap : 0;  // rows overwritten within this very call
    const int64_t n = nrows - skip;
    const int64_t first = (b->pushes + skip) % cap;
    PutArgs put{};
    int rc = put_args(b->rows, src_fields, skip, n, first, put);
    if (rc) return rc;
    if (b->device_counters) {  // the kernels take the first slot from the device
        put.first_slot = -1;
        put.src_first = reinterpret_cast<int64_t>(b->counters);
    }
    if (ShortIo io{}; !lead && skip == 0 && n > 1 && takes_push_many(*b, first, n, opt_priorities != nullptr, put.blocks) && short_io(put.t, io)) {
        const hipError_t e = launch_push_many(b->rows.table, io, put.t, b->sum, b->mn, b->maxp, opt_priorities, first, n, b->depth,
                                              b->alpha, s);
        if (e != hipSuccess) return fail(MRB_EHIP, "launch k_push_many: %s", hipGetErrorString(e));
        b->pushes += nrows;
        b->size = b->size + nrows < cap ? b->size + nrows : cap;
        return MRB_OK;
    }
    // A large copy gets its own launch; a small one rides along in the first tree launch.
    if (put.blocks > 2048u) {
        if (ShortIo io{}; !b->device_counters && short_io(put.t, io)) {
            const hipError_t e = launch_short_put(b->rows.table, io, put.t, first, n, s);
            if (e != hipSuccess) return fail(MRB_EHIP, "launch k_short_put: %s", hipGetErrorString(e));
        } else {
            launch_kernel(k_rows_put, dim3(put.blocks), dim3(kWG), 0, s, put);
            LAUNCH_CHECK("k_rows_put");
        }
        put.blocks = 0;
    }
    if (lead) {
        // the update's leaf round (a wave or two per entry), with this push's row copy as further workgroups
        const uint32_t waves = (lead->a.n > kPairedAbove ? 2u : 1u) * (uint32_t)lead->a.n;
        UpdateArgs la = lead->a;
        la.tile_blocks = (waves + 3) / 4;
        launch_kernel(k_tree_update, dim3(la.tile_blocks + put.blocks), dim3(kWG), 0, s, la.indices, la.priorities, la.sum,
                      la.mn, la.n, la.capacity, 0 | la.lo[0] << 8 | la.g[0] << 16, la.alpha, la, 0u, put);
        LAUNCH_CHECK("k_tree_update");
        put.blocks = 0;
    }
    rc = next_epoch(*b, s);
    if (rc) return rc;
    UpdateArgs a = update_args(*b);
    a.full_top = lead ? 1 : 0;
    // push-then-update: the running max sees every priority of the call, surviving or not, and is
    // raised only after the tree work (a fresh slot with an invalid priority keeps the old running max).
    // Few rows on a tree whose leaves the top workgroup rebuilds: it scans the priorities itself. Otherwise the
    // leaf-level waves, which compute every p^alpha anyway, collect their max beside the running max and the top
    // workgroup folds it in.
    // Only a call that overwrites rows of its own (more rows than capacity) needs a pass over all priorities.
    a.first_slot = b->device_counters ? -1 : first;
    a.n = n;
    const bool run = run_units(*b, a) != 0;
    const int fold = !opt_priorities ? 0
                     : (skip == 0 && nrows <= 1024 && !run) ? 1
                     : (skip == 0 && (run || a.nrounds > 0)) ? 2 : 0;
    if (opt_priorities) {
        a.priorities = opt_priorities + skip;
        a.fold_max = fold;
    }
    a.advance = b->device_counters ? nrows : 0;  // the call's last launch moves the device's counters on
    const bool stamp_after = opt_priorities && !fold;
    if (!lead && b->fused && nrows == 1 && b->depth <= kPushOneMaxDepth) {
        // one row: one wave walks from its leaf to the root (k_push_one)
        rc = ride_alone_if_large(a, put, s);
        if (rc) return rc;
        if (ShortIo io{}; put.blocks && !b->device_counters && short_io(put.t, io)) {
            const hipError_t e = launch_short_push_one(b->rows.table, io, put.t.nfields, a.sum, a.mn, a.maxp, a.first_slot, a.depth,
                                                       a.alpha, opt_priorities, most_granules(put.t), s);
            if (e != hipSuccess) return fail(MRB_EHIP, "launch k_short_push_one: %s", hipGetErrorString(e));
        } else {
            launch_kernel(b->device_counters ? k_push_one<true> : k_push_one<false>, dim3(1 + put.blocks), dim3(kWG), 0, s,
                          a.sum, a.mn, a.maxp, a.first_slot, a.capacity, a.leaves, a.depth, a.alpha, opt_priorities, a.err, put,
                          a.advance, 1 + put.blocks * (kWG / 64));
            LAUNCH_CHECK("k_push_one");
        }
        b->pushes += nrows;
        b->size = b->size + nrows < cap ? b->size + nrows : cap;
        return MRB_OK;
    }
    rc = tree_rebuild(*b, a, s, put.blocks ? &put : nullptr);
    if (rc) return rc;
    if (stamp_after) {
        a.priorities = opt_priorities;
        a.n = nrows;
        // (no indices: nothing to elect, the priorities are looked at and folded into the running max)
        launch_kernel(k_update_stamp, dim3(grid_exact((uint64_t)nrows)), dim3(kWG), 0, s, a.indices, a.priorities, a.stamp, a.powered, a.maxp,
                      (uint32_t)a.n, (uint32_t)a.capacity, a.epoch, a.alpha, static_cast<uint32_t*>(nullptr), 0);
        LAUNCH_CHECK("k_update_stamp");
    }
    b->pushes += nrows;
    b->size = b->size + nrows < cap ? b->size + nrows : cap;
    return MRB_OK;
}

int mrb_per_push(int64_t h, const void* const* src_fields, int64_t nrows, const float* opt_priorities, void* stream) {
    GET_PER(b, h);
    return per_push(b.get(), src_fields, nrows, opt_priorities, static_cast<hipStream_t>(stream));
}

int mrb_per_update(int64_t h, const int64_t* indices, const float* priorities, int64_t n, void* stream) {
    GET_PER(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (n > 0xffffffffll) return fail(MRB_EINVAL, "n %lld exceeds 2^32 - 1 entries per call", (long long)n);
    if (!indices || !priorities) return fail(MRB_EINVAL, "indices or priorities is NULL");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n > b->powered_cap) {
        // more entries than any call so far (and than the capacity): a larger array, at least twice the
        // old one; the old one stays allocated, kernels already queued may still use it
        const int64_t want = n > 2 * b->powered_cap ? n : 2 * b->powered_cap;
        float* bigger = nullptr;
        HIP_TRY(hipMalloc(reinterpret_cast<void**>(&bigger), (size_t)want * sizeof(float)));
        if (b->powered) b->retired.push_back(b->powered);
        b->powered = bigger;
        b->powered_cap = want;
    }
    return per_update(*b, indices, priorities, n, b->powered, s);
}

int mrb_per_update_noalloc(int64_t h, const int64_t* indices, const float* priorities, int64_t n, void* stream) {
    GET_PER(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (n > kNoAllocMaxEntries)
        return fail(MRB_EINVAL, "n %lld exceeds the %lld entries the static scratch holds; use mrb_per_update",
                    (long long)n, (long long)kNoAllocMaxEntries);
    if (!indices || !priorities) return fail(MRB_EINVAL, "indices or priorities is NULL");
    float* powered = nullptr;
    int rc = static_scratch(&powered);
    if (rc) return rc;
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev != b->device) return fail(MRB_ESTATE, "the buffer lives on device %d, the current device is %d", b->device, dev);
    return per_update(*b, indices, priorities, n, powered, static_cast<hipStream_t>(stream));
}

// Leaf tiles a push of n rows can meet when its first slot is known (no wrap) or only known on the device.
static uint32_t push_tiles(const Per& b, int64_t first, int64_t n) {
    if (b.device_counters) {
        UpdateArgs t{};
        t.capacity = b.rows.capacity;
        t.n = n;
        return push_units(t);
    }
    if (first + n > b.rows.capacity) return 0xffffffffu;  // wraps: not a single run of tiles
    return (uint32_t)((first + n - 1) / kBlockNodes) - (uint32_t)(first / kBlockNodes) + 1;
}

int mrb_per_update_push(int64_t h, const int64_t* indices, const float* priorities, int64_t n,
                        const void* const* src_fields, int64_t nrows, const float* opt_push_priorities, void* stream) {
    GET_PER(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (n > 0xffffffffll) return fail(MRB_EINVAL, "n %lld exceeds 2^32 - 1 entries per call", (long long)n);
    if (!indices || !priorities) return fail(MRB_EINVAL, "indices or priorities is NULL");
    if (nrows <= 0) return fail(MRB_EINVAL, "nrows %lld must be positive", (long long)nrows);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t cap = b->rows.capacity;
    const bool small_push = nrows <= cap && b->fused;
    // (1) one launch: the update by runs of leaves, whose workgroups also write the pushed rows' leaves; the ring's position
    // has to be the host's, and given priorities one run's
    if (small_push && !b->device_counters && nrows <= kOneMostRows && n <= kElectMax && takes_range_one(*b, n)) {
        const int64_t first = b->pushes % cap, last = first + nrows - 1;
        const int w = range_one_levels(b->depth, n);
        PutArgs put{};
        int rc = put_args(b->rows, src_fields, 0, nrows, first, put);
        if (rc) return rc;
        if (put.blocks <= kOneMostRiders && (!opt_push_priorities || (last < cap && first >> w == last >> w))) {
            const RangePush push{opt_push_priorities, (uint32_t)first, (uint32_t)nrows};
            const hipError_t e = launch_range_one_push(indices, priorities, n, b->sum, b->mn, b->maxp, cap, b->depth, b->alpha, push, put, s);
            if (e != hipSuccess) return fail(MRB_EHIP, "launch k_range_one_push: %s", hipGetErrorString(e));
            b->pushes += nrows;
            b->size = b->size + nrows < cap ? b->size + nrows : cap;
            return MRB_OK;
        }
    }
    // (2) one launch: the one-workgroup or one-wave update, then the walk of the one pushed row by the same workgroup
    const bool wg = n <= kWgBestEntries && b->depth >= 2 && b->depth <= kWgMaxDepth;
    const bool paths = n <= kPathEntries && b->depth <= kPathMaxDepth && b->depth >= 2;
    if (small_push && nrows == 1 && (wg || paths) && b->depth <= kPushOneMaxDepth) {
        if (!src_fields) return fail(MRB_EINVAL, "field pointer array is NULL");
        PutArgs put{};
        const int64_t first = b->pushes % cap;
        int rc = put_args(b->rows, src_fields, 0, 1, first, put);
        if (rc) return rc;
        if (b->device_counters) {
            put.first_slot = -1;
            put.src_first = reinterpret_cast<int64_t>(b->counters);
        }
        if (put.blocks <= (b->device_counters ? kRideWithCounters : 2048u)) {
            rc = next_epoch(*b, s);
            if (rc) return rc;
            UpdateArgs a = update_args(*b);
            a.indices = indices;
            a.priorities = priorities;
            a.n = n;
            a.advance = b->device_counters ? 1 : 0;
            const int64_t slot = b->device_counters ? -1 : first;
            // (readers: the waves that read the device's counters - the tree wave and every wave of the row copy)
            if (wg) {
                // (65 to 128 entries: 1024 threads, eight per entry - the kernel's one-step path below the staged top)
        const uint32_t threads = n > 64 && n <= 128 ? 1024u : n <= kWgMinThreads ? (uint32_t)kWgMinThreads : (uint32_t)((n + 63) / 64 * 64);
                a.readers = 1 + put.blocks * (threads / 64);
                put.threads = threads;
                launch_kernel(b->device_counters ? k_tree_wg_push<true> : k_tree_wg_push<false>, dim3(1 + put.blocks),
                              dim3(threads), 0, s, a.indices, a.priorities, a.sum, a.mn, a.maxp, (int)a.n,
                              a.depth | (int)threads << 8,
                              (int)a.capacity, a.alpha, a, slot, opt_push_priorities, put);
                LAUNCH_CHECK("k_tree_wg_push");
            } else {
                a.readers = 1 + put.blocks * (kWG / 64);
                launch_kernel(b->device_counters ? k_tree_paths_push<true> : k_tree_paths_push<false>, dim3(1 + put.blocks),
                              dim3(kWG), 0, s, a, slot, opt_push_priorities, put);
                LAUNCH_CHECK("k_tree_paths_push");
            }
            b->pushes += 1;
            b->size = b->size + 1 < cap ? b->size + 1 : cap;
            return MRB_OK;
        }
    }
    // (3) two launches on a tree with one round of levels below its top: the update's leaf round with the push's
    // row copy riding along, then one workgroup that rebuilds the pushed slots' leaf tiles and the whole top
    if (small_push && b->nrounds == 1 && n <= kElectMax && n > kFusedWG / 64 && b->depth >= 2 &&
        push_tiles(*b, b->pushes % cap, nrows) <= (uint32_t)kRunWaves) {
        int rc = next_epoch(*b, s);
        if (rc) return rc;
        LeadRound lead{update_args(*b)};
        lead.a.indices = indices;
        lead.a.priorities = priorities;
        lead.a.n = n;
        lead.a.inline_election = 1;
        return per_push(b.get(), src_fields, nrows, opt_push_priorities, s, &lead);
    }
    // (4) otherwise: the two calls, one after the other
    int rc = mrb_per_update(h, indices, priorities, n, stream);
    if (rc) return rc;
    return per_push(b.get(), src_fields, nrows, opt_push_priorities, s);
}

// Whether a sample of `rows` rows (of all its batches) goes to the LDS-top kernel, and the strata of a workgroup there;
// `rest` is what a row costs it to copy (see k_per_sample_lds). A wave per row carries a row faster, a thread per stratum
// walks the tree faster, so the line rises with the row's size. Measured, us, wave (workgroup) per row / LDS-top:
//   8-byte rows, 2^24 slots   2048 rows 6.8 / 6.1, 4096 8.6 / 6.1, 16,384 23 / 6.1
//   153 bytes, 10^6           2048 rows 6.6 / 7.3, 3000 7.4 / 7.4, 4096 8.9 / 7.3, 16,384 22 / 7.9, 65,536 71 / 13.3
//   521 bytes, 2^20           4096 rows 8.3 / 8.9, 6000 11.8 / 9.5, 16,384 22 / 11.1
//   (sixteen lanes, or a wave, / LDS-top)   8192 rows       10,240          12,288          14,336          16,384          20,480
//   2.4 KB, 2 * 10^5                       12.3 / 13.2     15.4 / 14.8     16.3 / 15.6     21.2 / 18.0     22.2 / 18.8     24.3 / 21.9
//   3 KB                                   13.9 / 13.2     16.7 / 15.8     17.8 / 16.9     22.6 / 19.4     23.7 / 20.7     26.5 / 24.5
//   3.5 KB in an odd field and others      17.6 / 16.6     21.5 / 20.4     22.4 / 21.1     31.5 / 25.5     32.5 / 26.3     35.6 / 31.3
//   4 KB                                   16.7 / 15.9     19.7 / 19.1     21.2 / 20.5     28.7 / 24.1     29.8 / 25.5     33.1 / 31.3
//   6 KB                                   21.8 / 20.4     26.7 / 26.0     30.0 / 27.7     34.4 / 33.0     37.4 / 34.7     45.0 / 41.9
// (The line of 12,288 was drawn before large fields had a loop of their own; 3 to 6 % from 8192 rows on are left there.)
// and 16 / 32 / 64 / 256 strata to a workgroup: 153 bytes, 16,384 rows 8.5 / 7.9 / 8.7 / 16.1, 65,536 25 / 17 / 13.3 /
// 16.7, 262,144 84 / 51 / 38 / 31; 521 bytes, 8192 rows 9.6 / 10.7 / 14.0 / 34.5, 32,768 21 / 13.8 / 16.8 / 36; 1 KB, 20,480 rows 13.0 / 12.5 / 13.0 /
// 21.9, 131,072 70 / 50 / 46 / 43; 3 KB, 12,288 rows 16.9 / 17.6 / 20.4 / 51, 32,768 38.0 / 34.8 / 34.5 / 58, 65,536 67.5 / 64.8 / 62.6 / 69.6.
// A workgroup has the strata of one batch only, so batches of a few rows leave most of it idle while it stages the top all
// the same (batches x rows of one): 8-byte rows, 10^6 slots 4096 x 1 6.6 / 20, 4096 x 2 11.0 / 20.6, 2048 x 4 10.9 / 12.1,
// 2048 x 6 14.6 / 9.9, 1024 x 8 10.8 / 6.4. (By sixteen lanes rows of 521 bytes and more lose nothing to small batches: 521 bytes
// 2048 x 4 6.3 / 12.7, 4096 x 5 13.0 / 22.6, 3 KB 4096 x 3 18.1 / 30.1, 4096 x 6 31.2 / 39.3, 2048 x 8 24.0 / 25.7, 6 KB 4096 x 3 30.4 / 40.8, 2048 x 8
// 38.1 / 39.0. The fewest rows of a batch were drawn before there were these, and let 4096 x 5 and the rows of 6 KB through.)
// `lanes`: whether sixteen lanes to a stratum could take it (takes_lanes), which are the better ones longer than a wave is. us,
// LDS-top / lanes:
//   row        slots       8192 rows      10,240        12,288        14,336        16,384        18,000        20,480
//   8 bytes    2 * 10^5     4.7 / 4.4     4.7 / 4.9     4.7 / 5.1     4.7 / 5.8
//   8          10^6         5.1 / 4.5     5.3 / 4.9     5.2 / 5.1     5.3 / 5.8
//   41         5 * 10^4     6.0 / 4.1     5.9 / 4.9     6.0 / 5.0     6.0 / 5.7     5.9 / 5.9     6.1 / 6.8     6.1 / 6.9
//   41         4 * 10^6     6.8 / 5.5     7.0 / 6.4     7.0 / 6.5     7.0 / 7.8     7.0 / 7.9
//   145        5 * 10^4     5.7 / 4.4     5.7 / 5.6     5.8 / 5.7     5.9 / 6.3     5.9 / 6.6
//   145        10^6         6.9 / 5.3     7.2 / 6.1     7.3 / 6.2     7.3 / 7.1     7.5 / 7.3     7.8 / 9.6
//   521        5 * 10^4     7.4 / 5.0     7.7 / 6.3     8.1 / 6.6     8.2 / 7.4     8.4 / 7.7     9.2 / 9.1     9.6 / 10.3
//   521        4 * 10^6     9.2 / 6.0     9.8 / 7.3    10.2 / 7.7    10.7 / 9.0    10.9 / 9.2    11.6 / 11.3   11.8 / 11.8
//   899        2 * 10^5                                 9.8 / 9.5                  10.8 / 14.2
//   1 KB       2 * 10^5                                18.9 / 10.9 (a wave's)      12.4 / 14.2
// (Of rows with nothing but scalars the line, 14,336, is right for some trees and 5 % off for others.)
static bool takes_lds(int64_t nbatch, int64_t batch, uint64_t rest, bool lanes) {
    const int64_t rows = nbatch * batch, fewest = rest <= 64 ? 5 : rest <= 256 ? 8 : 1;
    const int64_t least = lanes ? (rest <= 16 ? 14336 : rest <= 40 ? 20480 : 12288) : (rest <= 16 ? 3072 : rest <= 64 ? 5120 : 12288);
    return rest <= 384 && batch >= fewest && rows >= least;
}
// Whether sixteen lanes to a stratum (k_per_sample_lanes) can take a sample.
static bool takes_lanes(const Per& b, const WidePlan& plan) {
    return b.rows.row_split == 0 && b.rows.row_wave == 0 && b.depth >= kLanesFewestLevels && plan.narrow_items <= kLanesMostNarrow &&
           plan.wide_items <= 1280;
}
// Whether they are faster than a workgroup to a row (k_per_sample_light, k_per_sample_wide). That one's time hardly depends on the row
// but on how it walks the tree: on 20 levels in two groups of ten, which is its best, on 22 by the larger kernel, which is its worst.
// us, it / lanes (byte images, masks and halves: 147 and 899 bytes; the others rows of floats):
//   levels  row          1024 rows      1280           1536           1792           2048
//   16      41 bytes     3.8 / 3.5      4.1 / 3.5      4.4 / 3.5      4.5 / 3.5      5.7 / 3.5
//   16      521          3.8 / 4.0      4.1 / 4.0      4.5 / 4.0      4.8 / 4.0      6.1 / 4.1
//   16      899          3.9 / 4.6      4.4 / 4.7      4.8 / 4.7      5.2 / 4.7      6.9 / 4.8
//   18      41           3.8 / 4.0      4.1 / 4.0      4.5 / 4.0      4.7 / 4.0      6.1 / 4.0
//   18      147          3.8 / 4.3      4.2 / 4.3      4.6 / 4.3      4.8 / 4.3      6.2 / 4.4      (1408: 4.5 / 4.3)
//   18      899          4.0 / 5.0      4.4 / 5.0      4.9 / 5.0      5.3 / 5.1      7.0 / 5.1
//   20      41           3.6 / 4.2      3.8 / 4.2      4.3 / 4.2      4.5 / 4.2      5.8 / 4.2
//   20      147          3.6 / 4.6      3.9 / 4.6      4.4 / 4.6      4.6 / 4.6      5.9 / 4.6
//   20      521          3.6 / 4.4      3.9 / 4.4      4.4 / 4.4      4.6 / 4.4      5.9 / 4.6
//   20      899          4.0 / 5.1      4.4 / 5.1      4.7 / 5.1      5.1 / 5.2      6.7 / 5.3      (1920: 5.2 / 5.2)
//   21      147          4.9 / 4.9      5.3 / 4.9      5.7 / 4.9      6.1 / 4.9      6.9 / 5.0      (768: 4.6 / 4.9; 41 bytes 4.6 / 4.6)
//   21      899          5.2 / 5.3      5.8 / 5.4      6.2 / 5.4      6.6 / 5.5      7.7 / 5.6
//   22      147          5.4 / 4.9      5.8 / 4.9      7.6 / 4.9      8.6 / 5.0      7.0 / 5.0      (768: 4.9 / 5.0, 521 bytes 4.9 / 4.6; 512: 4.5 / 4.6)
//   24      41           4.5 / 4.8      5.0 / 4.8      5.3 / 4.8      5.5 / 4.8      6.9 / 4.8
//   24      147          4.6 / 5.2      5.1 / 5.2      5.4 / 5.2      5.7 / 5.3      7.0 / 5.3
//   26      41           4.7 / 5.4      5.2 / 5.4      5.6 / 5.5      5.8 / 5.5      7.1 / 5.5
// Rows that waves carry whole (above a kilobyte): lanes from 2048 rows on, but not where their launch is more workgroups than the chip holds
// at once and fills little of the second lot; both sides are in the table at lanes_strata (mrb_sample_lanes.hip).
static bool lanes_better(int depth, uint32_t wide, uint32_t narrow, int64_t rows) {
    if (wide > 64) {
        if (rows < 2048) return false;
        if (wide <= 192 || (wide > 256 && wide <= 512)) return true;
        return wide <= 256 ? rows <= 4096 || rows >= 5632 : rows <= 2048 || (rows >= 3600 && rows <= 4096) || rows >= 6000;
    }
    const bool light = wide <= 16 && narrow <= 16;  // a granule and a byte to a lane: 0.2 us less
    if (depth % kGroupMaxLevels == 0) return rows >= (light ? 1408 : wide <= 32 ? 1664 : 1920);
    if (depth == 21 || depth == 22) return rows >= (depth == 22 || wide <= 32 ? 1024 : 1280);
    if (depth < 18) return rows >= (wide <= 32 ? 1280 : 1536);
    return rows >= (light ? 1280 : wide <= 32 ? 1408 : 1664);
}
static int lds_strata(int64_t rows, uint64_t rest) {
    if (rows <= 20480 && rest > 16) return 16;
    return rows <= 40960 ? 32 : rows <= 98304 || rest > 64 ? 64 : 256;
}

// `nbatch` batches of `batch` stratified samples each, as nbatch successive mrb_per_sample calls on
// an unchanged tree would draw them. Outputs hold nbatch * batch rows, batch after batch.
static int per_sample_impl(Per* b, int64_t nbatch, int64_t batch, float beta, const float* uniforms,
                           int64_t* out_indices, float* out_weights, void* const* out_fields, hipStream_t s,
                           const NextRows* next = nullptr) {
    if (batch <= 0 || batch > (1ll << 24)) return fail(MRB_EINVAL, "batch %lld outside [1, 2^24]", (long long)batch);
    if (nbatch <= 0 || nbatch > 4096 || nbatch * batch > (1ll << 24))
        return fail(MRB_EINVAL, "%lld batches of %lld rows exceed one call (at most 4096 batches, 2^24 rows)",
                    (long long)nbatch, (long long)batch);
    if (!out_indices || !out_weights) return fail(MRB_EINVAL, "out_indices or out_weights is NULL");
    if (b->size <= 0) return fail(MRB_ESTATE, "sample from an empty buffer");
    IoTable t;
    int rc = make_table(b->rows, out_fields, nbatch * batch, t);
    if (rc) return rc;
    SampleArgs a{};
    a.sum = b->sum;
    a.mn = b->mn;
    a.depth = b->depth;
    a.leaves = b->leaves;
    a.capacity = b->rows.capacity;
    a.size = b->size;
    a.batch = batch;
    a.beta = beta;
    a.uniforms = uniforms;
    a.seed = b->seed;
    a.calls = b->calls;
    a.out_idx = out_indices;
    a.out_w = out_weights;
    a.err = b->err;
    if (b->device_counters) {
        a.size = -1;  // the kernels take the number of stored rows from the device
        // the generator's call counter is on the device too: the kernels read it there and add the number of the
        // batch (see generator_calls)
        if (!uniforms) a.calls = 0;
    }
    uint64_t rest = 0;  // granules of a row that the LDS-top kernel's threads do not copy for their own stratum alone
    for (int f = 0; f < t.nfields; ++f) rest += f < kLdsOwn && t.units[f] == 1 ? 0 : t.units[f];
    int path = (int)b->sample_path;
    if (path == 0) {
        WidePlan plan;
        dim3 grid;
        plan.nbatch = (uint32_t)nbatch;
        const bool lanes = !next && nbatch * batch >= 1024 && wide_plan(b->rows, t, nbatch * batch, plan, grid) && takes_lanes(*b, plan);
        path = takes_lds(nbatch, batch, rest, lanes) ? 2 : lanes && lanes_better(b->depth, plan.wide_items, plan.narrow_items, nbatch * batch) ? 3 : 1;
        if (path == 3) {
            const hipError_t e = launch_per_sample_lanes(a, plan, nbatch, s);
            if (e != hipSuccess) return fail(MRB_EHIP, "launch k_per_sample_lanes: %s", hipGetErrorString(e));
        }
    }
    if (rest > 1u << 23) path = 1;  // (it numbers a workgroup's granules in 32 bits)
    if (next) {
        rc = sample_wide(b->rows, a, t, nbatch, s, next);  // always the wide-row kernel: the gathered field is wide
        if (rc) return rc;
    } else if (path == 1) {
        rc = sample_wide(b->rows, a, t, nbatch, s);
        if (rc) return rc;
    } else if (path == 2) {
        int levels = b->lds_levels > 0 ? (int)b->lds_levels : 9;
        if (levels > b->depth) levels = b->depth;
        if (has_silent(b->depth)) levels = std::min(levels, b->depth - kSilentLevels - 1);
        const hipError_t e = launch_per_sample_lds(a, t, nbatch, lds_strata(nbatch * batch, rest), levels, (uint32_t)rest, s);
        if (e != hipSuccess) return fail(MRB_EHIP, "launch k_per_sample_lds: %s", hipGetErrorString(e));
    }
    if (!uniforms) {
        b->calls += (uint64_t)nbatch;
        if (b->device_counters) return counters_advance(*b, 0, nbatch, s);
    }
    return MRB_OK;
}

int mrb_per_sample(int64_t h, int64_t batch, float beta, const float* uniforms, int64_t* out_indices,
                   float* out_weights, void* const* out_fields, void* stream) {
    GET_PER(b, h);
    return per_sample_impl(b.get(), 1, batch, beta, uniforms, out_indices, out_weights, out_fields,
                           static_cast<hipStream_t>(stream));
}

int mrb_per_sample_many(int64_t h, int64_t nbatch, int64_t batch, float beta, const float* uniforms,
                        int64_t* out_indices, float* out_weights, void* const* out_fields, void* stream) {
    GET_PER(b, h);
    return per_sample_impl(b.get(), nbatch, batch, beta, uniforms, out_indices, out_weights, out_fields,
                           static_cast<hipStream_t>(stream));
}

int mrb_per_update_push_sample(int64_t h, const int64_t* indices, const float* priorities, int64_t n,
                               const void* const* src_fields, int64_t nrows, const float* opt_push_priorities,
                               int64_t batch, float beta, const float* uniforms, int64_t* out_indices,
                               float* out_weights, void* const* out_fields, void* stream) {
    GET_PER(b, h);
    // (everything the three calls would refuse is refused before the first of them runs)
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (!indices || !priorities) return fail(MRB_EINVAL, "indices or priorities is NULL");
    if (nrows <= 0) return fail(MRB_EINVAL, "nrows %lld must be positive", (long long)nrows);
    if (!src_fields) return fail(MRB_EINVAL, "field pointer array is NULL");
    if (batch <= 0 || batch > (1ll << 24)) return fail(MRB_EINVAL, "batch %lld outside [1, 2^24]", (long long)batch);
    if (!out_indices || !out_weights) return fail(MRB_EINVAL, "out_indices or out_weights is NULL");
    IoTable t;
    int rc = make_table(b->rows, out_fields, batch, t);
    if (rc) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t cap = b->rows.capacity;
    // one launch of one workgroup: the update of at most 384 entries on a tree of at most 14 levels, one row, a batch
    // of at most a thread per stratum, and rows small enough for one workgroup to copy; the counters on the host
    if (b->fused && b->sample_path == 0 && nrows == 1 && n <= kWgBestEntries && b->depth >= 2 &&
        b->depth <= kWgMaxDepth && batch <= kStepThreads) {
        PutArgs put{};
        const int64_t first = b->pushes % cap;
        rc = put_args(b->rows, src_fields, 0, 1, first, put);
        if (rc) return rc;
        if (put.t.prefix[put.t.nfields] <= kStepMaxPut && t.prefix[t.nfields] <= kStepMaxGather) {
            rc = next_epoch(*b, s);
            if (rc) return rc;
            UpdateArgs a = update_args(*b);
            a.indices = indices;
            a.priorities = priorities;
            a.n = n;
            StepLate late{};
            late.err = b->err;
            late.priority = opt_push_priorities;
            late.uniforms = uniforms;
            late.out_idx = out_indices;
            late.out_w = out_weights;
            late.size = b->size + 1 < cap ? b->size + 1 : cap;  // as the push leaves it
            late.seed = b->seed;
            late.calls = b->calls;
            late.beta = beta;
            late.put = put.t;
            late.get = t;
            // (with device_counters the kernel takes the slot, the row count and the generator's call counter from the
            // device and moves them on itself)
            const bool wide = n > 64 && n <= 128;  // 1024 threads, eight per entry (see k_tree_wg)
            auto* const kernel = b->device_counters ? (wide ? k_tree_wg_push_sample<true, 1024> : k_tree_wg_push_sample<true, kStepThreads>)
                                                    : (wide ? k_tree_wg_push_sample<false, 1024> : k_tree_wg_push_sample<false, kStepThreads>);
            launch_kernel(kernel, dim3(1), dim3(wide ? 1024 : kStepThreads), 0, s, indices, priorities, b->sum, b->mn, a.maxp,
                          (int)(cap << 16 | (b->device_counters ? 0 : first)), (int)(n << 18 | batch << 8) | b->depth, a.alpha,
                          late);
            LAUNCH_CHECK("k_tree_wg_push_sample");
            b->pushes += 1;
            b->size = late.size;
            if (!uniforms) b->calls += 1;
            return MRB_OK;
        }
    }
    rc = mrb_per_update_push(h, indices, priorities, n, src_fields, nrows, opt_push_priorities, stream);
    if (rc) return rc;
    return per_sample_impl(b.get(), 1, batch, beta, uniforms, out_indices, out_weights, out_fields, s);
}

int mrb_per_sample_next(int64_t h, int64_t batch, float beta, const float* uniforms, int slot_field, int row_field,
                        int64_t* out_indices, float* out_weights, void* const* out_fields, void* out_next_rows,
                        void* stream) {
    GET_PER(b, h);
    const RowStore& r = b->rows;
    if (slot_field < 0 || slot_field >= r.nfields || r.bytes[slot_field] != 8)
        return fail(MRB_EINVAL, "slot_field %d must name a field of 8 bytes (one int64 slot number per row)", slot_field);
    if (row_field < 0 || row_field >= r.nfields || r.align_log2[row_field] != 4)
        return fail(MRB_EINVAL, "row_field %d must name a field whose rows are multiples of 16 bytes", row_field);
    if (!out_next_rows) return fail(MRB_EINVAL, "out_next_rows is NULL");
    if (reinterpret_cast<uintptr_t>(out_next_rows) & 15u) return fail(MRB_EINVAL, "out_next_rows %p is not 16-byte aligned", out_next_rows);
    const NextRows next{slot_field, row_field, out_next_rows};
    return per_sample_impl(b.get(), 1, batch, beta, uniforms, out_indices, out_weights, out_fields,
                           static_cast<hipStream_t>(stream), &next);
}

int mrb_per_gather(int64_t h, const int64_t* indices, int64_t n, void* const* dst_fields, void* stream) {
    GET_PER(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (!indices) return fail(MRB_EINVAL, "indices is NULL");
    if (b->size <= 0) return fail(MRB_ESTATE, "gather from an empty buffer");
    return gather_rows(b->rows, indices, -1, b->size, 0, 0, n, nullptr, dst_fields, b->err,
                       static_cast<hipStream_t>(stream));
}

int mrb_per_export_tree(int64_t h, float* sum_heap, float* min_heap, int64_t* leaves, void* stream) {
    GET_PER(b, h);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t bytes = 2 * (size_t)b->leaves * sizeof(float);
    HIP_TRY(hipStreamSynchronize(s));
    if (has_silent(b->depth) && (sum_heap || min_heap)) {
        // (whatever device is current, as for the copies; what the caller has queued is done)
        int device = 0;
        HIP_TRY(hipGetDevice(&device));
        if (device != b->device) HIP_TRY(hipSetDevice(b->device));
        hipError_t e = launch_tree_silent(b->sum, b->mn, b->leaves, nullptr);
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (device != b->device) (void)hipSetDevice(device);
        if (e != hipSuccess) return fail(MRB_EHIP, "launch k_tree_silent: %s", hipGetErrorString(e));
    }
    if (sum_heap) HIP_TRY(hipMemcpy(sum_heap, b->sum, bytes, hipMemcpyDeviceToHost));
    if (min_heap) HIP_TRY(hipMemcpy(min_heap, b->mn, bytes, hipMemcpyDeviceToHost));
    if (leaves) *leaves = b->leaves;
    return MRB_OK;
}

int mrb_per_state(int64_t h, int64_t* size, int64_t* head, float* max_priority, void* stream) {
    GET_PER(b, h);
    if (b->device_counters) {  // the device's counters are the current ones (a graph replay advances only them)
        const int rc = counters_from_device(*b);
        if (rc) return rc;
    }
    if (size) *size = b->size;
    if (head) *head = b->pushes % b->rows.capacity;
    if (max_priority) {
        hipStream_t s = static_cast<hipStream_t>(stream);
        HIP_TRY(hipMemcpyAsync(max_priority, b->maxp, sizeof(float), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    return MRB_OK;
}

int mrb_per_check(int64_t h, uint32_t* flags, void* stream) {
    GET_PER(b, h);
    return read_and_clear_flags(b->err, flags, static_cast<hipStream_t>(stream));
}

int mrb_per_field_ptr(int64_t h, int field, void** dev_ptr) {
    GET_PER(b, h);
    if (field < 0 || field >= b->rows.nfields || !dev_ptr) return fail(MRB_EINVAL, "bad field %d", field);
    *dev_ptr = b->rows.data[field];
    return MRB_OK;
}

int mrb_per_destroy(int64_t h) {
    std::shared_ptr<Per> b;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_per.find(h);
        if (it == g_per.end()) return fail(MRB_EHANDLE, "unknown priority buffer handle %lld", (long long)h);
        b = it->second;
        g_per.erase(it);
    }
    HIP_TRY(hipDeviceSynchronize());
    return MRB_OK;
}

/* -------------------------------------------------------------- reservoir */

int mrb_res_create(int64_t capacity, int nfields, const int64_t* field_bytes, uint64_t seed, int64_t* out_handle) {
    if (!out_handle) return fail(MRB_EINVAL, "out_handle is NULL");
    auto b = std::make_shared<Res>();
    int rc = rows_alloc(b->rows, capacity, nfields, field_bytes, 16, &b->err);
    if (rc) return rc;
    b->seed = seed;
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(&b->stamp), (size_t)capacity * sizeof(unsigned long long)));
    HIP_TRY(hipMemset(b->stamp, 0, (size_t)capacity * sizeof(unsigned long long)));
    HIP_TRY(hipDeviceSynchronize());  // as in mrb_urb_create
    std::lock_guard<std::mutex> lk(g_mu);
    *out_handle = g_next++;
    g_res[*out_handle] = b;
    return MRB_OK;
}

int mrb_res_push(int64_t h, const void* const* src_fields, int64_t nrows, void* stream) {
    GET_RES(b, h);
    if (nrows <= 0) return fail(MRB_EINVAL, "nrows %lld must be positive", (long long)nrows);
    if (nrows > 0x7fffffffll) return fail(MRB_EINVAL, "nrows %lld exceeds 2^31 - 1 rows per call", (long long)nrows);
    hipStream_t s = static_cast<hipStream_t>(stream);
    IoTable t;
    int rc = make_table(b->rows, src_fields, nrows, t);
    if (rc) return rc;
    const int64_t cap = b->rows.capacity;
    // Rows of one call can only collide on a slot once replacement has begun.
    const bool elect = nrows > 1 && b->total + nrows > cap;
    int64_t per_row = 0;
    for (int f = 0; f < t.nfields; ++f) per_row += t.units[f];
    if (const int rows = elect ? res_rows_per_workgroup(nrows, per_row, cap) : 0) {
        launch_kernel(k_res_push, dim3((uint32_t)((nrows + rows - 1) / rows)), dim3(kResWG), 0, s, b->total, cap, b->seed,
                      (int)nrows, rows, t.nfields, (uint32_t)per_row, t);
        LAUNCH_CHECK("k_res_push");
    } else {
        rc = res_push_by_stamps(*b, t, nrows, elect, s);
        if (rc) return rc;
    }
    b->total += nrows;
    b->size = b->total < cap ? b->total : cap;
    return MRB_OK;
}

int mrb_res_sample(int64_t h, int64_t n, int64_t* out_indices, void* const* dst_fields, void* stream) {
    GET_RES(b, h);
    if (n <= 0) return fail(MRB_EINVAL, "n %lld must be positive", (long long)n);
    if (b->size <= 0) return fail(MRB_ESTATE, "sample from an empty buffer");
    int rc = gather_rows(b->rows, nullptr, -1, b->size, b->seed, b->calls + 1, n, out_indices, dst_fields, b->err,
                         static_cast<hipStream_t>(stream));
    if (rc) return rc;
    b->calls += 1;
    return MRB_OK;
}

int mrb_res_state(int64_t h, int64_t* size, int64_t* total) {
    GET_RES(b, h);
    if (size) *size = b->size;
    if (total) *total = b->total;
    return MRB_OK;
}

int mrb_res_field_ptr(int64_t h, int field, void** dev_ptr) {
    GET_RES(b, h);
    if (field < 0 || field >= b->rows.nfields || !dev_ptr) return fail(MRB_EINVAL, "bad field %d", field);
    *dev_ptr = b->rows.data[field];
    return MRB_OK;
}

int mrb_res_destroy(int64_t h) {
    std::shared_ptr<Res> b;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_res.find(h);
        if (it == g_res.end()) return fail(MRB_EHANDLE, "unknown reservoir buffer handle %lld", (long long)h);
        b = it->second;
        g_res.erase(it);
    }
    HIP_TRY(hipDeviceSynchronize());
    return MRB_OK;
}

/* -------------------------------------------------------- checkpoint hooks */

int mrb_urb_get_counters(int64_t h, int64_t* out4) {
    GET_URB(b, h);
    if (!out4) return fail(MRB_EINVAL, "out4 is NULL");
    if (b->device_counters) {
        const int rc = counters_from_device(*b);
        if (rc) return rc;
    }
    out4[0] = b->count, out4[1] = b->head, out4[2] = (int64_t)b->seed, out4[3] = (int64_t)b->calls;
    return MRB_OK;
}

int mrb_urb_set_counters(int64_t h, const int64_t* in4) {
    GET_URB(b, h);
    if (!in4) return fail(MRB_EINVAL, "in4 is NULL");
    const int64_t cap = b->rows.capacity;
    if (in4[0] < 0 || in4[0] > cap || in4[1] < 0 || in4[1] >= cap)
        return fail(MRB_EINVAL, "count %lld / head %lld do not fit capacity %lld", (long long)in4[0], (long long)in4[1],
                    (long long)cap);
    b->count = in4[0], b->head = in4[1], b->seed = (uint64_t)in4[2], b->calls = (uint64_t)in4[3];
    return b->device_counters ? counters_to_device(*b) : MRB_OK;
}

int mrb_per_get_counters(int64_t h, int64_t* out4) {
    GET_PER(b, h);
    if (!out4) return fail(MRB_EINVAL, "out4 is NULL");
    if (b->device_counters) {
        const int rc = counters_from_device(*b);
        if (rc) return rc;
    }
    out4[0] = b->size, out4[1] = b->pushes, out4[2] = (int64_t)b->seed, out4[3] = (int64_t)b->calls;
    return MRB_OK;
}

int mrb_per_set_counters(int64_t h, const int64_t* in4) {
    GET_PER(b, h);
    if (!in4) return fail(MRB_EINVAL, "in4 is NULL");
    const int64_t cap = b->rows.capacity;
    const int64_t want = in4[1] < cap ? in4[1] : cap;
    if (in4[1] < 0 || in4[0] != want)
        return fail(MRB_EINVAL, "size %lld does not follow from %lld pushes into capacity %lld", (long long)in4[0],
                    (long long)in4[1], (long long)cap);
    b->size = in4[0], b->pushes = in4[1], b->seed = (uint64_t)in4[2], b->calls = (uint64_t)in4[3];
    return b->device_counters ? counters_to_device(*b) : MRB_OK;
}

int mrb_res_get_counters(int64_t h, int64_t* out4) {
    GET_RES(b, h);
    if (!out4) return fail(MRB_EINVAL, "out4 is NULL");
    out4[0] = b->size, out4[1] = b->total, out4[2] = (int64_t)b->seed, out4[3] = (int64_t)b->calls;
    return MRB_OK;
}

int mrb_res_set_counters(int64_t h, const int64_t* in4) {
    GET_RES(b, h);
    if (!in4) return fail(MRB_EINVAL, "in4 is NULL");
    const int64_t cap = b->rows.capacity;
    const int64_t want = in4[1] < cap ? in4[1] : cap;
    if (in4[1] < 0 || in4[0] != want)
        return fail(MRB_EINVAL, "size %lld does not follow from %lld rows pushed into capacity %lld", (long long)in4[0],
                    (long long)in4[1], (long long)cap);
    b->size = in4[0], b->total = in4[1], b->seed = (uint64_t)in4[2], b->calls = (uint64_t)in4[3];
    return MRB_OK;
}

int mrb_per_load_leaves(int64_t h, const float* leaves, int64_t n, float max_priority, void* stream) {
    GET_PER(b, h);
    if (n < 0 || n > b->rows.capacity) return fail(MRB_EINVAL, "n %lld outside [0, capacity]", (long long)n);
    if (n > 0 && !leaves) return fail(MRB_EINVAL, "leaves is NULL");
    if (!(max_priority >= 0.0f) || max_priority > 3.0e38f) return fail(MRB_EINVAL, "max_priority %g is not a priority", (double)max_priority);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t nodes = 2 * (size_t)b->leaves;
    fill_zero(b->sum, nodes * sizeof(float), s);
    launch_kernel(k_fill_f32, dim3(grid_for(nodes)), dim3(kWG), 0, s, b->mn, FLT_MAX, (uint64_t)nodes);
    LAUNCH_CHECK("k_fill_f32");
    launch_kernel(k_fill_f32, dim3(1), dim3(kWG), 0, s, b->maxp, max_priority, (uint64_t)1);
    LAUNCH_CHECK("k_fill_f32");
    if (n == 0) return MRB_OK;
    int rc = next_epoch(*b, s);
    if (rc) return rc;
    // a push of slots [0, n) whose priorities are taken as they are: x^1 == x exactly
    UpdateArgs a = update_args(*b);
    a.alpha = 1.0f;
    a.priorities = leaves;
    a.first_slot = 0;
    a.n = n;
    return tree_rebuild(*b, a, s);
}

/* ------------------------------------------------------------ measurement aids */

int mrb_bench_launch(int kind, void* dst, const void* src, int64_t bytes, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (kind == 0) {
        launch_kernel(k_nothing, dim3(1), dim3(64), 0, s);
        LAUNCH_CHECK("k_nothing");
        return MRB_OK;
    }
    if (kind == 1) {
        if (!dst || !src || bytes <= 0) return fail(MRB_EINVAL, "copy of %lld bytes from %p to %p", (long long)bytes, src, dst);
        HIP_TRY(hipMemcpyDtoDAsync(dst, const_cast<void*>(src), (size_t)bytes, s));
        return MRB_OK;
    }
    return fail(MRB_EINVAL, "unknown kind %d", kind);
}

/* ------------------------------------------------------- discounted return */

}  // extern "C"

// Both directions of the recurrence (see k_discounted_return): `end_value` is the bootstrap value in or, kBack, its
// gradient out (may be NULL).
template <bool kBack>
static int discounted_return(const float* x, const uint8_t* done, float* end_value, float* out, int64_t timesteps,
                             int64_t batch, int64_t inner, float gamma, hipStream_t s) {
    if (!x || !done || (!kBack && !end_value) || !out) return fail(MRB_EINVAL, "a data pointer is NULL");
    if (timesteps <= 0 || batch <= 0 || inner <= 0)
        return fail(MRB_EINVAL, "timesteps %lld, batch %lld, inner %lld must be positive", (long long)timesteps,
                    (long long)batch, (long long)inner);
    if (!(gamma >= 0.0f && gamma <= 1.0f))
        return fail(MRB_EINVAL, "The discounted factor should be a number in range [0, 1], but got %g.", (double)gamma);
    const int64_t cols = batch * inner;
    if (cols > (1ll << 31) || cols > (1ll << 40) / timesteps)
        return fail(MRB_EINVAL, "%lld columns of %lld steps exceed one call (at most 2^31 columns, 2^40 elements)",
                    (long long)cols, (long long)timesteps);
    // A thread per column needs about 65 to 100 ns per step however few the columns (a trip to memory per 32 steps, and steps beyond a
    // multiple of 32 cost it more) and streams at up to 6 TB/s when there are many; chunks of 64 steps through LDS need 8 to 11 ns per
    // step and stream at 4.8 TB/s. So the line rises with the steps beyond a multiple of 32, and falls back behind 64. us, forward, per
    // column / by chunks (backward the chunks gain up to 8 % on that):
    //   steps           16,384         20,000         24,000         30,000         36,000         40,960    chunks are faster up to
    //      20       4.8 /  5.0     4.9 /  5.6     4.9 /  6.6     5.0 /  7.8     5.1 /  8.9     5.1 /  9.7    16,000  (but the line is at 8192)
    //      33       4.4 /  5.3     4.8 /  5.9     4.7 /  6.9     4.9 /  8.1     5.0 /  9.3     4.8 / 10.2    12,000
    //      48       6.8 /  5.4     7.0 /  6.0     7.1 /  7.0     7.1 /  8.2     7.2 /  9.4     7.1 / 10.1    25,000
    //      60       8.8 /  5.5     8.9 /  6.1     8.9 /  7.2     9.2 /  8.3     9.3 /  9.4     9.2 / 10.3    38,000
    //      64       7.0 /  5.6     7.4 /  6.1     7.9 /  7.1     8.2 /  8.2     8.2 /  9.5     8.3 / 10.2    28,000  (backward 8.8 / 8.3 at 30,001)
    //      65       7.3 /  6.1     7.7 /  6.7     8.0 /  7.8     8.3 /  9.2     8.4 / 10.6     8.5 / 11.5    25,000
    //      80       9.4 /  6.1     9.9 /  6.8    10.0 /  7.9    10.6 /  9.3    11.1 / 10.6    10.3 / 11.4    38,000
    // Beyond 95 steps the line is flat. 45,000 columns: 104 steps 14.4 / 13.2, 128 16.7 / 15.4, 192 23.8 / 19.9; 50,000: 14.7 / 13.7,
    // 17.0 / 18.6, 24.4 / 23.5 (the line lies at 40,960, in front of what 128 steps lose and at the price of what 192 would gain);
    // 65,536: 256 steps 31.6 / 29.7, 300 38.5 / 34.3, 1000 122 / 117; 81,920: 256 37.7 / 36.0, 300 46.8 / 41.5 (the line lies at 65,536).
    const int64_t beyond = timesteps % 32;
    const int64_t most = timesteps <= 32   ? 8192
                         : timesteps < 64  ? 10000 + 900 * beyond
                         : timesteps == 64 ? 31000
                         : timesteps < 96  ? std::min<int64_t>(24000 + 900 * beyond, 40960)
                         : timesteps < 256 ? 40960
                                           : 65536;
    const bool per_column = cols > most;
    if (per_column) {
        launch_kernel(k_discounted_return, dim3(grid_exact((uint64_t)cols)), dim3(kWG), 0, s, x, done, end_value, out,
                      timesteps, batch, inner, gamma, kBack ? 1 : 0);
        LAUNCH_CHECK("k_discounted_return");
        return MRB_OK;
    }
    const hipError_t e = launch_discounted_return_tiled(kBack, x, done, end_value, out, timesteps, batch, inner, gamma, s);
    if (e != hipSuccess) return fail(MRB_EHIP, "launch k_discounted_return_tiled: %s", hipGetErrorString(e));
    return MRB_OK;
}

extern "C" {

int mrb_discounted_return(const float* reward, const uint8_t* done, const float* last_value, float* out,
                          int64_t timesteps, int64_t batch, int64_t inner, float gamma, void* stream) {
    return discounted_return<false>(reward, done, const_cast<float*>(last_value), out, timesteps, batch, inner, gamma,
                                    static_cast<hipStream_t>(stream));
}

}  // extern "C"

#include "mrb_more.inc"
