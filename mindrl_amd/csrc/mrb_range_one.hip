#include "mrb_range_one.h"

#include "../../include/mrb.h"
#include "mrb_launch.h"
#include "mrb_meet.h"
#include "mrb_tree.h"

namespace mrb {

namespace {

struct Trees {
    float* sum;
    float* mn;
};

constexpr int kOneWG = 512;                        // (1024: the same to 0.3 us more)
constexpr int kOneFew = 1024 / kOneWG, kOneMany = kOneMostEntries / kOneWG;  // entries of a thread, at most
constexpr int kOneHeld = 2;                        // changed tiles of a wave that are requested ahead

// ---------------------------------------------------------------------------
// update_priorities of up to 4096 entries (PriorityReplayBufferUpdate,
// mindspore_rl/core/priority_replay_buffer.py:71-73,120) in ONE launch, divided by LEAVES as in k_tree_range: a workgroup owns
// a run of 2^w leaves, finds the entries aimed at them, elects the last one of each leaf in an LDS table, rebuilds the tiles
// that changed and goes on to the run's root; the last workgroup to get there rebuilds the levels above the runs
// (mrb_meet.h). Every workgroup reads all entries, so each knows which runs have one: those without leave at once.
// What bounds it is its chain: the launch, the entries' trip, the tiles' (requested as soon as the indices say which change,
// on their way while the powers are taken and the leaves elected), the roots' meeting (0.9 us; with one run there is none), and
// with more than a thousand entries the looking them over. us per call queued behind a busy device, the kernels before (two
// launches; one wave along the paths; one workgroup) / this:
//   64 entries   2^10 leaves 3.7 / 3.4, 2^16 7.7 / 5.0, 2^20 9.0 / 5.4, 2^22 9.7 / 6.0
//   256 entries  2^10 3.9 / 3.4, 2^14 6.5 / 4.9, 2^16 6.2 / 5.3, 2^19 6.8 / 5.6, 2^21 7.0 / 5.8
//   512 entries  2^14 6.0 / 5.1, 2^17 6.7 / 5.6, 2^20 7.4 / 6.1; 1024  2^14 6.3 / 5.3, 2^17 6.8 / 5.9, 2^20 7.8 / 7.0
//   2048 entries 2^10 7.7 / 6.6, 2^12 6.9 / 6.4, 2^14 6.6 / 6.3, 2^18 7.5 / 7.2, 2^20 8.6 / 8.5; 4096  2^14 7.0 / 6.8, 2^18 8.0 / 7.5
// and the host issues one launch instead of two (6.8 -> 4.1 us), which is what bounds a training program's step.
// kPush: the rows a push of the same call writes come after the entries - slots first_slot .. + nrows - 1 take the running
// max as the update leaves it, or their own priorities -, in the runs that hold those slots; further workgroups carry the
// row copy. (Only one workgroup may raise the running max for pushed rows, while others read it: one run with priorities.)
// 512 entries and 4 rows: 2^14 leaves 9.5 / 5.4, 2^17 8.7 / 5.9, 2^20 9.2 / 6.5; 64 and 1: 2^14 5.8 / 5.3, 2^20 10.4 / 5.6.
// ---------------------------------------------------------------------------
template <int kLog2, bool kPush, int kPer>  // (kPush: kPer == kOneFew)
__device__ __forceinline__ void range_one(const int64_t* __restrict__ indices, const float* __restrict__ priorities, float* sum,
                                          float* mn, float* maxp, int n, int capacity, int depth_w, float alpha, const RangePush& push) {
    __shared__ unsigned long long s_win[1 << kLog2];                  // per leaf: the latest entry's election_key (with its power)
    __shared__ uint32_t s_dirty[1 << (kLog2 - 8)];                    // per tile
    __shared__ float s_rs[1 << (kLog2 - 8)], s_rm[1 << (kLog2 - 8)];  // the tiles' roots
    __shared__ uint4 s_runs[kMeetMost / 4];                           // a word per run: whether it has an entry
    __shared__ float s_largest[kOneWG / 64];
    const int depth = depth_w & 255, w = depth_w >> 8, top = depth - w;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t run = blockIdx.x, leaves = 1u << w, tiles = leaves / kBlockNodes;
    uint32_t* const err = err_before(maxp);
    const Trees trees{sum, mn};
    // the entries, all at once
    int64_t idx[kPer];
    float p[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int j = q * kOneWG + (int)tid;
        idx[q] = j < n ? indices[j] : -1;
        p[q] = j < n ? priorities[j] : -1.0f;
    }
    // the runs' roots as they are, the launch's number (the last wave: of few entries it has none); the running max
    const bool finishes = wave == kOneWG / 64 - 1;
    float4 vs = make_float4(0.f, 0.f, 0.f, 0.f), vm = vs;
    uint32_t turn = 0;
    if (finishes) {
        turn = meet_turn(maxp);
        if (top && 4 * lane < (1u << top)) {  // (top is 0 or at least 2)
            vs = *reinterpret_cast<const float4*>(sum + (1u << top) + 4 * lane);
            vm = *reinterpret_cast<const float4*>(mn + (1u << top) + 4 * lane);
        }
    }
    float running = 0.0f;
    if (kPush) running = __uint_as_float(__hip_atomic_load(reinterpret_cast<unsigned int*>(maxp), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    // the tiles' roots as they are; the table is cleared while the entries are on their way
    const uint32_t root0 = ((1u << depth) + run * leaves) >> kRoundLevels;
    float was_s = 0.0f, was_m = 0.0f;
    if (tid < tiles) {
        was_s = sum[root0 + tid];
        was_m = mn[root0 + tid];
        s_dirty[tid] = 0;
    }
    uint32_t* const marks = reinterpret_cast<uint32_t*>(s_runs);
    if (tid < kMeetMost) marks[tid] = 0;
    for (uint32_t i = 2 * tid; i < leaves; i += 2 * kOneWG) *reinterpret_cast<ulonglong2*>(&s_win[i]) = make_ulonglong2(0, 0);
    lds_barrier();
    // which runs, and of this one which tiles, change
    bool in[kPer], mine[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int j = q * kOneWG + (int)tid;
        in[q] = idx[q] >= 0 && idx[q] < capacity;
        const uint32_t r = (uint32_t)((uint64_t)idx[q] >> w);
        if (in[q]) {
            marks[r] = 1;
            if (r == run) s_dirty[((uint32_t)idx[q] & (leaves - 1)) / kBlockNodes] = 1;
        }
        mine[q] = j < n && (in[q] ? r == run : run == 0);  // (entries that name no leaf are the first workgroup's to flag)
    }
    bool pushed = false;  // rows of the push lie in this run
    if (kPush) {
        for (uint32_t r = tid; r < push.nrows; r += kOneWG) {
            uint32_t slot = push.first_slot + r;
            if (slot >= (uint32_t)capacity) slot -= (uint32_t)capacity;
            const uint32_t of = slot >> w;
            marks[of] = 1;
            if (of == run) s_dirty[(slot & (leaves - 1)) / kBlockNodes] = 1;
        }
        const uint32_t end = push.first_slot + push.nrows, lo = run * leaves, hi = lo + leaves;
        pushed = (lo < end && hi > push.first_slot) || (end > (uint32_t)capacity && lo < end - (uint32_t)capacity);
    }
    if (tid < tiles) {
        s_rs[tid] = was_s;
        s_rm[tid] = was_m;
    }
    lds_barrier();
    unsigned long long rest = __ballot(lane < tiles && s_dirty[lane < tiles ? lane : 0] != 0);
    if (rest == 0 && run != 0) return;  // (the same in every wave)
    // the changed tiles are dealt to the waves in turn, the first ones requested now, before the powers are taken
    uint32_t nth = 0;
    const bool dirty = rest != 0;
    auto next_tile = [&]() -> uint32_t {
        for (; rest; rest &= rest - 1, ++nth)
            if (nth % (kOneWG / 64) == wave) {
                const uint32_t t = (uint32_t)__builtin_ctzll(rest);
                rest &= rest - 1;
                ++nth;
                return t;
            }
        return tiles;
    };
    uint32_t held[kOneHeld];
    float4 hs[kOneHeld], hm[kOneHeld];
#pragma unroll
    for (int h = 0; h < kOneHeld; ++h) {
        held[h] = next_tile();
        hs[h] = hm[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (held[h] < tiles) {
            const uint32_t first = (1u << depth) + run * leaves + held[h] * kBlockNodes;
            hs[h] = *reinterpret_cast<const float4*>(sum + first + 4 * lane);
            hm[h] = *reinterpret_cast<const float4*>(mn + first + 4 * lane);
        }
    }
    MeetPlan plan{};
    if (finishes && top) {
        const uint4 has = s_runs[lane];
        plan = meet_plan(has.x | has.y << 1 | has.z << 2 | has.w << 3, run, lane);
    }
    float largest = 0.0f, all = 0.0f;
    uint32_t todo = 0;  // bit q: an entry whose power is still to be taken
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const bool ok = valid_priority(p[q]);
        if (mine[q]) {
            if (!in[q]) atomicOr(err, MRB_DERR_INDEX);
            if (!ok) atomicOr(err, MRB_DERR_PRIORITY);
        }
        if (!in[q] || !ok || !(mine[q] || pushed)) continue;
        if (kPer > kOneFew) {
            todo |= 1u << q;
            continue;
        }
        const float power = powf_det(p[q], alpha);
        all = fmaxf(all, power);
        if (mine[q]) {
            largest = fmaxf(largest, power);
            atomicMax(&s_win[(uint32_t)idx[q] & (leaves - 1)], election_key(q * kOneWG + (int)tid, power));
        }
    }
    while (todo) {  // (a thread has one entry of its run, or none, as a rule: the lanes take theirs together)
        const int q = __builtin_ctz(todo);
        todo &= todo - 1;
        int64_t i = idx[0];
        float x = p[0];
#pragma unroll
        for (int k = 1; k < kPer; ++k) {
            i = q == k ? idx[k] : i;
            x = q == k ? p[k] : x;
        }
        const float power = powf_det(x, alpha);
        largest = fmaxf(largest, power);
        atomicMax(&s_win[(uint32_t)i & (leaves - 1)], election_key(q * kOneWG + (int)tid, power));
    }
    largest = wave_max(largest);
    if (lane == 0 && largest > 0.0f) raise_max(maxp, largest);
    if (kPush && pushed) {
        // the running max as the update leaves it: what it was when the kernel started or later, or an entry's power
        all = wave_max(fmaxf(all, running));
        if (lane == 0) s_largest[wave] = all;
        lds_barrier();
        running = wave_max(s_largest[lane & (kOneWG / 64 - 1)]);
        float raise = 0.0f;
        for (uint32_t r = tid; r < push.nrows; r += kOneWG) {
            uint32_t slot = push.first_slot + r;
            if (slot >= (uint32_t)capacity) slot -= (uint32_t)capacity;
            if (slot >> w != run) continue;
            float value = running;
            if (push.priorities) {
                const float x = push.priorities[r];
                if (valid_priority(x)) {
                    value = powf_det(x, alpha);
                    raise = fmaxf(raise, value);
                } else {
                    atomicOr(err, MRB_DERR_PRIORITY);  // (the fresh slot takes the running max)
                }
            }
            atomicMax(&s_win[slot & (leaves - 1)], election_key(n + (int)r, value));  // after all entries
        }
        raise = wave_max(raise);
        if (lane == 0 && raise > 0.0f) raise_max(maxp, raise);
    }
    if (!dirty) return;  // (the first run, for entries that name no leaf)
    lds_barrier();
    auto rebuild = [&](uint32_t t, float4 ls, float4 lm) {
        const uint32_t first = (1u << depth) + run * leaves + t * kBlockNodes;
        const ulonglong2 k01 = *reinterpret_cast<const ulonglong2*>(&s_win[t * kBlockNodes + 4 * lane]);
        const ulonglong2 k23 = *reinterpret_cast<const ulonglong2*>(&s_win[t * kBlockNodes + 4 * lane + 2]);
        if (k01.x) ls.x = lm.x = elected_priority(k01.x);
        if (k01.y) ls.y = lm.y = elected_priority(k01.y);
        if (k23.x) ls.z = lm.z = elected_priority(k23.x);
        if (k23.y) ls.w = lm.w = elected_priority(k23.y);
        if (k01.x | k01.y | k23.x | k23.y) {
            *reinterpret_cast<float4*>(sum + first + 4 * lane) = ls;
            *reinterpret_cast<float4*>(mn + first + 4 * lane) = lm;
        }
        float rs, rm;
        tile_parents(trees, kRoundLevels, first, lane, true, ls, lm, &rs, &rm, has_silent(depth));
        if (lane == 0) {
            s_rs[t] = rs;
            s_rm[t] = rm;
        }
    };
#pragma unroll
    for (int h = 0; h < kOneHeld; ++h)
        if (held[h] < tiles) rebuild(held[h], hs[h], hm[h]);
    for (uint32_t t = next_tile(); t < tiles; t = next_tile()) {
        const uint32_t first = (1u << depth) + run * leaves + t * kBlockNodes;
        rebuild(t, *reinterpret_cast<const float4*>(sum + first + 4 * lane), *reinterpret_cast<const float4*>(mn + first + 4 * lane));
    }
    lds_barrier();
    if (!finishes) return;
    // from the tiles' roots to the run's
    float cs = lane < tiles ? s_rs[lane] : 0.0f, cm = lane < tiles ? s_rm[lane] : 0.0f;
    run_parents(trees, w - kRoundLevels, root0, lane, lane < tiles, cs, cm);
    if (top == 0) return;
    // and from the runs' to the tree's
    if (!meet(maxp, err, turn, run, cs, cm, lane, plan, vs, vm)) return;
    tile_parents(trees, top, 1u << top, lane, 4 * lane < (1u << top), vs, vm);
}

template <int kLog2, int kPer>
__global__ __launch_bounds__(kOneWG) void k_range_one(const int64_t* __restrict__ indices, const float* __restrict__ priorities,
                                                      float* sum, float* mn, float* maxp, int n, int capacity, int depth_w, float alpha) {
    range_one<kLog2, false, kPer>(indices, priorities, sum, mn, maxp, n, capacity, depth_w, alpha, RangePush{});
}

template <int kLog2>
__global__ __launch_bounds__(kOneWG) void k_range_one_push(const int64_t* __restrict__ indices, const float* __restrict__ priorities,
                                                           float* sum, float* mn, float* maxp, int n, int capacity, int depth_w,
                                                           float alpha, uint32_t runs, RangePush push, PutArgs put) {
    if (__builtin_expect(blockIdx.x >= runs, 0)) {
        rows_put_part(put, blockIdx.x - runs, put.blocks);
        rider_ends();
    }
    range_one<kLog2, true, kOneFew>(indices, priorities, sum, mn, maxp, n, capacity, depth_w, alpha, push);
}

uint32_t runs_of(int64_t capacity, int w) { return (uint32_t)((capacity + ((int64_t)1 << w) - 1) >> w); }

}  // namespace

// One run where few entries meet a table of 16 KB: nobody to meet. Otherwise runs as small as there may be (256 runs, 256 leaves),
// which leaves each the least to do; few entries meet sooner over fewer runs, as long as these are not larger than 4096 leaves.
// Measured, us, 16 / 64 / 128 / 256 runs: 2^14 leaves (32 for the first), 128 entries 4.8 / 4.9, 512 5.0 / 5.1, 2048 6.5 / 6.3;
// 2^16, 128 5.7 / 5.0 / 5.3 / 5.2, 512 6.9 / 5.4 / 5.5 / 5.4, 2048 8.7 / 6.7 / 6.8 / 6.6; 2^18, 128 - / 5.2 / 5.5 / 5.5, 512 - / 6.9 / 6.0 / 5.8,
// 2048 - / 9.2 / 7.8 / 7.2; 2^20, 128 - / 5.8 / 5.8 / 5.6, 1024 - / 9.2 / 7.9 / 7.0. A table of 16,384 words is 128 KB of a compute
// unit's LDS.
int range_one_levels(int depth, int64_t n) {
    if (depth <= 9 || (depth <= 11 && n <= kOneFew * kOneWG)) return depth;
    const int w = depth - (n > 192 || depth >= 19 ? 8 : depth >= 15 ? 6 : 5);
    return w < 8 ? 8 : w > 14 ? 14 : w;
}

hipError_t launch_range_one(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                            int64_t capacity, int depth, float alpha, hipStream_t s) {
    const int w = range_one_levels(depth, n);
    auto* kernel = w <= 10 ? k_range_one<10, kOneFew> : w <= 12 ? k_range_one<12, kOneFew> : w == 13 ? k_range_one<13, kOneFew> : k_range_one<14, kOneFew>;
    if (n > kOneFew * kOneWG) {
        if (w > 12) return hipErrorInvalidValue;  // (more than 20 levels: not taken, see takes_range_one)
        kernel = w <= 10 ? k_range_one<10, kOneMany> : k_range_one<12, kOneMany>;
    }
    launch_kernel(kernel, dim3(runs_of(capacity, w)), dim3(kOneWG), 0, s, indices, priorities, sum, mn, maxp, (int)n, (int)capacity,
                  depth | w << 8, alpha);
    return hipGetLastError();
}

hipError_t launch_range_one_push(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                                 int64_t capacity, int depth, float alpha, const RangePush& push, const PutArgs& put, hipStream_t s) {
    const int w = range_one_levels(depth, n);
    const uint32_t runs = runs_of(capacity, w);
    PutArgs ride = put;  // (its workgroups were counted for kWG threads)
    ride.blocks = (put.blocks * kWG + kOneWG - 1) / kOneWG;
    ride.threads = kOneWG;
    auto* const kernel = w <= 10 ? k_range_one_push<10> : w <= 12 ? k_range_one_push<12> : w == 13 ? k_range_one_push<13> : k_range_one_push<14>;
    launch_kernel(kernel, dim3(runs + ride.blocks), dim3(kOneWG), 0, s, indices, priorities, sum, mn, maxp, (int)n, (int)capacity,
                  depth | w << 8, alpha, runs, push, ride);
    return hipGetLastError();
}

}  // namespace mrb
