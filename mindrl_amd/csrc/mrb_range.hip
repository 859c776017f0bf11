#include "mrb_range.h"

#include "../../include/mrb.h"
#include "mrb_launch.h"
#include "mrb_meet.h"
#include "mrb_rows.h"
#include "mrb_tree.h"

namespace mrb {

namespace {

struct Trees {
    float* sum;
    float* mn;
};

// ---------------------------------------------------------------------------
// update_priorities of a few thousand entries (PriorityReplayBufferUpdate,
// mindspore_rl/core/priority_replay_buffer.py:71-73,120), divided by LEAVES: a workgroup owns a run of 2^w leaves,
// looks every entry of the call over for those aimed at its leaves, elects the last one of each leaf in an LDS table
// with a word per leaf, rebuilds the tiles that changed, a wave each, and goes on with its w levels to the run's root.
// The last workgroup to get there rebuilds the levels above the runs (mrb_meet.h; all of them meet, also those without an entry, whose
// root is as it was). No stamps in memory, no pass of its own for the election, no wave for a clean tile, one launch instead of three or
// four. What it pays is that every workgroup reads all indices (out of its L2: 16 KB for 2048 entries), which is why larger calls keep the
// stamp pass (the rule, with both sides measured, is at takes_range).
// A call is bound by its chain of trips - indices, priorities of a run's own, tiles, the roots' meeting -, not
// by bytes. 2048 entries on 2^21 leaves 14.7 -> 8.6 us, and 8.4 with the meeting in the place of a second launch, which
// a host that is behind takes 2.7 us longer to issue. (On the device: 5000 entries at random on 2^20 leaves 9.8 -> 9.3, on 2^18 8.3 -> 8.0, on 2^16
// 7.5 and 7.5, on 2^14 7.6 -> 7.8 and 12,000 10.0 -> 10.4; one after the other 6.5 -> 6.1 on 2^14, but 6.5 -> 6.8 on 2^15, 6.6 -> 7.0 on 2^16 and 6.7 -> 7.0 on 2^17, where
// the few workgroups with entries come last and count in two steps.) Up to 1024 entries, up to 4096 on at most 20 levels, k_range_one,
// whose workgroups read the priorities with the indices, is faster.
// ---------------------------------------------------------------------------
// (no argument for what the kernel can tell: see PutArgs::threads)
__host__ __device__ constexpr int range_threads(int64_t n) { return n > 4096 ? 1024 : 512; }  // (256: 0.3 to 1.5 us more)
constexpr int kRangePer = 8;  // entries of a thread and trip, all requested at once, the next trip's before these are looked at

// kLog2: the table's leaves; w <= kLog2.
template <int kLog2>
__global__ __launch_bounds__(1024) void k_tree_range(const int64_t* __restrict__ indices, const float* __restrict__ priorities,
                                                         float* sum, float* mn, float* maxp, int n, int capacity, int depth_w,
                                                         float alpha) {
    __shared__ unsigned long long s_win[1 << kLog2];         // per leaf: the latest entry's election_key (with its power)
    __shared__ uint32_t s_dirty[1 << (kLog2 - 8)];           // per tile
    __shared__ float s_rs[1 << (kLog2 - 8)], s_rm[1 << (kLog2 - 8)];  // the tiles' roots
    const int depth = depth_w & 255, w = depth_w >> 8;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t run = blockIdx.x, leaves = 1u << w, tiles = leaves / kBlockNodes;
    const Trees trees{sum, mn};
    const int threads = range_threads(n), trip = kRangePer * threads;
    uint32_t* const err = err_before(maxp);
    const int top = depth - w;  // levels above the runs, at least two
    const uint32_t runs = ((uint32_t)capacity + leaves - 1) >> w;
    auto request = [&](int base, int64_t (&to)[kRangePer]) {
#pragma unroll
        for (int q = 0; q < kRangePer; ++q) {
            const int j = base + q * threads + (int)tid;
            to[q] = j < n ? indices[j] : -1;
        }
    };
    int64_t idx[kRangePer];
    request(0, idx);
    // the launch's number and the runs' roots as they are, this one's among them
    uint32_t turn = 0;
    float4 vs = make_float4(0.f, 0.f, 0.f, 0.f), vm = vs;
    float cs = 0.0f, cm = 0.0f;
    if (wave == 0) {
        turn = meet_turn(maxp);
        cs = sum[(1u << top) + run];
        cm = mn[(1u << top) + run];
        if (4 * lane < (1u << top)) {
            vs = *reinterpret_cast<const float4*>(sum + (1u << top) + 4 * lane);
            vm = *reinterpret_cast<const float4*>(mn + (1u << top) + 4 * lane);
        }
    }
    // the roots as they are, for the tiles that stay clean; the table is cleared while the entries are on their way
    const uint32_t root0 = ((1u << depth) + run * leaves) >> kRoundLevels;
    if (tid < tiles) {
        s_rs[tid] = sum[root0 + tid];
        s_rm[tid] = mn[root0 + tid];
        s_dirty[tid] = 0;
    }
    for (uint32_t i = 2 * tid; i < leaves; i += 2 * threads) *reinterpret_cast<ulonglong2*>(&s_win[i]) = make_ulonglong2(0, 0);
    lds_barrier();
    float largest = 0.0f;
    for (int base = 0; base < n; base += trip) {  // uniform
        int64_t next[kRangePer];
        if (base + trip < n) request(base + trip, next);
        uint32_t mine = 0;
        float p[kRangePer];
#pragma unroll
        for (int q = 0; q < kRangePer; ++q) {
            const int j = base + q * threads + (int)tid;
            const bool in = idx[q] >= 0 && idx[q] < capacity;
            // (entries that name no leaf are the first workgroup's to flag)
            const bool take = j < n && (in ? (uint32_t)((uint64_t)idx[q] >> w) == run : run == 0);
            if (take) {
                mine |= 1u << q;
                p[q] = priorities[j];
            }
        }
        while (mine) {  // (a thread has one entry of its run, or none, as a rule)
            const int q = __builtin_ctz(mine);
            mine &= mine - 1;
            int64_t i = idx[0];
            float x = p[0];
#pragma unroll
            for (int k = 1; k < kRangePer; ++k) {
                i = q == k ? idx[k] : i;
                x = q == k ? p[k] : x;
            }
            const bool in = i >= 0 && i < capacity, ok = valid_priority(x);
            if (!in) atomicOr(err, MRB_DERR_INDEX);
            if (!ok) atomicOr(err, MRB_DERR_PRIORITY);
            if (!in || !ok) continue;
            const float power = powf_det(x, alpha);
            largest = fmaxf(largest, power);
            const uint32_t at = (uint32_t)i & (leaves - 1);
            atomicMax(&s_win[at], election_key(base + q * threads + (int)tid, power));
            s_dirty[at / kBlockNodes] = 1;
        }
        if (base + trip < n) {
#pragma unroll
            for (int q = 0; q < kRangePer; ++q) idx[q] = next[q];
        }
    }
    largest = wave_max(largest);
    if (lane == 0 && largest > 0.0f) raise_max(maxp, largest);
    lds_barrier();
    // the tiles that changed, dealt to the waves
    const unsigned long long dirty = __ballot(lane < tiles && s_dirty[lane < tiles ? lane : 0] != 0);
    if (dirty == 0 && wave != 0) return;
    uint32_t nth = 0;
    for (unsigned long long rest = dirty; rest; rest &= rest - 1, ++nth) {
        if (nth % ((uint32_t)threads / 64) != wave) continue;
        const uint32_t t = (uint32_t)__builtin_ctzll(rest);
        const uint32_t first = (1u << depth) + run * leaves + t * kBlockNodes;
        float4 ls = *reinterpret_cast<const float4*>(sum + first + 4 * lane);
        float4 lm = *reinterpret_cast<const float4*>(mn + first + 4 * lane);
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
    }
    if (dirty != 0) {  // (the same in every wave)
        lds_barrier();
        if (wave != 0) return;
        // from the tiles' roots to the run's (at most six levels)
        cs = lane < tiles ? s_rs[lane] : 0.0f;
        cm = lane < tiles ? s_rm[lane] : 0.0f;
        run_parents(trees, w - kRoundLevels, root0, lane, lane < tiles, cs, cm);
    }
    // and from the runs' to the tree's
    const uint32_t mine = 4 * lane < runs ? (runs - 4 * lane >= 4 ? 15u : (1u << (runs - 4 * lane)) - 1) : 0u;
    const MeetPlan plan = meet_plan(mine, run, lane);
    if (!meet(maxp, err, turn, run, cs, cm, lane, plan, vs, vm)) return;
    tile_parents(trees, top, 1u << top, lane, 4 * lane < (1u << top), vs, vm);
}

// ---------------------------------------------------------------------------
// Very large trees (21 levels and more) under a call that names few of their leaves (65,536 of 2^24): scanning every
// 256-leaf tile would cost more in wave launches than the update itself, so the ENTRIES drive the lowest levels. A group
// of 2^(g0-2) lanes (g0 = 4..6) takes one entry; if that entry owns its block of 2^g0 leaves (it holds the largest of
// the block's stamps), the group replaces the leaves the stamps name, rebuilds the g0 levels above with tile_parents'
// operations and marks the tile of the next round.
// What bounds it: trips to memory that nothing is cached for, and four lines per entry written in part (ten with the silent levels, and
// that bound it: see kSilentLevels). The block's
// stamps, its nodes and the entry's own power are therefore requested together, as soon as the index is there, whether
// or not the entry turns out to own the block (nearly every one does), and the arguments are preloaded: two trips where
// there were five (arguments, index and priority, stamps, nodes, powers). An owner stores all leaves of its block, 64
// bytes of a line instead of the pieces that changed. 65,536 entries on 2^24 leaves that no cache holds, this launch by itself: 19.2 -> 17.7 us,
// without the silent levels some 5 less.
// ---------------------------------------------------------------------------
constexpr int kSparseWG = 256;

// Level 3 + S above the block, inside an entry's group of lanes.
template <int S>
__device__ __forceinline__ void sparse_step(const Trees& a, int g0, uint32_t first, uint32_t sub, bool active, float& cs, float& cm) {
    if (S < g0 - 2) {  // uniform
        cs = cs + butterfly_peer<S>(cs);
        cm = fminf(cm, butterfly_peer<S>(cm));
        if (S >= kSilentLevels - 2 && active && (sub & ((2u << S) - 1)) == 0) {
            a.sum[(first >> (3 + S)) + (sub >> (S + 1))] = cs;
            a.mn[(first >> (3 + S)) + (sub >> (S + 1))] = cm;
        }
    }
}

// plan: depth | g0 << 8 | g_dirty << 16. kG0: g0 where the compiler is to know it (four: trees of up to 24 levels), or 0.
template <int kG0>
__global__ __launch_bounds__(kSparseWG) void k_tree_sparse(const int64_t* __restrict__ indices,
                                                           const unsigned long long* __restrict__ stamp,
                                                           const float* __restrict__ powered, float* sum, float* mn, uint32_t* dirty,
                                                           int n, uint32_t capacity, uint32_t epoch, int plan) {
    const int depth = plan & 255, g0 = kG0 ? kG0 : (plan >> 8) & 255, g_dirty = plan >> 16;
    const uint32_t group = 1u << (g0 - 2);
    const uint32_t tid = blockIdx.x * kSparseWG + threadIdx.x;
    const uint32_t j = tid >> (g0 - 2), sub = tid & (group - 1);
    const Trees trees{sum, mn};
    int64_t idx = -1;
    if (j < (uint32_t)n) idx = indices[j];
    bool active = idx >= 0 && idx < (int64_t)capacity;
    const uint32_t block = active ? (uint32_t)idx >> g0 : 0u;
    const uint32_t first = (1u << depth) + (block << g0);  // heap index of the block's first leaf
    float4 vs = make_float4(0.f, 0.f, 0.f, 0.f), vm = vs;
    ulonglong2 s01 = make_ulonglong2(0, 0), s23 = s01;
    float own = 0.0f;
    if (active) {
        const ulonglong2* st = reinterpret_cast<const ulonglong2*>(stamp + ((uint64_t)block << g0) + 4 * sub);
        s01 = st[0];
        s23 = st[1];
        vs = *reinterpret_cast<const float4*>(sum + first + 4 * sub);
        vm = *reinterpret_cast<const float4*>(mn + first + 4 * sub);
        own = powered[j];  // (of an invalid priority: whatever lies there; no stamp names it)
    }
    // The block's owner is the entry with the largest stamp of this call among its leaves (an entry that is not valid has
    // raised none).
    const unsigned long long a01 = s01.x > s01.y ? s01.x : s01.y, a23 = s23.x > s23.y ? s23.x : s23.y;
    unsigned long long top = a01 > a23 ? a01 : a23;
    for (uint32_t m = 1; m < group; m <<= 1) {
        const unsigned long long o = __shfl_xor(top, (int)m);
        top = top > o ? top : o;
    }
    const unsigned long long mine = ((unsigned long long)epoch << 32) | j;
    active = active && top == mine;
    if (active) {
        auto leaf = [&](unsigned long long st, float& ls, float& lm) {
            if ((uint32_t)(st >> 32) != epoch) return;
            ls = lm = st == mine ? own : powered[(uint32_t)st];
        };
        leaf(s01.x, vs.x, vm.x);
        leaf(s01.y, vs.y, vm.y);
        leaf(s23.x, vs.z, vm.z);
        leaf(s23.y, vs.w, vm.w);
        *reinterpret_cast<float4*>(sum + first + 4 * sub) = vs;
        *reinterpret_cast<float4*>(mn + first + 4 * sub) = vm;
        if (sub == 0) dirty[block >> g_dirty] = epoch;
    }
    const float s0 = vs.x + vs.y, s1 = vs.z + vs.w;
    const float m0 = fminf(vm.x, vm.y), m1 = fminf(vm.z, vm.w);
    float cs = s0 + s1, cm = fminf(m0, m1);  // (the levels up to kSilentLevels are silent: these trees have 21 levels and more)
    sparse_step<0>(trees, g0, first, sub, active, cs, cm);
    sparse_step<1>(trees, g0, first, sub, active, cs, cm);
    sparse_step<2>(trees, g0, first, sub, active, cs, cm);
    sparse_step<3>(trees, g0, first, sub, active, cs, cm);
}

// The levels above: a workgroup owns 2^w nodes at depth `top` (w = top - 8, 9 to 12), a wave each tile of 256, and goes on to
// the run's root; the last of the 256 workgroups to get there rebuilds the eight levels above the runs (mrb_meet.h; all of them meet: which runs
// changed, nobody knows but they). Nodes, dirty word and the root as it is are requested together. With a launch of its own
// for the eight levels 16,384 entries on 2^22 leaves took 12.6 us, now 12.0, 65,536 on 2^24 23.9, now 22.9. (A launch for eight levels and one workgroup
// for the twelve above took 3 us more.)
__global__ __launch_bounds__(1024) void k_tree_runs(float* sum, float* mn, const uint32_t* __restrict__ dirty, float* maxp, uint32_t epoch, int top) {
    __shared__ float s_rs[16], s_rm[16];
    __shared__ uint32_t s_new[16];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int up = top - 2 * kRoundLevels;  // levels from the tiles' roots to the run's: 2^up waves
    const uint32_t tile = (blockIdx.x << up) + wave, first = (1u << top) + tile * kBlockNodes;
    const Trees trees{sum, mn};
    const float4 vs = *reinterpret_cast<const float4*>(sum + first + 4 * lane);
    const float4 vm = *reinterpret_cast<const float4*>(mn + first + 4 * lane);
    float rs = sum[first >> kRoundLevels], rm = mn[first >> kRoundLevels];
    const bool changed = dirty[tile] == epoch;
    uint32_t turn = 0;
    float4 roots_s = vs, roots_m = vm;
    if (wave == 0) {
        turn = meet_turn(maxp);
        roots_s = *reinterpret_cast<const float4*>(sum + kBlockNodes + 4 * lane);
        roots_m = *reinterpret_cast<const float4*>(mn + kBlockNodes + 4 * lane);
    }
    if (changed) tile_parents(trees, kRoundLevels, first, lane, true, vs, vm, &rs, &rm);
    if (lane == 0) {
        s_rs[wave] = rs;
        s_rm[wave] = rm;
        s_new[wave] = changed;
    }
    lds_barrier();
    if (wave != 0) return;
    const MeetPlan plan = meet_plan(15u, blockIdx.x, lane);
    const uint32_t tiles = 1u << up;
    const bool any = __any(lane < tiles && s_new[lane < tiles ? lane : 0]);
    float cs = lane < tiles ? s_rs[lane] : 0.0f, cm = lane < tiles ? s_rm[lane] : 0.0f;
    run_parents(trees, up, first >> kRoundLevels, lane, any && lane < tiles, cs, cm);  // (of a clean run: its root as it is)
    if (!meet(maxp, err_before(maxp), turn, blockIdx.x, cs, cm, lane, plan, roots_s, roots_m)) return;
    tile_parents(trees, kRoundLevels, kBlockNodes, lane, true, roots_s, roots_m);
}

}  // namespace

// Runs of 256 to 16,384 leaves: 256 of them - and eight levels left above, one tile - where that is possible (16 to 22
// levels). A table of 16,384 words is 128 KB of a compute unit's LDS.
int tree_range_levels(int depth) {
    const int w = depth - kRoundLevels;
    return w < 8 ? 8 : w > 14 ? 14 : w;
}

hipError_t launch_tree_range(const int64_t* indices, const float* priorities, int64_t n, float* sum, float* mn, float* maxp,
                             int64_t capacity, int depth, float alpha, hipStream_t s) {
    const int w = tree_range_levels(depth);
    const dim3 grid((uint32_t)((capacity + ((int64_t)1 << w) - 1) >> w)), threads(range_threads(n));
    auto* const kernel = w <= 10 ? k_tree_range<10> : w <= 12 ? k_tree_range<12> : w == 13 ? k_tree_range<13> : k_tree_range<14>;
    launch_kernel(kernel, grid, threads, 0, s, indices, priorities, sum, mn, maxp, (int)n, (int)capacity, depth | w << 8, alpha);
    return hipGetLastError();
}

hipError_t launch_tree_sparse(const int64_t* indices, const unsigned long long* stamp, const float* powered, float* sum, float* mn,
                              uint32_t* dirty, int64_t n, int64_t capacity, int depth, int g0, int g_dirty, uint32_t epoch,
                              hipStream_t s) {
    const dim3 grid((uint32_t)(((n << (g0 - 2)) + kSparseWG - 1) / kSparseWG));
    launch_kernel(g0 == 4 ? k_tree_sparse<4> : k_tree_sparse<0>, grid, dim3(kSparseWG), 0, s, indices, stamp, powered, sum, mn, dirty, (int)n, (uint32_t)capacity,
                  epoch, depth | g0 << 8 | g_dirty << 16);
    return hipGetLastError();
}

hipError_t launch_tree_runs(float* sum, float* mn, const uint32_t* dirty, float* maxp, int top, uint32_t epoch, hipStream_t s) {
    launch_kernel(k_tree_runs, dim3(1u << kRoundLevels), dim3(64u << (top - 2 * kRoundLevels)), 0, s, sum, mn, dirty, maxp, epoch, top);
    return hipGetLastError();
}

}  // namespace mrb
