// What the kernels of several source files share of a push's tree work, and the arguments of the tree kernels (no kernels here).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mrb_rows.h"
#include "mrb_tree.h"

namespace mrb {

constexpr int kMaxRounds = 3;

struct UpdateArgs {
    // entries
    const int64_t* indices;   // NULL: entry j targets slot (first_slot + j) mod capacity
    const float* priorities;  // NULL: the targeted leaves take the running max priority as it is
    int64_t n;
    int64_t first_slot;       // negative: (pushes mod capacity), read from the device (see Counters)
    // buffer
    int64_t capacity;
    int64_t leaves;
    int depth;
    float alpha;
    uint32_t epoch;
    unsigned long long* stamp;  // [leaves]
    float* sum;
    float* mn;
    float* powered;  // [n] priorities^alpha of this call's entries (update_priorities only)
    float* maxp;  // running max priority (device scalar)
    float* maxp_next;  // a push with priorities in progress: the largest p^alpha its leaf-level waves have seen
    uint32_t* err;
    // rebuild plan: round r starts at depth lo[r] and rebuilds g[r] levels; the top starts at top_depth
    int nrounds;
    int lo[kMaxRounds];
    int g[kMaxRounds];
    int top_depth;
    uint32_t* dirty[kMaxRounds];  // per round: one epoch word per block of 1 << g[r] nodes at depth lo[r]
    int fold_max;                // push with priorities: the top workgroup also raises the running max, 1 = from a
                                 // scan of the priorities, 2 = from maxp_next, where the leaf-level waves left it
    int inline_election;         // small update_priorities: no stamp pass, the leaf-level waves scan the entries
    // sparse updates of very large trees: the lowest sparse_g0 levels are rebuilt per entry
    // (k_tree_sparse) instead of per tile
    int sparse_g0;               // 0 = not used
    int full_top;                // a push that follows an update in the same call: the top is rebuilt over all its
                                 // tiles, not only those above the pushed slots (the update changed others)
    // device-resident counters: rows this launch - the push's last - adds to them when it is done (0: none), and
    // the workgroups of this launch that read the ring position (see counters_push_done)
    int64_t advance;
    uint32_t readers;
    uint32_t tile_blocks;  // workgroups of k_tree_update that work on tiles (those behind them carry a push's row copy)
};

// ---------------------------------------------------------------------------
// A push under at most 16 leaf tiles on a tree of more than 8 levels, in ONE launch: a run of slots changes one path
// of tiles - a wave rebuilds each leaf tile, then the tile eight levels up that holds their roots (two where the run
// crosses its end, one more where it wraps around the ring), then the tile above that, up to the root. Which tiles
// these are follows from the slots, so all of them are requested when the kernel starts: of their nodes only the
// lower tiles' roots change, and those reach the wave that holds the tile through LDS. The call is then one trip to
// memory and two to four rebuilds in a row (within one workgroup, whose waves share a compute unit: no fence), where
// a launch per eight levels pays a launch, a trip and a rebuild for each. Measured, us per call before and now, plain /
// with priorities: 64 rows into 2^24 leaves (three launches before) 12.0 / 10.6 and 3.8 / 5.6; 16 rows into 2^20 (one
// launch that rebuilt the whole top) 4.2 / 6.5 and 3.8 / 5.3; 1024 rows into 2^21 4.8 / 7.4 and 4.3 / 5.6; 64 rows into 2^12 (one workgroup that
// rebuilt the whole tree) 4.3 / 6.2 and 2.6 / 3.4, into 2^9 3.6 / 5.6 and 2.4 / 3.2. With 4096
// priorities the powers of one compute unit are the bound (5.6 / 8.7): k_push_many, which shares them out, takes pushes with
// priorities where it can (takes_push_many). The row copy rides along as further workgroups of the
// kernels that call this (k_push_run, k_short_push_run).
//   threads    of the workgroup
//   units      leaf tiles from the first slot's on, around the ring's end: waves with work
// ---------------------------------------------------------------------------
constexpr int kFusedWG = 1024;
constexpr int kRunWaves = kFusedWG / 64;
constexpr int kRunLevels = 3;  // tiles above the leaf tiles on a path: trees of at most 8 + 3 * 8 levels

__device__ __forceinline__ void push_run_body(const UpdateArgs& a, uint32_t units, uint32_t threads) {
    __shared__ float s_s[kRunLevels][kRunWaves], s_m[kRunLevels][kRunWaves];
    __shared__ uint32_t s_new[kRunLevels][kRunWaves];  // whether the wave has a new root for the level above
    __shared__ float s_largest[kRunWaves];             // the largest p^alpha the wave has written (a push with priorities)
    const uint32_t lane = threadIdx.x & 63;
    // (read as a scalar: sixteen waves share the compute unit's issue slots, and what follows from the wave's number
    // alone - its tiles - then costs them nothing)
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // (a launch that moves the device's counters on: thread 0 takes them now, for the advance at the end)
    CounterTicket ticket{};
    if (a.advance > 0 && threadIdx.x == 0) ticket = counters_take(a.err);
    // (slots and row counts fit 32 bits: the capacity is at most 2^30, the run at most 16 tiles)
    const uint32_t capacity = (uint32_t)a.capacity, n = (uint32_t)a.n;
    uint32_t first_slot = (uint32_t)a.first_slot;
    if (a.first_slot < 0) first_slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)ring_position(counters_behind(a.err), a.capacity));
    const uint32_t ring_tiles = (capacity + kBlockNodes - 1) / kBlockNodes;  // the ring ends at `capacity`
    const uint32_t t0 = first_slot / kBlockNodes;
    auto tile_of = [&](uint32_t unit) -> uint32_t {
        const uint32_t t = t0 + unit;
        return t >= ring_tiles ? t - ring_tiles : t;
    };
    // of the waves whose leaf tiles lie under one tile l + 1 rounds up the first holds it (the tiles' numbers rise from
    // wave to wave, and start again from zero where the run wraps)
    auto holds = [&](uint32_t w, int l) -> bool {
        const uint32_t up = tile_of(w) >> (8 * (l + 1));
        return w < units && (w == 0 || (up != tile_of(w - 1) >> (8 * (l + 1)) && up != t0 >> (8 * (l + 1))));
    };
    const uint32_t my_tile = tile_of(wave);
    // The wave's leaf tile, the priorities of its leaves and the running max, all requested before anything is used.
    const uint32_t leaf = my_tile * kBlockNodes + 4 * lane, leaf_first = (1u << a.depth) + my_tile * kBlockNodes;
    const bool work = wave < units;  // wave-uniform
    float4 ls = make_float4(0.f, 0.f, 0.f, 0.f), lm = ls;
    float old_max = 0.0f, pv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t in = 0;  // bit c: the push writes leaf + c
    if (work) {
        ls = *reinterpret_cast<const float4*>(a.sum + leaf_first + 4 * lane);
        lm = *reinterpret_cast<const float4*>(a.mn + leaf_first + 4 * lane);
        old_max = *a.maxp;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t slot = leaf + c, e = slot >= first_slot ? slot - first_slot : slot + capacity - first_slot;
            if (slot < capacity && e < n) {
                in |= 1u << c;
                if (a.priorities) pv[c] = a.priorities[e];
            }
        }
    }
    // the tiles above
    float4 vs[kRunLevels], vm[kRunLevels];
#pragma unroll
    for (int l = 0; l < kRunLevels; ++l) {
        const int d = a.depth - kRoundLevels * (l + 1);  // the tile's depth
        vs[l] = make_float4(0.f, 0.f, 0.f, 0.f);
        vm[l] = vs[l];
        if (d <= 0 || !holds(wave, l)) continue;  // wave-uniform
        if (d == 1) {  // a level of two nodes
            vs[l].x = a.sum[2], vs[l].y = a.sum[3];
            vm[l].x = a.mn[2], vm[l].y = a.mn[3];
        } else if (4 * lane < (1u << d)) {
            const uint32_t first = (1u << d) + (my_tile >> (8 * (l + 1))) * kBlockNodes + 4 * lane;
            vs[l] = *reinterpret_cast<const float4*>(a.sum + first);
            vm[l] = *reinterpret_cast<const float4*>(a.mn + first);
        }
    }
    float rs = 0.0f, rm = 0.0f, largest = 0.0f;
    const bool changed = work && __any(in != 0);  // (the ring position may be the device's: the last tile may not be met)
    bool rebuilt = changed;
    if (changed) {
        float q[4] = {old_max, old_max, old_max, old_max};
        if (a.priorities) {
            const float4 pw = powf_det_x4(make_float4(pv[0], pv[1], pv[2], pv[3]), a.alpha);  // the four together
            const float p4[4] = {pw.x, pw.y, pw.z, pw.w};
            bool bad = false;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bool ok = valid_priority(pv[c]);  // invalid: the fresh slot stays at the running max
                if (ok) q[c] = p4[c];
                if (in >> c & 1u) {
                    if (ok) largest = fmaxf(largest, p4[c]);
                    bad = bad || !ok;
                }
            }
            if (bad && a.fold_max) atomicOr(a.err, MRB_DERR_PRIORITY);
        }
        if (in & 1u) ls.x = lm.x = q[0];
        if (in & 2u) ls.y = lm.y = q[1];
        if (in & 4u) ls.z = lm.z = q[2];
        if (in & 8u) ls.w = lm.w = q[3];
        if (in) {
            *reinterpret_cast<float4*>(a.sum + leaf_first + 4 * lane) = ls;
            *reinterpret_cast<float4*>(a.mn + leaf_first + 4 * lane) = lm;
        }
        if (a.fold_max) largest = wave_max(largest);
        tile_parents(a, kRoundLevels, leaf_first, lane, true, ls, lm, &rs, &rm, has_silent(a.depth));
    }
    if (lane == 0) s_largest[wave] = largest;
#pragma unroll
    for (int l = 0; l < kRunLevels; ++l) {
        const int d = a.depth - kRoundLevels * (l + 1);
        if (d <= 0) break;  // uniform
        if (lane == 0) {
            s_s[l][wave] = rs;
            s_m[l][wave] = rm;
            s_new[l][wave] = rebuilt;
        }
        lds_barrier();
        if (l == 0 && a.fold_max && wave == threads / 64 - 1) {
            // the running max, by the last wave: every leaf that takes it as it was has been written
            const float q = wave_max(lane < units ? s_largest[lane] : 0.0f);
            if (lane == 0 && q > 0.0f) raise_max(a.maxp, q);
        }
        rebuilt = false;
        if (!holds(wave, l)) continue;  // wave-uniform
        const uint32_t tile0 = (my_tile >> (8 * (l + 1))) * kBlockNodes;  // this tile's first node within its level
        auto take = [&](uint32_t u, int c) {
            if (!s_new[l][u]) return;
            const float ps = s_s[l][u], pm = s_m[l][u];
            switch (c) {
                case 0: vs[l].x = ps, vm[l].x = pm; break;
                case 1: vs[l].y = ps, vm[l].y = pm; break;
                case 2: vs[l].z = ps, vm[l].z = pm; break;
                default: vs[l].w = ps, vm[l].w = pm; break;
            }
        };
        if (l == 0) {
            // the leaf tiles are consecutive: which wave holds a node's follows from the node (all lookups at once)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t tile = tile0 + 4 * lane + c;  // the leaf tile under the node
                const uint32_t u = tile >= t0 ? tile - t0 : tile + ring_tiles - t0;  // (around the ring's end)
                if (tile < ring_tiles && u < units) take(u, c);
            }
        } else {
            for (uint32_t u = wave; u < units; ++u) {  // scalar: the waves that hold the tiles below (at most three)
                if (!holds(u, l - 1)) continue;
                const uint32_t at = (tile_of(u) >> (8 * l)) - tile0;
                if (at / 4 == lane) take(u, at & 3);
            }
        }
        if (d == 1) {
            if (lane == 0) {
                a.sum[1] = vs[l].x + vs[l].y;
                a.mn[1] = fminf(vm[l].x, vm[l].y);
            }
        } else {
            tile_parents(a, d < kRoundLevels ? d : kRoundLevels, (1u << d) + tile0, lane, 4 * lane < (1u << d), vs[l], vm[l], &rs, &rm);
            rebuilt = true;
        }
    }
    counters_push_done(a.err, a.advance, a.capacity, a.readers, &ticket);
}

// The walk of a push of one row (see k_push_one).
constexpr int kPushOneMaxDepth = 30;
// The walk of one wave. kAfterUpdate: the walk follows an update_priorities in the same launch (same workgroup),
// so the running max is read where the update's atomic maxima were performed (past this compute unit's cache),
// and the siblings are requested only now, after the update's stores.
// `taken`: this launch moves the device's counters on, `ticket` holds them as the caller took them - the position is theirs,
// and, unless the caller has reported already (`report`), the wave's report (see counters_report) goes out behind the
// walk's own requests, so that nothing the walk waits for queues up behind the atomic.
// kSilent (has_silent(depth)): lanes 32 to 47 bring the sixteen leaves around the row's instead of the siblings on the levels above the
// leaves, and four butterflies go from the leaf to the node four levels up, which need not write what lies between.
template <bool kAfterUpdate, bool kSilent>
__device__ __forceinline__ void push_one_levels(float* sum, float* mn, float* maxp, int64_t first_slot, int64_t capacity, int64_t leaves,
                                                int depth, float alpha, const float* priority, uint32_t* err, uint32_t lane,
                                                CounterTicket& ticket, bool taken, bool report, uint32_t readers) {
    // negative: the ring position is on the device (see Counters)
    const int64_t slot = taken             ? ticket_position(ticket, capacity)
                         : first_slot >= 0 ? first_slot
                                           : ring_position(counters_behind(err), capacity);
    const uint32_t v = (uint32_t)leaves + (uint32_t)slot;
    constexpr int kStart = kSilent ? kSilentLevels + 1 : 0;  // levels above the leaves that the walk starts from
    const int top = depth - kStart;
    float sib_s = 0.0f, sib_m = 0.0f;
    const bool leaf_lane = kSilent && lane >> 4 == 2u;
    if ((lane >= 1 && lane <= (uint32_t)top) || leaf_lane) {
        const uint32_t node = leaf_lane ? (v & ~15u) + (lane & 15u) : (v >> (((uint32_t)depth - lane) & 31u)) ^ 1u;
        sib_s = sum[node];
        sib_m = mn[node];
    }
    // the leaf: the running max as the call finds it, or the given priority's power (an invalid one is flagged
    // and the row takes the running max, as a plain push would give it)
    const float running = kAfterUpdate ? __uint_as_float(__hip_atomic_load(reinterpret_cast<unsigned int*>(maxp), __ATOMIC_RELAXED,
                                                                           __HIP_MEMORY_SCOPE_AGENT))
                                       : *maxp;
    const float p = priority ? *priority : 0.0f;
    if (report) counters_report(ticket, err, readers, lane);
    const bool given = priority != nullptr && valid_priority(p);
    if (priority != nullptr && !given && lane == 0) atomicOr(err, MRB_DERR_PRIORITY);
    const float q = given ? powf_det_call(p, alpha) : running;
    float cs = q, cm = q;
    uint32_t node = v;
    if (lane == 0) {
        sum[node] = cs;
        mn[node] = cm;
    }
    if (kSilent) {
        static_assert(!kSilent || kStart == 4, "sixteen leaves");
        const bool own = lane == 32u + (v & 15u);
        float s = own ? q : sib_s, m = own ? q : sib_m;
        s = s + butterfly_peer<0>(s);
        m = fminf(m, butterfly_peer<0>(m));
        s = s + butterfly_peer<1>(s);
        m = fminf(m, butterfly_peer<1>(m));
        s = s + butterfly_peer<2>(s);
        m = fminf(m, butterfly_peer<2>(m));
        s = s + butterfly_peer<3>(s);
        m = fminf(m, butterfly_peer<3>(m));
        cs = lane_value(s, 32);
        cm = lane_value(m, 32);
        node = v >> kStart;
        if (lane == 0) {
            sum[node] = cs;
            mn[node] = cm;
        }
    }
#pragma unroll
    for (int L = kPushOneMaxDepth - kStart; L >= 1; --L) {
        if (L <= top) {  // wave-uniform
            const float os = lane_value(sib_s, L), om = lane_value(sib_m, L);
            const bool right = (node & 1u) != 0;
            cs = right ? os + cs : cs + os;
            cm = right ? fminf(om, cm) : fminf(cm, om);
            node >>= 1;
            if (lane == 0) {
                sum[node] = cs;
                mn[node] = cm;
            }
        }
    }
    // last: the leaf has read the running max as the call found it
    if (given && lane == 0 && q > 0.0f) raise_max(maxp, q);
}
template <bool kAfterUpdate>
__device__ __forceinline__ void push_one_walk(float* sum, float* mn, float* maxp, int64_t first_slot, int64_t capacity, int64_t leaves,
                                              int depth, float alpha, const float* priority, uint32_t* err, uint32_t lane,
                                              CounterTicket& ticket, bool taken, bool report, uint32_t readers) {
    if (has_silent(depth))  // uniform
        push_one_levels<kAfterUpdate, true>(sum, mn, maxp, first_slot, capacity, leaves, depth, alpha, priority, err, lane, ticket, taken, report, readers);
    else
        push_one_levels<kAfterUpdate, false>(sum, mn, maxp, first_slot, capacity, leaves, depth, alpha, priority, err, lane, ticket, taken, report, readers);
}

}  // namespace mrb
