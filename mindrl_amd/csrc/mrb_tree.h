// What the kernels that rebuild the trees share: the values an update writes, its election among entries aimed at one leaf,
// and the parents of a tile.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mrb_device.h"

namespace mrb {

constexpr int kRoundLevels = 8;   // levels rebuilt above a tile
constexpr int kBlockNodes = 256;  // nodes of a tile (a float4 per lane of a wave)

// On trees of kSilentDepth levels and more the kSilentLevels levels above the leaves are silent: nobody reads them, so an update need not
// write them. A walk down meets the leaves from a node at least four levels up (the samples' node groups are cut so), a rebuild
// takes a tile's leaves and goes on from its root, and who walks up from a leaf takes the leaves around it in the trip that brings the siblings
// (push_one_levels, tree_paths_body: a push of one row with its priority on 2^20 leaves 2.6 -> 2.35 us, 64 entries on 2^23 10.2 -> 8.0). An export
// writes them first (k_tree_silent). They are
// 224 of the 255 nodes above a tile of 256 leaves, and 14 of the 15 above a block of 16 - six of the ten pieces of lines that an entry's
// block costs k_tree_sparse. us per update, all levels / without these:
//   entries   levels   random         ascending            entries   levels   random, ascending in turn
//    65,536   24       24.6 / 19.5    22.8 / 18.4           2048     21        8.4 / 7.8
//   262,144   24       85.4 / 53.8    55.2 / 41.0           3072     22        9.8 / 9.0
//   131,072   22       31.9 / 25.2    23.3 / 20.4           4000     20        9.2 / 8.6
//    16,384   21       12.0 / 11.1    11.2 / 10.2           1024     19        6.3 / 6.0
// (Trees of up to 14 levels, kWgMaxDepth, have kernels that read every level: k_tree_wg and the one-launch step.)
constexpr int kSilentDepth = 15, kSilentLevels = 3;
__host__ __device__ constexpr bool has_silent(int depth) { return depth >= kSilentDepth; }

// A silent node, `up` levels above the leaves, from those under it: requested, and worked out with the additions the tree is built with.
struct SilentNode {
    float4 s0, s1, m0, m1;
    __device__ __forceinline__ void request(const float* sum, const float* mn, uint32_t node, uint32_t up) {
        const uint32_t at = (node << up) & ~3u;  // (of two leaves: the four they are among)
        s0 = *reinterpret_cast<const float4*>(sum + at);
        m0 = *reinterpret_cast<const float4*>(mn + at);
        if (up == 3) {
            s1 = *reinterpret_cast<const float4*>(sum + at + 4);
            m1 = *reinterpret_cast<const float4*>(mn + at + 4);
        }
    }
    __device__ __forceinline__ void take(uint32_t node, uint32_t up, float& s, float& m) const {
        const float sl = s0.x + s0.y, sh = s0.z + s0.w, ml = fminf(m0.x, m0.y), mh = fminf(m0.z, m0.w);
        const float s4 = sl + sh, m4 = fminf(ml, mh);
        s = up == 1 ? (node & 1u ? sh : sl) : up == 2 ? s4 : s4 + ((s1.x + s1.y) + (s1.z + s1.w));
        m = up == 1 ? (node & 1u ? mh : ml) : up == 2 ? m4 : fminf(m4, fminf(fminf(m1.x, m1.y), fminf(m1.z, m1.w)));
    }
};

__device__ __forceinline__ bool valid_priority(float p) { return p >= 0.0f && p <= 3.0e38f; }

// Folds q into the running max priority. Atomics on one address are serialised by the memory
// system (~11 ns each), so the wave first looks at the current value: the max only grows, hence a
// q that does not exceed what is already there can never matter, and nearly every wave skips.
__device__ __forceinline__ void raise_max(float* maxp, float q) {
    if (q > *reinterpret_cast<volatile float*>(maxp)) atomicMax(reinterpret_cast<unsigned int*>(maxp), __float_as_uint(q));
}

// The LDS word a small update's entry bids for its leaf with: the entry's position in the call (plus one, so
// that zero means no bid) above its priority's bits. An integer max over the bids elects the last entry aimed
// at the leaf, and the winner's priority comes back with it (no second trip to the call's arrays).
__device__ __forceinline__ unsigned long long election_key(int64_t j, float p) {
    return ((unsigned long long)(j + 1) << 32) | (unsigned long long)__float_as_uint(p);
}
__device__ __forceinline__ float elected_priority(unsigned long long key) { return __uint_as_float((uint32_t)key); }

// One butterfly step of tile_parents: level 3 + S above the tile, one node per 2^(S+1) lanes.
template <int S, typename Trees>
__device__ __forceinline__ void parents_step(const Trees& a, int g, uint32_t first, uint32_t lane, bool active,
                                             float& cs, float& cm) {
    cs = cs + butterfly_peer<S>(cs);
    cm = fminf(cm, butterfly_peer<S>(cm));
    if (active && g >= 3 + S && (lane & ((2u << S) - 1)) == 0) {
        a.sum[(first >> (3 + S)) + (lane >> (S + 1))] = cs;
        a.mn[(first >> (3 + S)) + (lane >> (S + 1))] = cm;
    }
}

// The g levels above a tile whose nodes (four per lane, vs / vm) are final: parents by in-lane
// operations and wave shuffles, stored by the lanes of dirty blocks (`active`). `first`: heap index
// of the tile's first node. `a`: anything with the two trees, `sum` and `mn` in heap order.
// root_s / root_m (optional): the node eight levels above a full tile, as computed here (what is stored when g >= 8).
// silent: the tile is of leaves, and the levels above them are silent.
template <typename Trees>
__device__ __forceinline__ void tile_parents(const Trees& a, int g, uint32_t first, uint32_t lane, bool active,
                                             const float4& vs, const float4& vm, float* root_s = nullptr,
                                             float* root_m = nullptr, bool silent = false) {
    // one level up: two nodes per lane; two levels up: one node per lane
    const float s0 = vs.x + vs.y, s1 = vs.z + vs.w;
    const float m0 = fminf(vm.x, vm.y), m1 = fminf(vm.z, vm.w);
    float cs = s0 + s1, cm = fminf(m0, m1);
    if (active && !silent && g >= 1) {
        *reinterpret_cast<float2*>(a.sum + (first >> 1) + 2 * lane) = make_float2(s0, s1);
        *reinterpret_cast<float2*>(a.mn + (first >> 1) + 2 * lane) = make_float2(m0, m1);
    }
    if (active && !silent && g >= 2) {
        a.sum[(first >> 2) + lane] = cs;
        a.mn[(first >> 2) + lane] = cm;
    }
    // three to six levels up: 32, 16, 8, 4 nodes per full tile, a butterfly inside each row of 16 lanes
    parents_step<0>(a, g, first, lane, active && !silent, cs, cm);
    parents_step<1>(a, g, first, lane, active, cs, cm);
    parents_step<2>(a, g, first, lane, active, cs, cm);
    parents_step<3>(a, g, first, lane, active, cs, cm);
    // seven and eight levels up: the four rows' values, read as scalars (left + right as everywhere)
    const float s_lo = lane_value(cs, 0) + lane_value(cs, 16), s_hi = lane_value(cs, 32) + lane_value(cs, 48);
    const float m_lo = fminf(lane_value(cm, 0), lane_value(cm, 16)), m_hi = fminf(lane_value(cm, 32), lane_value(cm, 48));
    if (active && g >= 7 && (lane & 31) == 0) {
        a.sum[(first >> 7) + (lane >> 5)] = lane < 32 ? s_lo : s_hi;
        a.mn[(first >> 7) + (lane >> 5)] = lane < 32 ? m_lo : m_hi;
    }
    if (active && g >= 8 && lane == 0) {
        a.sum[first >> 8] = s_lo + s_hi;
        a.mn[first >> 8] = fminf(m_lo, m_hi);
    }
    if (root_s) *root_s = s_lo + s_hi;
    if (root_m) *root_m = fminf(m_lo, m_hi);
}

// The `levels` levels (at most six) above up to 64 consecutive nodes, one to a lane (cs, cm; `first` is the first one's heap
// index); lane 0 is left with the root.
template <int S, typename Trees>
__device__ __forceinline__ void run_step(const Trees& a, int levels, uint32_t first, uint32_t lane, bool active, float& cs, float& cm) {
    if (S < levels) {  // uniform
        if constexpr (S < 4) {
            cs = cs + butterfly_peer<S>(cs);
            cm = fminf(cm, butterfly_peer<S>(cm));
        } else if constexpr (S == 4) {
            const float s0 = lane_value(cs, 0) + lane_value(cs, 16), s1 = lane_value(cs, 32) + lane_value(cs, 48);
            const float m0 = fminf(lane_value(cm, 0), lane_value(cm, 16)), m1 = fminf(lane_value(cm, 32), lane_value(cm, 48));
            cs = lane < 32 ? s0 : s1;
            cm = lane < 32 ? m0 : m1;
        } else {
            cs = lane_value(cs, 0) + lane_value(cs, 32);
            cm = fminf(lane_value(cm, 0), lane_value(cm, 32));
        }
        if (active && (lane & ((2u << S) - 1)) == 0) {
            a.sum[(first + lane) >> (S + 1)] = cs;
            a.mn[(first + lane) >> (S + 1)] = cm;
        }
    }
}
template <typename Trees>
__device__ __forceinline__ void run_parents(const Trees& a, int levels, uint32_t first, uint32_t lane, bool active, float& cs, float& cm) {
    run_step<0>(a, levels, first, lane, active, cs, cm);
    run_step<1>(a, levels, first, lane, active, cs, cm);
    run_step<2>(a, levels, first, lane, active, cs, cm);
    run_step<3>(a, levels, first, lane, active, cs, cm);
    run_step<4>(a, levels, first, lane, active, cs, cm);
    run_step<5>(a, levels, first, lane, active, cs, cm);
}

}  // namespace mrb
