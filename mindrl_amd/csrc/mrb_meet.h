// How workgroups of one launch hand their subtrees' roots to the last of them.
//
// Every workgroup leaves its root, sum and minimum, in a word of its own and raises a counter; the one that finds it was the
// last takes all the roots and rebuilds what lies above them. A second launch for those levels costs 1.5 us on the device and
// 2.5 us of the host's time (its arguments go to device memory and are read back once); a fence per workgroup would cost
// 60 ns each, one after the other, on a part whose dies have caches of their own. So there is no fence: a root's words carry
// the launch's number beside the value, the last workgroup looks at that, and reads again those (few, if any) whose stores
// the counter has overtaken. It waits for stores that are on their way, never for a workgroup that has yet to run, so it
// ends however the workgroups are scheduled; nothing has to be cleared between launches; and a launch replayed from a graph
// finds its number on the device.
//
// Calls that change one buffer must not run side by side (mrb.h). Where two did all the same, they share the counters and the
// number, so what the counters hold afterwards is anybody's guess and a root may never come. Two things keep that from outliving
// those calls. Whoever counts itself at or behind the last place, not only at it, takes the roots, after all of them have
// this launch's number: from whatever count a launch starts, at least one workgroup does, with every root, and several write
// the same values. And the wait ends after kMeetLooks looks, which leaves the roots that did not come as they were and says so
// in the buffer's flags.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mrb.h"

namespace mrb {

constexpr int kMeetMost = 256;  // roots: a tile's worth of nodes
// Atomics on one word are served one after the other, 11 ns each. More than kMeetDirect workgroups count themselves in groups of
// 16 roots, of which the last to come counts for its group: one trip more (0.6 us), 32 in a row at most instead of 256.
constexpr int kMeetGroup = 16;
constexpr uint32_t kMeetDirect = 96;
// Looks at the roots at most. One is a trip to memory, half a microsecond or more, and stores on their way take a few: 30 ms and more.
constexpr uint32_t kMeetLooks = 1u << 16;

// kMeetBehindMaxp bytes behind a buffer's running max (one allocation, see counters_behind).
constexpr int kMeetBehindMaxp = 64;
struct Meet {
    uint32_t arrived;  // of the launch in progress
    uint32_t turn;     // launches so far, of a lap of 2^32 - 1
    uint32_t pad[30];
    uint32_t group[kMeetMost / kMeetGroup][32];  // as `arrived`, of the workgroups of a group; a line each
    unsigned long long root[kMeetMost][2];   // launch number << 32 | bits: sum, minimum
    unsigned long long largest[kMeetMost];  // and, of a push, the largest power
};

__device__ __forceinline__ Meet* meet_of(float* maxp) { return reinterpret_cast<Meet*>(reinterpret_cast<char*>(maxp) + kMeetBehindMaxp); }

// The number of launches before this one; its own is one more, never 0, which is what a word that no launch of the lap has
// written holds (requested when a kernel starts: the last workgroup moves it on).
__device__ __forceinline__ uint32_t meet_turn(float* maxp) {
    return __hip_atomic_load(&meet_of(maxp)->turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether a workgroup that `before` others came ahead of, of `count` that come, is to take the roots.
__device__ __forceinline__ bool meet_last(uint32_t before, uint32_t count) { return before + 1 >= count; }
__device__ __forceinline__ bool meet_here(unsigned long long word, uint32_t tag) { return (uint32_t)(word >> 32) == tag; }
// By one thread, when every root has been looked at for the last time: ready for the next launch.
__device__ __forceinline__ void meet_over(Meet* m, uint32_t tag) {
    m->arrived = 0;
    m->turn = tag;
    if (__builtin_expect(tag == 0xffffffffu, 0)) {  // the lap's last: its numbers come again
        m->turn = 0;
#pragma clang loop unroll(disable)
        for (int r = 0; r < kMeetMost; ++r) m->root[r][0] = m->root[r][1] = m->largest[r] = 0;
    }
}

// Who meets: a bit for each of a lane's four roots that changes - the same in every workgroup -, and, worked out from them by
// one whole wave (early, while it waits for memory), how many count themselves.
struct MeetPlan {
    uint32_t changed;
    uint32_t count;     // on `arrived`
    uint32_t of_group;  // on the group's counter; 0: there are none
};
__device__ __forceinline__ MeetPlan meet_plan(uint32_t changed, uint32_t which, uint32_t lane) {
    MeetPlan p{changed, 0, 0};
    uint32_t of = 0;
    unsigned long long any = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const unsigned long long bits = __ballot(changed >> c & 1u);
        p.count += (uint32_t)__popcll(bits);
        of += (uint32_t)__popcll(bits >> (which / kMeetGroup * (kMeetGroup / 4)) & 15u);
        any |= bits;
    }
    if (p.count <= kMeetDirect) return p;  // uniform
    any |= any >> 1;
    any |= any >> 2;
    p.count = (uint32_t)__popcll(any & 0x1111111111111111ull);
    p.of_group = of;
    return p;
}

// Called by one whole wave of each of the workgroups that change their root (number `which`). In the last one's it returns true;
// vs, vm - four roots to a lane, as memory held them when the kernel started - then hold the new ones where
// the plan has the root's bit. (Two trips to memory: the counter's answer, which the compiler waits for where one lane asks, and
// the roots, more where stores are still on their way.)
__device__ __forceinline__ bool meet(float* maxp, uint32_t* err, uint32_t turn, uint32_t which, float root_s, float root_m, uint32_t lane,
                                     const MeetPlan& p, float4& vs, float4& vm) {
    const uint32_t changed = p.changed;
    Meet* const m = meet_of(maxp);
    const uint32_t tag = turn + 1;
    uint32_t before = 0;
    if (lane == 0) {
        const unsigned long long number = (unsigned long long)tag << 32;
        __hip_atomic_store(&m->root[which][0], number | __float_as_uint(root_s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&m->root[which][1], number | __float_as_uint(root_m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::: "memory");  // issued in this order
    }
    if (p.of_group) {  // uniform
        uint32_t* const counter = m->group[which / kMeetGroup];
        if (lane == 0) before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!meet_last((uint32_t)__builtin_amdgcn_readfirstlane((int)before), p.of_group)) return false;
        if (lane == 0) *counter = 0;  // ready for the next launch
    }
    if (lane == 0) {
        before = __hip_atomic_fetch_add(&m->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float s[4] = {vs.x, vs.y, vs.z, vs.w}, t[4] = {vm.x, vm.y, vm.z, vm.w};
    for (uint32_t looks = 1;; ++looks) {
        unsigned long long a[4], b[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            a[c] = b[c] = 0;
            if (changed >> c & 1u) {
                a[c] = __hip_atomic_load(&m->root[4 * lane + c][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                b[c] = __hip_atomic_load(&m->root[4 * lane + c][1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (!meet_last((uint32_t)__builtin_amdgcn_readfirstlane((int)before), p.count)) return false;
        bool open = false;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (changed >> c & 1u) {
                open = open || !meet_here(a[c], tag) || !meet_here(b[c], tag);
                s[c] = __uint_as_float((uint32_t)a[c]);
                t[c] = __uint_as_float((uint32_t)b[c]);
            }
        }
        if (!__any(open)) break;
        if (looks == kMeetLooks) {
            const float was_s[4] = {vs.x, vs.y, vs.z, vs.w}, was_m[4] = {vm.x, vm.y, vm.z, vm.w};
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (!meet_here(a[c], tag) || !meet_here(b[c], tag)) s[c] = was_s[c], t[c] = was_m[c];
            if (lane == 0) atomicOr(err, MRB_DERR_OVERLAP);
            break;
        }
    }
    vs = make_float4(s[0], s[1], s[2], s[3]);
    vm = make_float4(t[0], t[1], t[2], t[3]);
    if (lane == 0) meet_over(m, tag);
    return true;
}

}  // namespace mrb
