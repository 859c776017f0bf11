// What mrb_returns.h takes from the device's language and from the header of this name beside it, on the host: a workgroup's lanes
// are fibers that run one after the other, in an order of g_rng's, each as far as the next place where its wave or its workgroup
// meets. Between two such places nothing orders the lanes.
#pragma once
#include <setjmp.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <random>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(x)
#define __builtin_amdgcn_sched_barrier(x) (void)0
using hipError_t = int;
using hipStream_t = void*;

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Index { uint32_t x; };
inline Index threadIdx, blockIdx;

namespace sim {

struct Lane {
    ucontext_t start;
    jmp_buf at;
    bool started = false, done = false;
    int waits = 0;  // 1: for its wave, 2: for its workgroup
    std::vector<char> stack = std::vector<char>(65536);
};
inline std::vector<Lane> g_lanes;
inline uint32_t g_now;
inline std::function<void()> g_body;
inline jmp_buf g_back;
inline std::mt19937 g_rng(1);

inline void wait(int kind) {
    Lane& me = g_lanes[g_now];
    me.waits = kind;
    if (!_setjmp(me.at)) _longjmp(g_back, 1);
}
inline void enter() {
    g_body();
    g_lanes[g_now].done = true;
    _longjmp(g_back, 1);
}
inline void go_on(uint32_t i) {
    g_now = i;
    threadIdx.x = i;
    Lane& l = g_lanes[i];
    if (_setjmp(g_back)) return;
    if (l.started) _longjmp(l.at, 1);
    l.started = true;
    setcontext(&l.start);
}
// Runs one workgroup of `threads` to its end; false: lanes wait at different places.
inline bool run(uint32_t block, uint32_t threads, std::function<void()> body) {
    blockIdx.x = block;
    g_body = std::move(body);
    g_lanes = std::vector<Lane>(threads);
    for (auto& l : g_lanes) {
        getcontext(&l.start);
        l.start.uc_stack.ss_sp = l.stack.data();
        l.start.uc_stack.ss_size = l.stack.size();
        l.start.uc_link = nullptr;
        makecontext(&l.start, enter, 0);
    }
    std::vector<uint32_t> order(threads);
    for (uint32_t i = 0; i < threads; ++i) order[i] = i;
    for (;;) {
        std::shuffle(order.begin(), order.end(), g_rng);
        bool moved = false;
        for (const uint32_t i : order)
            if (!g_lanes[i].done && !g_lanes[i].waits) go_on(i), moved = true;
        bool all = true, ended = true;
        for (uint32_t w = 0; w < threads; w += 64) {
            bool here = true;
            for (uint32_t i = w; i < w + 64; ++i) here = here && g_lanes[i].waits == 1;
            for (uint32_t i = w; here && i < w + 64; ++i) g_lanes[i].waits = 0;
            moved = moved || here;
        }
        for (auto& l : g_lanes) {
            ended = ended && l.done;
            all = all && l.waits == 2;
        }
        if (ended) return true;
        if (all)
            for (auto& l : g_lanes) l.waits = 0;
        else if (!moved)
            return false;
    }
}

}  // namespace sim

namespace mrb {

inline void lds_barrier() { sim::wait(2); }
inline void wave_lds_fence() { sim::wait(1); }
inline int64_t g_through = 0;  // results that were stored so
template <typename V>
inline void store_through(void* to, V v) {
    memcpy(to, &v, sizeof(v));
    g_through += sizeof(v) / 4;
}

}  // namespace mrb
