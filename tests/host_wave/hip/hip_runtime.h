// Waves on the host: just enough of the device's language to run mrb_meet.h on the CPU. A lane is a fiber; a wave's lanes meet at
// the operations that look across lanes; every memory operation on a shared word gives another wave a turn, and a store may
// arrive later than what follows it, as on the device.
#pragma once
#include <setjmp.h>
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <functional>
#include <memory>
#include <random>
#include <vector>

#define __device__
#define __host__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_AGENT 0

struct float4 { float x, y, z, w; };
inline float4 make_float4(float x, float y, float z, float w) { return float4{x, y, z, w}; }
inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }

namespace sim {

struct Lane {
    ucontext_t start;
    jmp_buf at;
    bool started = false;
    std::vector<char> stack = std::vector<char>(32768);
    bool done = false, waits = false;
    unsigned long long value = 0;  // what it brought to the operation it waits at
};
struct Wave {
    std::vector<std::unique_ptr<Lane>> lanes;
    unsigned long long first = 0, ballot = 0;
    std::function<void(uint32_t)> body;
};
struct Late {
    unsigned long long* to;
    unsigned long long value;
};

inline jmp_buf g_back;
inline Wave* g_wave;
inline Lane* g_lane;
inline std::vector<Late> g_late;  // stores on their way
inline std::mt19937 g_rng(1);
inline uint64_t g_steps;          // turns taken

// (a fiber is entered once by its context and then by jumps, which need no system call)
inline void yield() {
    if (!_setjmp(g_lane->at)) _longjmp(g_back, 1);
}
inline void go_on() {
    if (_setjmp(g_back)) return;
    if (g_lane->started) _longjmp(g_lane->at, 1);
    g_lane->started = true;
    setcontext(&g_lane->start);
}
inline unsigned long long together(unsigned long long value, bool ballot) {
    Lane* const me = g_lane;
    Wave* const wave = g_wave;
    me->value = value;
    me->waits = true;
    yield();
    return ballot ? wave->ballot : wave->first;
}
inline void arrive(size_t i) {
    *g_late[i].to = g_late[i].value;
    g_late.erase(g_late.begin() + (long)i);
}
inline void enter() {
    for (size_t i = 0; i < g_wave->lanes.size(); ++i)
        if (g_wave->lanes[i].get() == g_lane) g_wave->body((uint32_t)i);
    g_lane->done = true;
    yield();
}

// Runs the waves to their ends, in an order of g_rng's; false: not ended within `most` turns.
inline bool run(std::vector<Wave>& waves, uint64_t most) {
    for (auto& w : waves)
        for (int i = 0; i < 64; ++i) {
            w.lanes.push_back(std::make_unique<Lane>());
            Lane& l = *w.lanes.back();
            getcontext(&l.start);
            l.start.uc_stack.ss_sp = l.stack.data();
            l.start.uc_stack.ss_size = l.stack.size();
            l.start.uc_link = nullptr;
            makecontext(&l.start, enter, 0);
        }
    std::vector<Wave*> open;
    for (auto& w : waves) open.push_back(&w);
    g_steps = 0;
    while (!open.empty()) {
        if (++g_steps > most) return false;
        if (!g_late.empty() && g_rng() % 8 == 0) arrive(g_rng() % g_late.size());
        const size_t k = g_rng() % open.size();
        g_wave = open[k];
        bool ended = true, all = true;
        for (auto& l : g_wave->lanes) {
            if (!l->done && !l->waits) {
                g_lane = l.get();
                go_on();
            }
            ended = ended && l->done;
            all = all && (l->done || l->waits);
        }
        if (ended) {
            open.erase(open.begin() + (long)k);
        } else if (all) {
            g_wave->ballot = 0;
            bool some = false;
            for (int i = 0; i < 64; ++i) {
                Lane& l = *g_wave->lanes[(size_t)i];
                if (l.done) continue;
                if (!some) g_wave->first = l.value;
                some = true;
                g_wave->ballot |= (unsigned long long)(l.value != 0) << i;
                l.waits = false;
            }
        }
    }
    while (!g_late.empty()) arrive(0);
    return true;
}

template <typename T>
void store(T* to, T value) {
    if (sizeof(T) == 8) {
        g_late.push_back({(unsigned long long*)to, (unsigned long long)value});  // (on its way)
    } else {
        *to = value;
    }
}
template <typename T>
T load(const T* from) {
    return *from;  // (a wave's loads are followed by an operation across its lanes, which is a turn's end)
}
template <typename T>
T add(T* to, T value) {
    yield();
    const T v = *to;
    *to += value;
    return v;
}

}  // namespace sim

#define __hip_atomic_store(p, v, order, scope) sim::store(p, v)
#define __hip_atomic_load(p, order, scope) sim::load(p)
#define __hip_atomic_fetch_add(p, v, order, scope) sim::add(p, v)
#define __builtin_amdgcn_readfirstlane(x) ((int)(uint32_t)sim::together((uint32_t)(x), false))
inline unsigned long long __ballot(bool x) { return sim::together(x, true); }
inline bool __any(bool x) { return sim::together(x, true) != 0; }
inline void atomicOr(uint32_t* p, uint32_t v) { *p |= v; }
