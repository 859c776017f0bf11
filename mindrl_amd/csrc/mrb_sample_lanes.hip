// Samples of thousands of rows, sixteen lanes to a stratum: the kernel and its launch.
#include "mrb_samples.h"
#include "mrb_launch.h"

namespace mrb {

namespace {

// ---------------------------------------------------------------------------
// PER sample, a thousand to some ten thousand rows of up to 20 KB (PriorityReplayBufferSample,
// mindspore_rl/core/priority_replay_buffer.py:70,92-106): SIXTEEN LANES walk a stratum, so a wave walks four at once. The levels 3, 6,
// 9 (and 12) under the root are staged in LDS and walked there three at a time, 32 bytes to a step; of what is left below up to
// eight levels come with one trip, sixteen nodes to a lane. Same outputs, bit for bit, as k_per_sample_wide.
//
// The kernels with a wave or a workgroup to a row read eight kilobytes of tree for each (the 1024 nodes ten levels under the root, and ten
// further down) and dispatch two to six waves; one with a thread to a stratum (k_per_sample_lds) makes three to five dependent trips.
// Here a row costs a kilobyte of tree at most, half a wave, and two trips. What bounds it: up to a few thousand small rows the walkers'
// chain - some 9000 cycles when one wave did everything, of which the weight's power was a quarter and the fields' addresses a fifth, so
// these went to other waves -, beyond that the rows' bytes and the waves to dispatch. us, before / now (fields of a row as in a
// transition: observation, action, reward, next observation, done):
//   41 bytes, 2 * 10^5 slots   2048 rows 6.1 / 4.1, 8192 6.0 / 4.5;   153 bytes, 10^6   2048 rows 6.0 / 4.4, 4096 7.0 / 4.6, 12,288 7.4 / 6.3
//   521 bytes, 2 * 10^5        2048 rows 6.2 / 4.4, 4096 8.2 / 4.8, 16,384 9.0 / 7.9;   521 bytes, 4 * 10^6   1024 rows 5.4 / 4.7, 4096 9.3 / 5.3
//   2.4 KB, 2 * 10^5           2048 rows 7.2 / 5.8, 4096 9.6 / 7.7, 8192 16.6 / 12.8;   7.5 KB   4096 rows 18.6 / 16.5, 16,384 61.8 / 46
//   (46 is the rate of a copy: 246 MB at 5.3 TB/s.)
// ---------------------------------------------------------------------------
constexpr int kLanes = 16;     // that walk a stratum
constexpr int kLanesMost = 8;  // levels they take at once
constexpr int kLanesNarrow = kLanesMostNarrow / kLanes;  // narrow bytes of a lane, at most

// Where level l's nodes lie in LDS: from 2^(l - 2) on, behind those of level l - 3 (l is 3, 6, 9 or 12; level 3's from 4 on,
// where 16 bytes begin).
__device__ __forceinline__ uint32_t top_at(uint32_t node, int l) { return node - (l == 3 ? 4u : 3u << (l - 2)); }

// Walks the g levels (at most eight) of which each of a row of sixteen lanes holds sixteen nodes; group_walk for sixteen lanes, with
// every row of a wave in a walk of its own.
__device__ __forceinline__ uint32_t row_walk(f32x16 v, int g, uint32_t lane, float& mass, float& picked) {
    const f32x8 q8 = __builtin_shufflevector(v, v, 0, 2, 4, 6, 8, 10, 12, 14) + __builtin_shufflevector(v, v, 1, 3, 5, 7, 9, 11, 13, 15);
    const f32x4 q4 = __builtin_shufflevector(q8, q8, 0, 2, 4, 6) + __builtin_shufflevector(q8, q8, 1, 3, 5, 7);
    const float q2a = q4.x + q4.y, q2b = q4.z + q4.w;
    float S[4], P[4];
    S[0] = q2a + q2b;
    P[0] = butterfly_peer<0>(S[0]);
    S[1] = S[0] + P[0];
    P[1] = butterfly_peer<1>(S[1]);
    S[2] = S[1] + P[1];
    P[2] = butterfly_peer<2>(S[2]);
    S[3] = S[2] + P[2];
    P[3] = butterfly_peer<3>(S[3]);
    float m = mass;
    bool ok = true;
#pragma unroll
    for (int s = 3; s >= 0; --s) {
        const bool bit = (lane >> s) & 1;
        const float left = bit ? P[s] : S[s];
        const bool right = s + 4 < g && !(m <= left);
        ok = ok && right == bit;
        m = right ? m - left : m;
    }
    uint32_t in = 0;
    bool r = 3 < g && !(m <= q2a);
    m = r ? m - q2a : m;
    in = r ? 8u : 0u;
    const float h4a = r ? q4.z : q4.x;
    const f32x4 h8 = r ? q8.hi : q8.lo;
    const f32x8 hv = r ? v.hi : v.lo;
    r = 2 < g && !(m <= h4a);
    m = r ? m - h4a : m;
    in += r ? 4u : 0u;
    const float g8a = r ? h8.z : h8.x;
    const f32x4 gv = r ? hv.hi : hv.lo;
    r = 1 < g && !(m <= g8a);
    m = r ? m - g8a : m;
    in += r ? 2u : 0u;
    const float fa = r ? gv.z : gv.x, fb = r ? gv.w : gv.y;
    r = 0 < g && !(m <= fa);
    m = r ? m - fa : m;
    in += r ? 1u : 0u;
    const float mine = r ? fb : fa;
    const uint32_t row = lane & 48u;
    const uint32_t w = (uint32_t)__builtin_ctzll(__ballot(ok) >> row | 0x8000ull);
    mass = __shfl(m, (int)(row + w));
    picked = __shfl(mine, (int)(row + w));
    return 16u * w + (uint32_t)__shfl((int)in, (int)(row + w));
}

// Where a lane's granules of a row lie, kPer lanes to a row (CopyWork's addresses, with the row left open): worked out before the slot is known.
template <int kInF, int kPer>
struct LaneWork {
    const gbyte* from[kInF];
    gbyte* to[kInF];
    uint32_t stride[kInF], bytes[kInF];  // from a row to the next in the buffer, and in the caller's matrix
    uint32_t live;
    __device__ __forceinline__ void prepare(const WidePlan& plan, uint32_t lane) {  // (lane: the number of its first granule)
        live = 0;
#pragma unroll
        for (int j = 0; j < kInF; ++j) {
            if (j * kPer + lane < plan.wide_items) live |= 1u << j;
            from[j] = as_global(plan.f[0].src);  // (a lane with fewer granules than others loads the row's first one for them)
            to[j] = nullptr;
            stride[j] = plan.f[0].ss;
            bytes[j] = 0;
        }
        auto take = [&](int q) {
            const WideField e = plan.f[q];
            const uint32_t units = q < plan.nwide ? (e.rb + 15) >> 4 : 0u;
#pragma unroll
            for (int j = 0; j < kInF; ++j) {
                const uint32_t rel = j * kPer + lane - e.first;  // wraps for granules of earlier fields
                if (rel < units) {
                    const uint32_t at = granule_offset(rel, 4, e.rb);
                    from[j] = as_global(e.src) + at;
                    to[j] = as_global(e.dst) + at;
                    stride[j] = e.ss;
                    bytes[j] = e.rb;
                }
            }
        };
        // the first entries unconditionally: their (wave-uniform) loads go out together at once
#pragma unroll
        for (int q = 0; q < kFastWide; ++q) take(q);
        for (int q = kFastWide; q < plan.nwide; ++q) take(q);
    }
    __device__ __forceinline__ void load(uint32_t slot, granule_t (&held)[kInF]) const {
        if (live == 0) return;
#pragma unroll
        for (int j = 0; j < kInF; ++j) held[j] = __builtin_nontemporal_load((const g16*)(from[j] + (uint64_t)slot * stride[j]));
    }
    __device__ __forceinline__ void store(uint32_t k, const granule_t (&held)[kInF]) const {
#pragma unroll
        for (int j = 0; j < kInF; ++j)
            if (live & (1u << j)) *(g16*)(to[j] + (uint64_t)k * bytes[j]) = held[j];
    }
};

// The bytes of a row's narrow fields, kLanes lanes to a row.
struct LaneBytes {
    const gbyte* from[kLanesNarrow];
    gbyte* to[kLanesNarrow];
    uint32_t stride[kLanesNarrow], bytes[kLanesNarrow];
    __device__ __forceinline__ void prepare(const WidePlan& plan, uint32_t sub) {
#pragma unroll
        for (int j = 0; j < kLanesNarrow; ++j) {
            from[j] = nullptr;
            to[j] = nullptr;
            stride[j] = bytes[j] = 0;
        }
        for (int q = plan.nwide; q < plan.nwide + plan.nnarrow; ++q) {
            const WideField e = plan.f[q];
#pragma unroll
            for (int j = 0; j < kLanesNarrow; ++j) {
                const uint32_t rel = sub + kLanes * j - e.first;  // wraps for bytes of earlier fields
                if (rel < e.rb) {
                    from[j] = as_global(e.src) + rel;
                    to[j] = as_global(e.dst) + rel;
                    stride[j] = e.ss;
                    bytes[j] = e.rb;
                }
            }
        }
    }
    __device__ __forceinline__ void load(uint32_t slot, uint32_t items, uint8_t (&held)[kLanesNarrow]) const {
#pragma unroll
        for (int j = 0; j < kLanesNarrow; ++j) {
            held[j] = 0;
            if (j * kLanes < (int)items && to[j]) held[j] = from[j][(uint64_t)slot * stride[j]];
        }
    }
    __device__ __forceinline__ void store(uint32_t k, uint32_t items, const uint8_t (&held)[kLanesNarrow]) const {
#pragma unroll
        for (int j = 0; j < kLanesNarrow; ++j)
            if (j * kLanes < (int)items && to[j]) to[j][(uint64_t)k * bytes[j]] = held[j];
    }
};

// shape: depth | levels in LDS << 8 | levels of a trip << 16, and, where the counters live on the device:
constexpr int kLanesCounters = 1 << 24;  // the generator's is to be read there
constexpr int kLanesStored = 1 << 25;    // the number of stored rows is
// A workgroup is kStrata / 4 waves that walk, four strata each, and four waves that copy: while the ones walk, the others work out
// where their pieces of a row lie; while these copy, the walkers take the weights.
// kWave: a row's wide granules are a copy wave's, rows in turn; otherwise sixteen lanes' (at most kInF * kLanes of them).
constexpr int kLanesCopyWaves = 4;
template <int kStrata, bool kWave, int kInF>
__global__ __launch_bounds__(16 * kStrata + 64 * kLanesCopyWaves) void k_per_sample_lanes(
    const float* __restrict__ sum, const float* __restrict__ uniforms, const float* __restrict__ mn, int shape, uint32_t batch, uint32_t nrows,
    uint32_t capacity, uint64_t seed, uint64_t calls, SampleTail tail, WidePlan plan) {
    constexpr int kWalkers = kStrata * kLanes, kThreads = kWalkers + 64 * kLanesCopyWaves;
    constexpr int kTop = (1024 + kThreads - 1) / kThreads;
    extern __shared__ float s_top[];  // 5/4 * 2^levels, and two
    __shared__ uint32_t s_slot[kStrata];
    const int depth = shape & 255, levels = (shape >> 8) & 255, trip = (shape >> 16) & 15;
    const uint32_t tid = threadIdx.x, lane = tid & 63, sub = tid & (kLanes - 1);
    const bool walks = __builtin_amdgcn_readfirstlane((int)tid) < kWalkers;
    const uint32_t k0 = blockIdx.x * kStrata;
    // the top, the draws and the total, all at once
    f32x4 low[kTop], few;
    if (levels == 12) {
#pragma unroll
        for (int i = 0; i < kTop; ++i)
            if (1024 % kThreads == 0 || i * kThreads + tid < 1024) low[i] = *reinterpret_cast<const f32x4*>(sum + 4096 + 4 * (i * kThreads + tid));
    }
    const uint32_t small = tid < 128 ? 512 + 4 * tid : tid < 144 ? 64 + 4 * (tid - 128) : tid < 146 ? 8 + 4 * (tid - 144) : 0;
    const bool has_small = small != 0 && small < (2u << levels);
    if (has_small) few = *reinterpret_cast<const f32x4*>(sum + small);
    auto stage = [&] {
        if (levels == 12) {
#pragma unroll
            for (int i = 0; i < kTop; ++i)
                if (1024 % kThreads == 0 || i * kThreads + tid < 1024)
                    *reinterpret_cast<f32x4*>(s_top + top_at(4096 + 4 * (i * kThreads + tid), 12)) = low[i];
        }
        if (has_small) *reinterpret_cast<f32x4*>(s_top + top_at(small, tid < 128 ? 9 : tid < 144 ? 6 : 3)) = few;
        lds_barrier();
    };
    if (walks) {
        const uint32_t k = k0 + tid / kLanes;
        uint32_t opaque_zero = 0;  // (vector loads: see sample_wide_body)
        asm volatile("" : "+v"(opaque_zero));
        const float total = sum[1 + opaque_zero], pmin = mn[1 + opaque_zero];
        float u = (uniforms && k < nrows ? uniforms + k : sum + 1)[opaque_zero];
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t nth = batch < nrows ? k / batch : 0, stratum = k - nth * batch;
        if (!uniforms) u = rng_uniform(seed, (shape & kLanesCounters ? (uint64_t)counters_behind(tail.err)[kCntCalls] + calls : calls) + nth, (uint64_t)stratum);
        stage();
        float mass = (u + (float)stratum) * (total / (float)batch);  // each operation rounded once
        uint32_t node = 1;
        float picked = total;
        for (int d = 3; d <= levels; d += 3) {
            const f32x4* const from = reinterpret_cast<const f32x4*>(s_top + top_at(node << 3, d));
            const f32x4 lo = from[0], hi = from[1];
            node = (node << 3) + walk8(make_float4(lo.x, lo.y, lo.z, lo.w), make_float4(hi.x, hi.y, hi.z, hi.w), mass, picked);
        }
        for (int d = levels; d < depth; d += trip) {  // uniform
            const int g = depth - d < trip ? depth - d : trip;
            f32x4 r0, r1, r2, r3;
            group_request(sum, node, g, (int)sub, r0, r1, r2, r3);
            node = (node << g) + row_walk(group_finish(g, (int)sub, r0, r1, r2, r3), g, lane, mass, picked);
        }
        node -= 1u << depth;
        if (sub == 0) s_slot[tid / kLanes] = node < capacity ? node : capacity - 1;
        lds_barrier();
        int64_t size = tail.size;
        if (shape & kLanesStored) size = counters_behind(tail.err)[kCntSize];
        const float power = powf_det((sub == 0 ? picked : pmin) / total * (float)size, -tail.beta);
        const float max_w = __shfl(power, (int)(lane | (kLanes - 1)));
        if (k < nrows && sub == 0) {
            tail.out_idx[k] = (int64_t)node;
            tail.out_w[k] = power / max_w;
            if (!(total > 0.0f) || total > 3.0e38f) atomicOr(tail.err, MRB_DERR_TOTAL);
            if ((int64_t)node >= size) atomicOr(tail.err, MRB_DERR_UNFILLED);
        }
        return;
    }
    const uint32_t at = (tid - kWalkers) / kLanes;  // the lane's row, of 16
    const uint32_t rows = nrows - k0 < (uint32_t)kStrata ? nrows - k0 : (uint32_t)kStrata;
    stage();
    LaneWork<kInF, kWave ? 64 : kLanes> work;
    LaneBytes bytes;
    work.prepare(plan, kWave ? lane : sub);
    bytes.prepare(plan, sub);
    const uint32_t narrow = plan.narrow_items;
    lds_barrier();
    granule_t held[kInF];
    uint8_t nheld[kLanesNarrow];
    const bool here = at < rows;
    const uint32_t slot = here ? s_slot[at] : 0;
    if (here) bytes.load(slot, narrow, nheld);
    if (!kWave) {
        if (here) {
            work.load(slot, held);
            work.store(k0 + at, held);
        }
    } else {
        const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)((tid - kWalkers) >> 6));
        for (uint32_t base = 0;;) {
            if (wave < rows) work.load((uint32_t)__builtin_amdgcn_readfirstlane((int)s_slot[wave]), held);
            for (uint32_t r = wave; r < rows; r += kLanesCopyWaves) {
                granule_t next[kInF];
                if (r + kLanesCopyWaves < rows) work.load((uint32_t)__builtin_amdgcn_readfirstlane((int)s_slot[r + kLanesCopyWaves]), next);
                work.store(k0 + r, held);
#pragma unroll
                for (int j = 0; j < kInF; ++j) held[j] = next[j];
            }
            base += 64 * kInF;
            if (base >= plan.wide_items) break;
            work.prepare(plan, base + lane);
        }
    }
    if (here) bytes.store(k0 + at, narrow, nheld);
}

// Trips below `levels` staged ones.
int lanes_trips(int depth, int levels) { return (depth - levels + kLanesMost - 1) / kLanesMost; }

}  // namespace

// Staged levels: twelve, or as few of them as take no trip more, which are less to stage (17 levels, 8192 rows of 153 bytes: twelve
// 5.0 us, nine 4.6; 16 levels, 1536 rows: 4.05 / 3.85; 22 levels, 4096 rows of 521 bytes: 5.5 / 5.3), but nine on 18 levels and
// more, where the trips are to memory that is not in the cache.
// Strata of a workgroup where a copy wave carries whole rows: as few as leave the launch's workgroups on the chip all at once, then
// as many as there may be, for the waves there are to dispatch. What the compute units hold, beyond which a launch takes a step (2304 rows
// in the table's last three lines), is some 1024 workgroups of four strata, 768 of eight and 512 of sixteen where a lane holds two
// granules; 768, 512 and 512 where it holds four; 512, 512 and 256 where it holds eight. 2 * 10^5 slots, us with 4 / 8 / 16 strata, and,
// for comparison, a workgroup to a row:
//   row         2048 rows                   2304                        3000                        4096                        5120                        8192
//   1 KB      5.1 /  5.2 /  6.7,  6.4    5.4 /  5.7 /  6.8,  7.4    5.7 /  5.9 /  6.9,  7.6    6.1 /  6.2 /  7.2,  8.5    7.0 /  6.6 /  8.7,  9.6   11.6 /  7.9 /  9.4, 14.5
//   2.4 KB    5.8 /  6.0 /  7.5,  7.1    6.4 /  6.7 /  7.7,  8.1    6.8 /  7.1 /  8.0,  8.4   10.6 /  7.7 /  8.7,  9.5   11.7 / 11.9 / 10.5, 11.1   18.9 / 16.4 / 12.5, 16.4
//   4 KB      6.7 /  7.0 /  8.7,  7.5    7.3 /  7.7 /  8.9,  8.5    8.0 /  8.4 /  9.9,  8.9   12.3 /  9.6 / 11.2, 10.2   14.0 / 14.6 / 13.1, 11.9   21.7 / 19.7 / 16.4, 17.9
//   7.5 KB    9.1 /  9.4 / 11.7, 10.4   14.3 / 12.9 / 12.0, 12.8   14.9 / 14.1 / 13.6, 14.3   18.9 / 17.1 / 16.3, 18.6   22.2 / 21.8 / 22.3, 22.4   31.8 / 29.1 / 26.3, 33.2
//   13 KB    14.2 / 15.0 / 18.6, 15.7   20.9 / 19.8 / 19.1, 16.9   21.9 / 21.6 / 21.1, 21.1   26.8 / 24.6 / 24.8, 26.7   32.1 / 32.0 / 33.9, 31.9   45.6 / 42.5 / 41.8, 48.0
//   20 KB    20.6 / 22.7 / 34.2, 22.9   30.6 / 31.8 / 34.9, 25.0   34.1 / 34.4 / 36.5, 30.9   40.5 / 37.4 / 38.8, 39.8   49.0 / 48.9 / 57.0, 47.8   (6000) 55.0 / 52.9 / 59.6, 55.0
// (Where the workgroup to a row is the faster one, and the lines that keep the lanes away from it: lanes_better, mrb.hip.)
static uint32_t lanes_strata(uint32_t wide, uint32_t rows) {
    if (wide <= 64) return 16;  // sixteen lanes carry a row
    if (wide <= 128) return rows <= 3072 ? 4 : rows <= 8192 ? 8 : 16;
    if (wide <= 256) return rows <= 3072 ? 4 : rows <= 4096 ? 8 : 16;
    if (wide <= 512) return rows <= 2048 ? 4 : rows > 4096 && rows <= 5120 ? 8 : 16;
    return rows <= 2048 ? 4 : rows <= 6144 ? 8 : 16;
}

hipError_t launch_per_sample_lanes(const SampleArgs& a, const WidePlan& plan, int64_t nbatch, hipStream_t s) {
    const int most = a.depth >= 16 ? 12 : (a.depth - 4) / 3 * 3, fewest = a.depth >= 18 ? 9 : 3;
    int levels = most;
    while (levels > fewest && lanes_trips(a.depth, levels - 3) == lanes_trips(a.depth, most)) levels -= 3;
    const int trips = lanes_trips(a.depth, levels), trip = (a.depth - levels + trips - 1) / trips;
    const uint32_t nrows = (uint32_t)(nbatch * a.batch), w = plan.wide_items;
    const uint32_t strata = lanes_strata(w, nrows);
    const SampleTail tail{a.mn, a.out_idx, a.out_w, a.err, a.size, a.beta};
    const int shape = a.depth | levels << 8 | trip << 16 | (a.size < 0 ? kLanesStored | (a.uniforms ? 0 : kLanesCounters) : 0);
    auto* kernel = w <= 16 ? k_per_sample_lanes<16, false, 1> : w <= 32 ? k_per_sample_lanes<16, false, 2> : k_per_sample_lanes<16, false, 4>;
    if (w > 64) {
        if (strata == 4) kernel = w <= 128 ? k_per_sample_lanes<4, true, 2> : w <= 256 ? k_per_sample_lanes<4, true, 4> : k_per_sample_lanes<4, true, 8>;
        else if (strata == 8) kernel = w <= 128 ? k_per_sample_lanes<8, true, 2> : w <= 256 ? k_per_sample_lanes<8, true, 4> : k_per_sample_lanes<8, true, 8>;
        else kernel = w <= 128 ? k_per_sample_lanes<16, true, 2> : w <= 256 ? k_per_sample_lanes<16, true, 4> : k_per_sample_lanes<16, true, 8>;
    }
    launch_kernel(kernel, dim3((nrows + strata - 1) / strata), dim3(kLanes * strata + 64 * kLanesCopyWaves), (size_t)(5 << levels) + 8, s,
                  a.sum, a.uniforms, a.mn, shape, (uint32_t)a.batch, nrows, (uint32_t)a.capacity, a.seed, a.calls, tail, plan);
    return hipGetLastError();
}

}  // namespace mrb
