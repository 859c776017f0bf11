#include "mrb_push_many.h"

#include "../../include/mrb.h"
#include "mrb_launch.h"
#include "mrb_meet.h"
#include "mrb_push.h"
#include "mrb_tree.h"

namespace mrb {

namespace {

struct Trees {
    float* sum;
    float* mn;
};

// ---------------------------------------------------------------------------
// A push under up to 256 leaf tiles, in ONE launch of several workgroups. Each rebuilds kTiles leaf tiles, a wave each, and the
// last to finish takes their roots (see mrb_meet.h) up to the tree's root; what it needs of the levels above is requested when
// the kernel starts. What bounds it is that chain: the launch, a trip to memory, the powers, eight levels, the roots' meeting
// (0.9 us), eight levels more each. One compute unit takes the powers of a tile's four leaves per lane in 1.3 us; with a
// workgroup per tile a thread takes one, 0.35 us, so with priorities kTiles is 1 - until so many workgroups raise the one counter
// that it costs more (11 ns each: 65 tiles 5.9 against 7.0 us with four tiles to a workgroup, 129 6.7 / 7.2, 254 8.4 / 7.7). A single
// tile (kAlone) meets nobody. In front of this one workgroup did it all up to 16 tiles (k_push_run), beyond that launches per eight
// levels (k_tree_update, k_tree_top). Device time per call, us, before / now (i4;f4 rows, 2^24 leaves):
//   with priorities  2 rows 5.4 / 3.5, 200 5.5 / 4.7, 1000 6.5 / 5.2, 4096 10.9 / 5.6, 32768 12.3 / 6.9, 65000 14.1 / 7.8
//   plain            2 rows 3.9 / 3.2 (where they lie under one tile), 4096 9.1 / 4.8, 32768 9.6 / 5.3, 65000 10.1 / 5.9
// (524-byte rows, 2^21 leaves: 4096 rows plain 5.6 / 4.7 and with priorities 8.8 / 5.5, 16384 rows 12.8 / 5.7 and 15.1 / 6.8.) Plain pushes
// in between are k_short_push_run's: the rule, with both sides measured, is at takes_push_many (mrb.hip).
//   plan: depth | columns of workgroups that rebuild tiles << 8; those behind them, (x, y), copy rows of field y
// ---------------------------------------------------------------------------
constexpr uint32_t kManyApart = 160;

template <int kTiles, bool kAlone>
__global__ __launch_bounds__(kWG) void k_push_many(float* sum, float* mn, float* maxp, const float* __restrict__ priorities,
                                                   const RowTable* __restrict__ table, uint32_t first_slot, uint32_t n, uint32_t plan,
                                                   float alpha, uint32_t blocks, ShortIo io) {
    __shared__ float s_s[2], s_m[2];
    __shared__ __attribute__((aligned(16))) float s_q[kTiles == 1 ? kBlockNodes : 4];
    __shared__ float s_most[4];
    __shared__ uint32_t s_new[2], s_before;
    const uint32_t groups = plan >> 8;
    if (__builtin_expect(blockIdx.x >= groups || blockIdx.y != 0, 0)) {
        if (blockIdx.x >= groups) put_fields(table, io, first_slot, n, blockIdx.x - groups, blocks);
        rider_ends();
    }
    const int depth = (int)(plan & 255u);
    const Trees trees{sum, mn};
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t t0 = first_slot / kBlockNodes, tiles = (first_slot + n - 1) / kBlockNodes - t0 + 1;
    const uint32_t unit = blockIdx.x * kTiles + wave;
    const bool work = wave < kTiles && unit < tiles;  // wave-uniform
    // the wave's leaf tile, the priorities of its leaves, the running max and the launch's number
    const uint32_t leaf = (t0 + unit) * kBlockNodes + 4 * lane, leaf_first = (1u << depth) + (t0 + unit) * kBlockNodes;
    float4 ls = make_float4(0.f, 0.f, 0.f, 0.f), lm = ls;
    float old_max = 0.0f, pv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t in = 0;  // bit c: the push writes leaf + c
    const uint32_t mine = (t0 + blockIdx.x) * kBlockNodes + threadIdx.x - first_slot;  // kTiles == 1: the entry whose power this thread takes
    float given = 0.0f;
    if (kTiles == 1) {
        old_max = *maxp;
        if (priorities && mine < n) given = priorities[mine];
    }
    if (work) {
        ls = *reinterpret_cast<const float4*>(sum + leaf_first + 4 * lane);
        lm = *reinterpret_cast<const float4*>(mn + leaf_first + 4 * lane);
        if (kTiles != 1) old_max = *maxp;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t e = leaf + c - first_slot;  // (a slot in front of the first wraps around to a large number)
            if (e < n) {
                in |= 1u << c;
                if (kTiles != 1 && priorities) pv[c] = priorities[e];
            }
        }
    }
    const uint32_t tag = kAlone ? 0 : meet_turn(maxp) + 1;
    // What lies above the leaf tiles: their roots are under one tile or two, held by waves 0 and 1 of the workgroup that comes
    // last (every one may be it, so each requests them), and so on up.
    const uint32_t up = (t0 >> 8) + wave;
    bool holds[kRunLevels];  // wave-uniform
    float4 vs[kRunLevels], vm[kRunLevels];
#pragma unroll
    for (int l = 0; l < kRunLevels; ++l) {
        const int d = depth - kRoundLevels * (l + 1);
        vs[l] = make_float4(0.f, 0.f, 0.f, 0.f);
        vm[l] = vs[l];
        holds[l] = d > 0 && (wave == 0 || (wave == 1 && (l == 0 ? (t0 + tiles - 1) >> 8 != t0 >> 8
                                                               : holds[l - 1] && up >> (8 * l) != t0 >> (8 * l + 8))));
        if (!holds[l]) continue;
        if (d == 1) {  // a level of two nodes
            vs[l].x = sum[2], vs[l].y = sum[3];
            vm[l].x = mn[2], vm[l].y = mn[3];
        } else if (4 * lane < (1u << d)) {
            const uint32_t first = (1u << d) + (up >> (8 * l)) * kBlockNodes + 4 * lane;
            vs[l] = *reinterpret_cast<const float4*>(sum + first);
            vm[l] = *reinterpret_cast<const float4*>(mn + first);
        }
    }
    Meet* const m = meet_of(maxp);
    float rs = 0.0f, rm = 0.0f;
    if (kTiles == 1 && priorities) {
        const bool ok = mine < n && valid_priority(given);
        float q = old_max;
        if (ok) q = powf_det(given, alpha);
        s_q[threadIdx.x] = q;
        if (mine < n && !ok) atomicOr(err_before(maxp), MRB_DERR_PRIORITY);
        const float most = wave_max(ok ? q : 0.0f);
        if (lane == 0) s_most[wave] = most;
        lds_barrier();
    }
    if (work) {
        float q[4] = {old_max, old_max, old_max, old_max}, largest = 0.0f;
        if (kTiles == 1 && priorities) {
            const float4 q4 = *reinterpret_cast<const float4*>(&s_q[4 * lane]);
            q[0] = q4.x, q[1] = q4.y, q[2] = q4.z, q[3] = q4.w;
            largest = fmaxf(fmaxf(s_most[0], s_most[1]), fmaxf(s_most[2], s_most[3]));
        }
        if (kTiles != 1 && priorities) {
            const float4 pw = powf_det_x4(make_float4(pv[0], pv[1], pv[2], pv[3]), alpha);
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
            if (bad) atomicOr(err_before(maxp), MRB_DERR_PRIORITY);
            largest = wave_max(largest);
        }
        if (in & 1u) ls.x = lm.x = q[0];
        if (in & 2u) ls.y = lm.y = q[1];
        if (in & 4u) ls.z = lm.z = q[2];
        if (in & 8u) ls.w = lm.w = q[3];
        if (in) {
            *reinterpret_cast<float4*>(sum + leaf_first + 4 * lane) = ls;
            *reinterpret_cast<float4*>(mn + leaf_first + 4 * lane) = lm;
        }
        tile_parents(trees, kRoundLevels, leaf_first, lane, true, ls, lm, &rs, &rm, has_silent(depth));
        if (lane == 0 && !kAlone) {
            const unsigned long long number = (unsigned long long)tag << 32;
            __hip_atomic_store(&m->root[unit][0], number | __float_as_uint(rs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&m->root[unit][1], number | __float_as_uint(rm), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (priorities) __hip_atomic_store(&m->largest[unit], number | __float_as_uint(largest), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // all four waves' roots are on their way: the workgroup counts itself (see meet(): the last one waits for stores that have
    // been issued, never for a workgroup)
    if (!kAlone) lds_barrier();
    uint32_t before = 0;
    if (threadIdx.x == 0 && !kAlone) before = __hip_atomic_fetch_add(&m->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // waves 0 and 1: the roots under their tiles; waves 2 and 3: the largest power (2) - requested on the chance that this is
    // the last workgroup
    const bool powers = wave == 2 && priorities != nullptr;
    const bool takes = powers || (wave < 2 && holds[0]);
    unsigned long long a[4], b[4];
    auto request = [&]() {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t u = powers ? 4 * lane + c : up * kBlockNodes + 4 * lane + c - t0;
            a[c] = b[c] = (unsigned long long)tag << 32;  // (nobody's)
            if (kAlone) {
                a[c] = __float_as_uint(powers ? fmaxf(fmaxf(s_most[0], s_most[1]), fmaxf(s_most[2], s_most[3])) : rs);
                b[c] = __float_as_uint(rm);
            } else if (takes && u < tiles) {
                a[c] = __hip_atomic_load(powers ? &m->largest[u] : &m->root[u][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (!powers) b[c] = __hip_atomic_load(&m->root[u][1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    };
    request();
    if (!kAlone) {
        if (threadIdx.x == 0) s_before = before;
        lds_barrier();
        if (!meet_last(s_before, groups)) return;  // uniform
    }
    bool late = false;
    if (takes && !kAlone) {
        for (uint32_t looks = 0; looks < kMeetLooks; ++looks) {
            bool open = false;
#pragma unroll
            for (int c = 0; c < 4; ++c) open = open || !meet_here(a[c], tag) || !meet_here(b[c], tag);
            late = __any(open);
            if (!late) break;
            request();
        }
    }
    if (__builtin_expect(late, 0)) {  // what did not come stays as it was (see mrb_meet.h); a look at each root below would cost every push 0.1 us
        const float was_s[4] = {vs[0].x, vs[0].y, vs[0].z, vs[0].w}, was_m[4] = {vm[0].x, vm[0].y, vm[0].z, vm[0].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (meet_here(a[c], tag) && meet_here(b[c], tag)) continue;
            a[c] = powers ? 0 : __float_as_uint(was_s[c]);
            b[c] = __float_as_uint(was_m[c]);
        }
        if (lane == 0) atomicOr(err_before(maxp), MRB_DERR_OVERLAP);
    }
    if (!kAlone) {
        lds_barrier();  // every wave has the roots that it waited for
        if (threadIdx.x == kWG - 1) meet_over(m, tag);  // (of the wave that waits for none)
    }
    if (powers) {
        float largest = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) largest = fmaxf(largest, __uint_as_float((uint32_t)a[c]));
        largest = wave_max(largest);
        // (every leaf that takes the running max as it was has been written)
        if (lane == 0 && largest > 0.0f) raise_max(maxp, largest);
    }
    if (takes && !powers) {
        float* const s4[4] = {&vs[0].x, &vs[0].y, &vs[0].z, &vs[0].w};
        float* const m4[4] = {&vm[0].x, &vm[0].y, &vm[0].z, &vm[0].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (up * kBlockNodes + 4 * lane + c - t0 < tiles) {
                *s4[c] = __uint_as_float((uint32_t)a[c]);
                *m4[c] = __uint_as_float((uint32_t)b[c]);
            }
        }
    }
#pragma unroll
    for (int l = 0; l < kRunLevels; ++l) {
        const int d = depth - kRoundLevels * (l + 1);
        if (d <= 0) break;  // uniform
        if (l > 0 && kAlone) {
            // one path of tiles, all wave 0's (its last root is in every lane)
            if (!holds[l]) break;
            const uint32_t node = up >> (8 * (l - 1));
            if ((node & 255u) / 4 == lane) {
                switch (node & 3u) {
                    case 0: vs[l].x = rs, vm[l].x = rm; break;
                    case 1: vs[l].y = rs, vm[l].y = rm; break;
                    case 2: vs[l].z = rs, vm[l].z = rm; break;
                    default: vs[l].w = rs, vm[l].w = rm; break;
                }
            }
        } else if (l > 0) {
            if (lane == 0 && wave < 2) {
                s_s[wave] = rs;
                s_m[wave] = rm;
                s_new[wave] = holds[l - 1];
            }
            lds_barrier();
            if (holds[l]) {
#pragma unroll
                for (uint32_t u = 0; u < 2; ++u) {
                    // the node that wave u's tile has as its root, if it lies in this wave's tile
                    const uint32_t node = ((t0 >> 8) + u) >> (8 * (l - 1));
                    if (!s_new[u] || node >> 8 != up >> (8 * l) || (node & 255u) / 4 != lane) continue;
                    const float ps = s_s[u], pm = s_m[u];
                    switch (node & 3u) {
                        case 0: vs[l].x = ps, vm[l].x = pm; break;
                        case 1: vs[l].y = ps, vm[l].y = pm; break;
                        case 2: vs[l].z = ps, vm[l].z = pm; break;
                        default: vs[l].w = ps, vm[l].w = pm; break;
                    }
                }
            }
            lds_barrier();  // read before the next level's are written
        }
        if (!holds[l]) continue;  // wave-uniform
        if (d == 1) {
            if (lane == 0) {
                sum[1] = vs[l].x + vs[l].y;
                mn[1] = fminf(vm[l].x, vm[l].y);
            }
        } else {
            tile_parents(trees, d < kRoundLevels ? d : kRoundLevels, (1u << d) + (up >> (8 * l)) * kBlockNodes, lane, 4 * lane < (1u << d),
                         vs[l], vm[l], &rs, &rm);
        }
    }
}

}  // namespace

hipError_t launch_push_many(const RowTable* table, const ShortIo& io, const IoTable& t, float* sum, float* mn, float* maxp, const float* priorities,
                            int64_t first_slot, int64_t n, int depth, float alpha, hipStream_t s) {
    const uint32_t tiles = (uint32_t)((first_slot + n - 1) / kBlockNodes - first_slot / kBlockNodes + 1);
    const uint32_t per = tiles == 1 || (priorities && tiles <= kManyApart) ? 1 : 4, groups = (tiles + per - 1) / per;
    uint32_t blocks;
    const dim3 grid = put_grid(t, groups, blocks);
    auto* kernel = k_push_many<4, false>;
    if (per == 1) kernel = k_push_many<1, false>;
    if (tiles == 1) kernel = k_push_many<1, true>;
    launch_kernel(kernel, grid, dim3(kWG), 0, s, sum, mn, maxp,
                  priorities, table, (uint32_t)first_slot, (uint32_t)n, (uint32_t)depth | groups << 8, alpha, blocks, io);
    return hipGetLastError();
}

}  // namespace mrb
