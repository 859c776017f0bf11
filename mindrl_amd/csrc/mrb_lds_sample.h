// Samples of thousands of rows: the LDS-top kernels' body (no kernels here).
#pragma once
#include <type_traits>

#include "mrb_samples.h"

namespace mrb {

// ---------------------------------------------------------------------------
// PER sample, many narrow rows: one workgroup per kStrata strata. The top
// `lds_levels` levels of the sum tree (nodes [1, 2 << lds_levels)) are staged
// in LDS once per workgroup, so each thread's descent reads HBM/L2 only for
// the levels below; then the workgroup gathers its rows with coalesced
// writes. Same outputs, bit for bit, as k_per_sample_wide.
// What bounds it: a chain of trips (the arguments and the top, the descent's two or three, the rows), and, with few
// workgroups, the compute units that have none: 256 strata to a workgroup used 64 of them for a batch of 16,384. The
// rows' granules are numbered over all fields and four to a thread are in flight at once; field by field every field was
// a trip of its own. 16,384 rows of
// 153 bytes 17.1 -> 7.9 us, 13,764 of 139 bytes 15.8 -> 8.1, 16,384 of 521 bytes 35 -> 11.1.
// ---------------------------------------------------------------------------
// sum .. calls repeat members of `a` as plain leading parameters: those are preloaded into scalar
// registers, so the staging loads go out when the wave starts instead of a round trip to the
// kernel-argument segment later.
// kLarge: large fields are copied by themselves, four granules of a thread in flight: what a granule's field is need not be looked up for
// each, and where it lies is a multiplication instead of a division - these kernels, not the memory, were what bounded large rows. Batches
// of more than 20 MB are stored through the L2 (store_granule). us, all by the lookup / so, from 2 * 10^5 rows:
//   row       1 x 12,288 rows   1 x 16,384     2 x 12,288     5 x 8192       5 x 16,384     1 x 65,536     1 x 131,072 (256 strata to a workgroup)
//   128 B                                                                                                  16.2 / 12.8
//   512 B                                                                                                  45.6 / 28.7
//   1 KB                                                                     36.6 / 30.9    31.7 / 25.8    78.4 / 47.0
//   2.4 KB                                     32.8 / 25.4    47.0 / 42.2    87.3 / 84.9    73.5 / 69.2
//   4 KB      26.4 / 21.3       34.1 / 26.5    49.8 / 42.5    74.5 / 70.7                   115.1 / 106.4
//   6 KB      38.8 / 27.6       46.2 / 38.4    70.2 / 62.5   102.0 / 100.5
// (With ordinary loads 2.4 KB 28.6, 45.1, 4 KB 45.4, 71.2.)
// A field is large with 2048 granules and more for a workgroup's strata. (Batches of fewer strata than a workgroup has bring a thread
// less, and are not slower so: 4096 batches of 3 rows of 4.8 KB 39.6 / 35.3, of 8 rows of 2 KB 39.6 / 36.1, of 8 rows of twice 1 KB 38.7 / 39.3,
// 2048 of 40 rows of twice 512 bytes 37.8 / 38.3.)
// But rows of a small buffer come from the caches, many of them several times, and the streaming loads of this copy do not find
// them there for long; least of all the rows of no whole granules, whose lines two granules share. What the rows held take is compared with
// a line for odd rows, and for others with one for batches of up to 64 MB and one for larger ones. us, all by the lookup / so, by the MB of the rows held, each behind calls of the other:
//                                                    10            20            30            45            64            90            128           180           256
//   1 KB, 1 x 42,000 (43 MB)                    19.8 / 13.7   19.8 / 15.5   19.5 / 17.7   20.1 / 17.7   20.9 / 17.8   21.6 / 18.2
//   3 KB, 1 x 21,000 (65 MB)                    23.3 / 16.9   23.7 / 19.9   24.5 / 23.9   25.7 / 23.5   27.1 / 23.4   28.3 / 23.7
//   1 KB, 1 x 80,000 (83 MB)                                  23.2 / 26.6   24.1 / 27.7   25.6 / 26.5   27.4 / 26.1   28.9 / 27.8
//   4 KB, 1 x 21,000 (86 MB)                                  28.4 / 25.3   29.2 / 30.7   30.6 / 30.4   31.8 / 28.9   33.5 / 29.2
//   4 KB, 2 x 6200 (51 MB)                      18.7 / 18.1   19.6 / 20.9   20.2 / 19.8   21.2 / 20.8   21.7 / 21.4   22.8 / 22.0
//   1 KB, 2 x 31,000 (64 MB)                    20.1 / 20.9   21.3 / 23.4   22.5 / 21.8   23.8 / 22.3   24.7 / 23.3   25.3 / 24.0
//   2.4 KB, 5 x 5000 (60 MB)                    21.9 / 24.6   23.3 / 24.4   24.0 / 24.8   25.0 / 25.5   25.7 / 25.6   26.5 / 25.7
//   3 KB, 5 x 5000 (77 MB)                      25.3 / 27.9   27.1 / 28.0   28.0 / 29.3   28.7 / 30.0   29.9 / 30.5   30.6 / 30.6   31.6 / 30.7
//   1.1 KB (odd), 1 x 42,000 (47 MB)            22.5 / 18.3   22.1 / 22.0   21.9 / 24.8   22.8 / 24.5                 24.5 / 23.8   25.3 / 23.9   26.3 / 24.3
//   1.1 KB (odd), 5 x 5000 (28 MB)              14.9 / 18.2   15.9 / 17.9   16.3 / 17.9   16.8 / 17.9   17.2 / 18.1   17.4 / 18.1   17.9 / 18.1   18.4 / 18.4   18.7 / 18.6
//   3 KB (odd), 1 x 12,400 (43 MB)              20.3 / 17.8   20.0 / 22.1   19.9 / 23.3   20.4 / 22.5   21.4 / 22.0   22.2 / 22.1   22.7 / 22.5   23.3 / 22.6   24.4 / 23.0
//   1.1 KB (odd), 5 x 12,500 (69 MB)            23.1 / 30.0   24.2 / 33.4   25.2 / 30.8   26.4 / 30.1   27.7 / 30.1   28.7 / 30.4   29.7 / 30.4   30.8 / 31.0   32.6 / 31.2
//   3 KB (odd), 5 x 5000 (87 MB)                              32.3 / 38.0   33.4 / 38.9   34.4 / 39.2   35.5 / 40.0   36.4 / 39.8   37.2 / 40.4   40.2 / 40.1   43.5 / 40.5
//   512 B, 1 x 98,400 (51 MB, 256 strata)       30.1 / 14.8   30.4 / 20.2   30.6 / 20.2   31.2 / 20.7
//   512 B, 1 x 180,000 (94 MB, 256 strata)                    33.1 / 29.0   33.9 / 28.9   34.4 / 28.3   35.8 / 29.0   37.6 / 31.6
// (Where nothing else comes between calls, the lookup finds more of 30 to 100 MB in the memory's cache: 60 MB, 1 KB 1 x 42,000 18.6 / 17.6,
// 2 x 10,500 12.3 / 12.2, 5 x 5000 13.2 / 14.0, 2.4 KB 5 x 5000 23.7 / 25.7, 4 KB 2 x 10,500 33.3 / 30.3; of odd ones 100 MB, 1.1 KB 5 x 5000 15.8 / 18.2.
// Odd rows in batches of more than 96 MB keep the lookup, whatever the buffer; out of 3 GB 3 KB 1 x 50,000 takes 72.0, and would take 62.8.)
// ---------------------------------------------------------------------------
constexpr int kLargeTrip = 4;
constexpr uint64_t kLargeOdd = 96ull << 20;
inline bool large_field(const IoTable& t, int f, int strata, int64_t nbatch, uint64_t bytes, uint64_t held) {
    if (t.vec_log2[f] != 4 || t.units[f] * (uint64_t)strata < (uint64_t)(2 * kLargeTrip * kWG) || t.units[f] > 1u << 14) return false;
    const uint64_t mb = 1 << 20;
    if (t.row_bytes[f] % 16 != 0) return bytes <= kLargeOdd && held > 144 * mb;
    return strata == 256 || held > (bytes > 64 * mb ? 56 * mb : nbatch > 1 ? 24 * mb : 0);
}
__device__ __forceinline__ uint8_t* uniform_pointer(uint8_t* p) {
    const uint64_t v = (uint64_t)p;
    return (uint8_t*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

// rest: granules of a row in the other fields. large (kLarge): a bit for each field that is large; bit 31: store through the L2. blockIdx.y:
// the batch, of several that are drawn at once (each stratified on its own, with the generator's next call counter).
template <int kStrata, bool kLarge>
__device__ __forceinline__ void sample_lds(const float* __restrict__ sum, const float* __restrict__ uniforms, const float* __restrict__ mn, int depth,
                                           int lds_levels, int batch, float beta, uint64_t seed, uint64_t calls, uint32_t rest, uint32_t large,
                                           const SampleArgs& a, const IoTable& t) {
    extern __shared__ float s_top[];  // [2 << lds_levels] floats, then kStrata + 1 int64: the slots, the number of stored rows
    __shared__ float s_max_w;
    // the field table (see k_res_push); units: of the fields that make up `rest`
    __shared__ uint8_t *s_io[MRB_MAX_FIELDS], *s_store[MRB_MAX_FIELDS];
    __shared__ uint32_t s_bytes[MRB_MAX_FIELDS], s_stride[MRB_MAX_FIELDS], s_units[MRB_MAX_FIELDS], s_vl[MRB_MAX_FIELDS];
    __shared__ uint32_t s_large[kLarge ? MRB_MAX_FIELDS : 1];  // granules of a row of a large field, else 0
    const uint32_t ntop = 2u << lds_levels;
    int64_t* s_slot = reinterpret_cast<int64_t*>(s_top + (ntop < 4 ? 4 : ntop));
    const int64_t row0 = (int64_t)blockIdx.y * batch;  // the batch's first row of the call's
    const int64_t k0 = (int64_t)blockIdx.x * kStrata;
    const int64_t k = threadIdx.x < kStrata ? k0 + threadIdx.x : batch;
    if (threadIdx.x >= kWG) {
        const int f = (int)threadIdx.x - kWG;
        if (f < t.nfields) {
            s_io[f] = t.io[f];
            s_store[f] = t.store[f];
            s_bytes[f] = t.row_bytes[f];
            s_stride[f] = t.stride[f];
            s_units[f] = (f < kLdsOwn && t.units[f] == 1) || (kLarge && large >> f & 1u) ? 0 : t.units[f];
            if (kLarge) s_large[f] = large >> f & 1u ? t.units[f] : 0;
            s_vl[f] = t.vec_log2[f];
        }
        // The helper wave: the weights' common denominator (pmin / total * size)^-beta, once per
        // workgroup, off the strata's path (two loads and a power: as long as staging the top).
        // (the number of stored rows: the argument, or read from the device when the counters live there)
        if (threadIdx.x == kWG) s_slot[kStrata] = a.size >= 0 ? a.size : counters_behind(a.err)[kCntSize];
        __syncthreads();
        if (threadIdx.x == kWG) s_max_w = powf_det(mn[1] / sum[1] * (float)s_slot[kStrata], -beta);
        __syncthreads();
        return;
    }
    // the stratum's draw is requested together with the top of the tree
    float u = 0.0f;
    if (k < batch && uniforms) u = uniforms[row0 + k];
    if (ntop >= 4) {
        for (uint32_t i = threadIdx.x * 4; i < ntop; i += kWG * 4)
            *reinterpret_cast<float4*>(s_top + i) = *reinterpret_cast<const float4*>(sum + i);
    } else if (threadIdx.x < ntop) {
        s_top[threadIdx.x] = sum[threadIdx.x];
    }
    __syncthreads();
    AnyGranule own[kLdsOwn];
    float weight = 0.0f;
    if (k < batch) {
        const float total = s_top[1];
        if (!uniforms) u = rng_uniform(seed, generator_calls(uniforms, calls, a.size, a.err) + blockIdx.y, (uint64_t)k);
        float mass = (u + (float)k) * (total / (float)batch);  // each operation rounded once
        uint32_t node = 1;
        int d = 0;
        // through the staged levels three at a time: the eight descendants of `node` three levels down are 32
        // contiguous, aligned bytes of LDS - one read instead of three dependent ones -, the two levels between
        // are rebuilt with the additions the tree was built with
        for (; d + 3 <= lds_levels; d += 3) {
            const float4 lo = *reinterpret_cast<const float4*>(s_top + ((size_t)node << 3));
            const float4 hi = *reinterpret_cast<const float4*>(s_top + ((size_t)node << 3) + 4);
            float unused;
            node = (node << 3) + walk8(lo, hi, mass, unused);
        }
        for (; d < lds_levels; ++d) {
            const float left = s_top[2 * node];
            if (mass <= left) {
                node = 2 * node;
            } else {
                mass -= left;
                node = 2 * node + 1;
            }
        }
        // Below the staged levels every dependent load brings up to five levels at once: the 32 (16, 8,
        // 4, 2) descendants of `node` five (four, ... one) levels down are 128 (64, ... 8) contiguous,
        // aligned bytes - a whole cache line in the first case; the levels between are rebuilt with
        // the additions the tree was built with. The remaining levels are taken five at a time, and so that the last load brings
        // four at least (the levels it would start from otherwise may be silent, see kSilentLevels): eight are 4 + 4, seven 3 + 4, six 2 + 4.
        float picked = depth <= lds_levels ? s_top[node] : 0.0f;
        while (d < depth) {  // wave-uniform
            const int rest = depth - d;
            const int g = rest <= 5 ? rest : rest <= 8 ? rest - 4 : 5;
            node = descend_group(sum, node, g, mass, picked);
            d += g;
        }
        const int64_t idx = (int64_t)node - ((int64_t)1 << depth);
        const int64_t slot = idx < a.capacity ? idx : a.capacity - 1;
        // the row's scalar fields are requested now, before the weight's arithmetic and the barrier
#pragma unroll
        for (int f = 0; f < kLdsOwn; ++f)
            if (f < t.nfields && t.units[f] == 1)
                own[f].load(as_global(t.store[f]) + (uint64_t)slot * t.stride[f], t.vec_log2[f]);
        a.out_idx[row0 + k] = idx;
        const int64_t size = s_slot[kStrata];  // left there by the helper wave before the first barrier
        weight = powf_det(picked / total * (float)size, -beta);
        sample_flags(a, total, idx, size);
        s_slot[threadIdx.x] = slot;
    }
    __syncthreads();
    const uint32_t rows = (uint32_t)((batch - k0) < kStrata ? (batch - k0) : kStrata);
    if (k < batch) {
        a.out_w[row0 + k] = weight / s_max_w;
#pragma unroll
        for (int f = 0; f < kLdsOwn; ++f)
            if (f < t.nfields && t.units[f] == 1)
                own[f].store(as_global(t.io[f]) + (uint64_t)(row0 + k) * t.row_bytes[f], t.vec_log2[f]);
    }
    // the other granules, coalesced over the workgroup's rows: of large fields field by field,
    for (int f = 0; kLarge && f < t.nfields; ++f) {
        const uint32_t units = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_large[f]);
        if (units == 0) continue;
        const uint32_t bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_bytes[f]), stride = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_stride[f]);
        const gbyte* const store = as_global((const uint8_t*)uniform_pointer(s_store[f]));
        gbyte* const io = as_global(uniform_pointer(s_io[f])) + (uint64_t)(row0 + k0) * bytes;
        const uint32_t work = rows * units;
        const float inverse = 1.0f / (float)units;
        for (uint32_t base = threadIdx.x; base < work; base += kLargeTrip * kWG) {
            granule_t held[kLargeTrip];
            gbyte* to[kLargeTrip];
#pragma unroll
            for (int q = 0; q < kLargeTrip; ++q) {
                const uint32_t w = base + q * kWG < work ? base + q * kWG : base;  // (past the end: the thread's first again)
                uint32_t r = (uint32_t)((float)w * inverse), unit = w - r * units;  // (within one of the quotient: w is below 2^23)
                if ((int)unit < 0) r -= 1, unit += units;
                if (unit >= units) r += 1, unit -= units;
                const uint32_t off = granule_offset(unit, 4, bytes);
                held[q] = __builtin_nontemporal_load((const g16*)(store + (uint64_t)s_slot[r] * stride + off));
                to[q] = io + (r * bytes + off);
            }
#pragma unroll
            for (int q = 0; q < kLargeTrip; ++q) asm volatile("" : "+v"(held[q]));
            auto store_all = [&](auto through) {
#pragma unroll
                for (int q = 0; q < kLargeTrip; ++q)
                    if (base + q * kWG < work) store_granule<decltype(through)::value>((g16*)to[q], held[q]);
            };
            if (large >> 31) store_all(std::true_type{});  // uniform
            else store_all(std::false_type{});
        }
    }
    // of the others field by field and row by row
    const uint32_t work = rows * rest;
    for (uint32_t base = threadIdx.x; base < work; base += kLargeTrip * kWG) {
        gbyte* to[kLargeTrip];
        uint32_t vl[kLargeTrip];
        AnyGranule held[kLargeTrip];
#pragma unroll
        for (int q = 0; q < kLargeTrip; ++q) {
            uint32_t w = base + (uint32_t)q * kWG;
            to[q] = nullptr;
            if (w >= work) continue;
            int f = 0;
            while (w >= rows * s_units[f]) w -= rows * s_units[f++];  // (ends at a field of `rest`: w is below their total)
            const uint32_t units = s_units[f], r = w / units;
            vl[q] = s_vl[f];
            const uint32_t off = granule_offset(w - r * units, vl[q], s_bytes[f]);
            held[q].load(as_global(s_store[f]) + (uint64_t)s_slot[r] * s_stride[f] + off, vl[q]);
            to[q] = as_global(s_io[f]) + (uint64_t)(row0 + k0 + r) * s_bytes[f] + off;
        }
#pragma unroll
        for (int q = 0; q < kLargeTrip; ++q)
            if (to[q]) held[q].store(to[q], vl[q]);
    }
}

}  // namespace mrb
