// The discounted return's tiled kernel and its gradient's (see mrb_discounted_return, mrb_discounted_return_grad; the
// kernel for many columns is k_discounted_return in mrb_kernels.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mrb_device.h"

namespace mrb {

// ---------------------------------------------------------------------------
// Discounted return (mindspore_rl/utils/discounted_return.py:84-92) and its gradient. Both are one recurrence over
// the time axis per (batch, inner) column,
//   last = x[t] + ((1 - done[t']) * gamma) * last, each operation rounded once,
// the return backwards in time (x = reward, t' = t, last starts at the bootstrap value), the gradient forwards
// (kBack; x = the incoming gradient, t' = t - 1, last starts at zero: with c_t = (1 - done_t) * gamma the adjoint of
// G_t = R_t + c_t G_{t+1} is A_t = dG_t + c_{t-1} A_{t-1}, dR_t = A_t, and the bootstrap value's gradient is
// c_{T-1} A_{T-1}). Step s of the return is time T - 1 - s and its flags', of the gradient time s with the flags of time
// s - 1. (The gradient's step 0 has no factor: it multiplies a zero, so any flag will do.)
// ---------------------------------------------------------------------------

// Fewer columns, where a thread per column leaves the memory system idle: a workgroup takes kCols columns and walks
// their steps in chunks of kDrChunk through three LDS buffers, as a pipeline. Wave 0 runs the recurrence out of LDS (lane =
// column) and meets the movers - four waves, or eight - at a barrier in the MIDDLE of every chunk, so that the next chunk's
// first steps are there, and are read, before it comes to them. Between the barriers in chunks c - 1 and c the movers
//   take     chunk c - 2's results out of its LDS buffer,
//   deposit  chunk c + 1, requested kDrAhead stages ago, into that buffer, each mover over what it has itself read there,
//   request  chunk c + 1 + kDrAhead into the registers just emptied (independent, coalesced loads),
//   store    and write chunk c - 2's results to memory.
// (lds_barrier: requests and results stay in flight across it.)
//
// What bounds it: for few columns the recurrence, a chain of two dependent operations per step in ONE wave; for many
// the memory. A chain in registers alone takes 10 cycles a step; an LDS access of that wave costs it 9 to 20 more, wherever it is
// put (between the two operations of a step it costs most), so there are few: a column's steps lie one after the other, one 16-byte
// read brings four steps' values and one more their factors, sixteen steps ahead; and up to sixteen columns to a workgroup it leaves
// only every fourth result (4 bytes, where four results are 16: 16 cycles a step against 21), from which the movers, who have time, work
// out the three before. More columns are bound by the movers and the memory: there it leaves all results (at 32 columns with every
// fourth [2000, 8000] took 32.5 us, with all 30.3). Loads are cached: neighbouring groups on one die share 128-byte lines, and read as
// streams their second halves came from memory again (13.4 -> 12.5 us at [1000, 4096]). us before / now, forward and backward:
//   [1000, 4096] 14.3 14.2 / 11.8 11.8, [1000, 32] 12.4 12.9 / 11.2 11.4, [2000, 3001] 27.6 27.7 / 20.9 21.1, [65, 4825] 5.3 5.4 / 4.4 4.5,
//   [1000, 8192] 17.8 17.5 / 15.8 16.5, [2000, 8000] 28.5 29.1 / 28.4 29.2, [2000, 7501] 40.0 40.5 / 33.4 33.7, [1000, 16384] 30.2 30.8 / 28.7 28.5,
//   [1011, 204, 3] 14.6 14.6 / 12.2 12.0, [1000, 3000, 3] 25.8 26.1 / 19.4 18.9; [4000, 8192], 300 MB that no cache holds, 56.6 55.7 / 52.9 54.5.
// Up to 32 MB of results are stored through the L2 at once. What a non-temporal store leaves of a 128-byte line that two groups share is
// written twice, and a plain one's lines are written when the kernel ends; but more of them push the inputs out of the memory's
// cache. us, non-temporal / plain / through: [135, 52] 4.6 / 4.0 / 4.1, [353, 444] 6.3 / 5.9 / 6.0, [1494, 290] 16.6 / 16.4 / 16.1, [128, 5000] 4.7 / - / 4.3,
// [200, 8000] 6.0 / 6.3 / 5.6, [1000, 4096] 11.9 / 13.1 / 11.6, [2000, 3001] 21.0 / 21.7 / 20.3, [1000, 2500, 3] 15.0 / - / 13.9, [1000, 8192] 15.9 / - / 15.7;
// [4000, 4096] 37.7 / - / 37.4, [2000, 7501] 28.3 / - / 28.5, [3000, 1365, 3] 29.2 / - / 31.8, [2000, 2700, 3] 25.8 / - / 27.1, [8000, 4096] 72.6 / - / 82.6. And with
// sixty-four columns [1000, 16384] 23.4 / 24.1 / 23.5, [1000, 24000] 36.6 / - / 37.9, [1000, 32768] 44.6 / - / 56.4.
// A single group shares no line, and who reads its results next finds them in the L2 they went through only where they may stay: as
// non-temporal ones. us, non-temporal / through, alone and with the maximum over the steps behind it: [20, 1] 3.14 / 3.33, 5.9 / 6.3,
// [64, 8] 3.01 / 3.04, 10.7 / 13.3, [128, 8] 3.51 / 3.56, 15.5 / 22.0, [1000, 16] 11.2 / 11.1, 17.6 / 18.8; of several groups [20, 17] 3.14 / 2.92, 7.3 / 6.8,
// [128, 17] 3.94 / 3.55, 20.3 / 15.4, [128, 128] 3.63 / 3.66, 12.5 / 11.1, [1000, 100] 11.9 / 11.5, 36.1 / 29.5. (2048 columns are where such a
// reader loses, [300, 2048] 20.0 / 26.4 where [300, 1000] gains, 33.8 / 26.0; and of some 4095 columns the gradient does near the line,
// [1950, 4095] 21.3 / 22.3.)
// kCols is small so that a few thousand columns spread over all
// compute units, several workgroups to each when there are more. The pad of four floats puts the sixteen columns'
// 16-byte reads into different banks, and the movers' scalar writes likewise.
//
// Every mover issues the SAME number of loads and stores in every stage but the last, without a branch around any of them: a step
// past the end of the time axis is replaced by the last one (loaded again, not stored), a
// column past the last one by a column before it. Only so can the compiler count what is in flight: with a branch per
// element, or a way out of the loop in the middle of its three stages, it would wait for EVERYTHING before a deposit.
//   kQuad   a mover carries four neighbouring columns of one step, one 16-byte load and store (4-byte aligned when
//           the number of columns is not a multiple of four) and the four flags as one 4-byte load; needs inner == 1
//           and at least four columns. The last quad is moved back so that it ends with the last column.
//   else    a mover carries four steps of one column.
constexpr int kDrChunk = 64;  // steps
constexpr int kDrAhead = 3;   // chunks on their way from memory at any time
constexpr int kDrBuffers = 3;
constexpr int kDrPitch = kDrChunk + 4;
constexpr int64_t kDrThrough = 8 << 20;
inline bool returns_through(int64_t timesteps, int64_t cols, int group) { return group < 64 && cols > group && timesteps * cols <= kDrThrough; }

typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));      // four floats at any float's address
typedef uint32_t u32_u __attribute__((aligned(1)));                         // four flags at any address
#define MRB_GLOBAL __attribute__((address_space(1)))

// kThrough: the results are stored through the L2 (a kernel of its own: with both in one, a call of few columns took 1 to 3 % longer).
template <bool kBack, bool kQuad, int kCols, int kMovers, bool kThrough>
__global__ __launch_bounds__(64 + kMovers) void k_discounted_return_tiled(
    const float* __restrict__ x, const uint8_t* __restrict__ done, float* __restrict__ end_value, float* __restrict__ out,
    int64_t timesteps, int64_t batch, int64_t inner, float gamma) {
    constexpr int kPer = kDrChunk * kCols / 4 / kMovers;  // groups of four elements of a chunk that a mover carries
    constexpr int kSteps = kDrChunk / kPer;                 // steps the movers cover at once
    constexpr bool kAll = kCols > 16;                       // the recurrence leaves every result, else every fourth
    constexpr int kSpan = 256 / kCols;                      // consecutive steps that a wave of movers carries
    static_assert(kAll || kDrChunk / kSpan <= 2 * (kDrPitch - kDrChunk), "a pad for each");

    static_assert(kPer >= 1 && kSteps * kPer == kDrChunk && kSteps % 4 == 0, "the movers share a chunk evenly");
    __shared__ float s_x[kDrBuffers][kCols][kDrPitch];  // a step's value in, its result out
    __shared__ float s_f[kDrBuffers][kCols][kDrPitch];  // its factor (1 - done) * gamma
    const int64_t cols = batch * inner;
    // Workgroups are dealt to the chip's eight dies in turn, and each die has its own L2. Neighbouring column groups
    // share cache lines (a group's flags of a step are kCols bytes), so they go to the SAME die.
    const uint32_t groups = (uint32_t)((cols + kCols - 1) / kCols), per = groups >> 3, more = groups & 7u, die = blockIdx.x & 7u;
    const uint32_t group = die * per + (die < more ? die : more) + (blockIdx.x >> 3);
    // every group is full when there are kCols columns at all: the last one is moved back
    const int64_t c_last = cols > kCols ? cols - kCols : 0;
    const int64_t c0 = (int64_t)group * kCols < c_last ? (int64_t)group * kCols : c_last;
    const int ncols = (int)(cols - c0 < kCols ? cols - c0 : kCols);
    const int lane = threadIdx.x & 63;
    const int64_t nchunks = (timesteps + kDrChunk - 1) / kDrChunk;
    const float scaled_live = (1.0f - 0.0f) * gamma, scaled_done = (1.0f - 1.0f) * gamma;
    // the column (of this group) that LDS column q holds
    auto column_of = [&](int q) -> int {
        if (kQuad) {
            const int quad = 4 * (q >> 2);
            return (quad < ncols - 4 ? quad : ncols - 4) + (q & 3);
        }
        return q < ncols ? q : ncols - 1;
    };

    // The result in front of the first step that a wave of movers carries, kept in the pads: the step before belongs to another wave,
    // which may have put the next chunk there.
    auto in_front = [&](int buf, int q, int at) -> float& {
        const int nth = at / kSpan;
        return nth < 4 ? s_x[buf][q][kDrChunk + nth] : s_f[buf][q][kDrChunk + nth - 4];
    };

    if (threadIdx.x < 64) {
        // ---- wave 0: the recurrence
        const int q = lane < kCols ? lane : 0;
        const int64_t col = c0 + column_of(q);
        float last = kBack ? 0.0f : end_value[col];
        f32x4 xa[4], fa[4], xb[4], fb[4];
        auto fetch = [&](int buf, int at, f32x4 (&xs)[4], f32x4 (&fs)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xs[i] = *reinterpret_cast<const f32x4*>(&s_x[buf][q][at + 4 * i]);
                fs[i] = *reinterpret_cast<const f32x4*>(&s_f[buf][q][at + 4 * i]);
            }
        };
        auto sixteen = [&](int buf, int at, f32x4 (&xs)[4], const f32x4 (&fs)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    last = xs[i][j] + fs[i][j] * last;
                    if (kAll) xs[i][j] = last;
                }
                if (kAll)
                    *reinterpret_cast<f32x4*>(&s_x[buf][q][at + 4 * i]) = xs[i];
                else
                    s_x[buf][q][at + 4 * i + 3] = last;
                if (!kAll && (at + 4 * i + 4) % kSpan == 0 && at + 4 * i + 4 < kDrChunk) in_front(buf, q, at + 4 * i + 4) = last;
            }
        };
        lds_barrier();
        if (lane < kCols) fetch(0, 0, xa, fa);
        int buf = 0;
        for (int64_t c = 0; c < nchunks; ++c) {
            const int next = buf == kDrBuffers - 1 ? 0 : buf + 1;
            if (lane < kCols) {
                if (!kAll) in_front(buf, q, 0) = last;
                fetch(buf, 16, xb, fb);
                sixteen(buf, 0, xa, fa);
                fetch(buf, 32, xa, fa);
                sixteen(buf, 16, xb, fb);
            }
            lds_barrier();
            // (a short last chunk runs doubled steps to the end of its half: nobody looks at what they leave)
            if (lane < kCols && timesteps - c * kDrChunk > kDrChunk / 2) {
                fetch(buf, 48, xb, fb);
                sixteen(buf, 32, xa, fa);
                fetch(next, 0, xa, fa);  // (behind the last chunk: what nobody uses)
                sixteen(buf, 48, xb, fb);
            }
            buf = next;
        }
        if (nchunks == 1) lds_barrier();
        lds_barrier();
        return;
    }
    // ---- the movers
    const int m = (int)threadIdx.x - 64;
    // kQuad: columns 4 * quad .. of step `step`; else: column `own` of steps `step` .. + 3; and kSteps steps on
    const int quad = m % (kCols / 4), own = m % kCols;
    const int step = kQuad ? m / (kCols / 4) : 4 * (m / kCols);
    const int64_t col = c0 + (kQuad ? column_of(4 * quad) : column_of(own));
    const int64_t mb = kQuad ? col : col / inner;
    constexpr int kFlags = kQuad ? 1 : 4;
    f32x4 xs[kDrAhead][kPer];
    uint32_t ds[kDrAhead][kPer][kFlags];
    // Addresses: a wave-uniform base per chunk - the row of its earliest time - plus a 32-bit offset (a chunk spans
    // 64 rows, and the host takes this kernel for at most a few ten thousand columns). Step k of chunk c is at row k of the chunk when time runs with the
    // steps and at row `last` - k when it runs against them, `last` being the chunk's last existing step.
    const uint32_t row_x = (uint32_t)cols * 4u, row_f = (uint32_t)batch, off_x = (uint32_t)col * 4u, off_f = (uint32_t)mb;
    auto last_of = [&](int64_t c) -> int {  // chunk c's last step that exists; past the end: its first, doubled throughout
        const int64_t left = timesteps - 1 - c * kDrChunk;
        return left >= kDrChunk - 1 ? kDrChunk - 1 : left >= 0 ? (int)left : 0;
    };
    auto first_of = [&](int64_t c) -> int64_t {  // chunk c's first step (past the end: the last step)
        return c * kDrChunk < timesteps ? c * kDrChunk : timesteps - 1;
    };
    auto row_of = [&](int k, int last) -> uint32_t {
        const int kk = k < last ? k : last;
        return (uint32_t)(kBack ? kk : last - kk);
    };
    auto base_of = [&](int64_t c) -> int64_t {  // the earliest time of chunk c
        return kBack ? first_of(c) : timesteps - 1 - first_of(c) - last_of(c);
    };
    // (Read through addresses that the compiler knows nothing of: what it knows to be constant it would request behind the barriers
    // in front of its use, a trip to memory later.)
    const MRB_GLOBAL char* from_x = (const MRB_GLOBAL char*)x;
    const MRB_GLOBAL char* from_f = (const MRB_GLOBAL char*)done;
    asm volatile("" : "+s"(from_x), "+s"(from_f));
    auto request = [&](int64_t c, f32x4 (&xr)[kPer], uint32_t (&dr)[kPer][kFlags]) {
        const int last = last_of(c);
        const int64_t t0 = base_of(c);
        const MRB_GLOBAL char* const bx = from_x + t0 * cols * 4;
        const MRB_GLOBAL char* const bf = from_f + (kBack && t0 > 0 ? t0 - 1 : t0) * batch;
        const uint32_t back = kBack && t0 == 0 ? 1u : 0u;  // the first chunk's flags start a row late: step 0 takes any
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (kQuad) {
                const uint32_t row = row_of(i * kSteps + step, last);
                xr[i] = *(const MRB_GLOBAL f32x4_u*)(bx + (row * row_x + off_x));
                dr[i][0] = *(const MRB_GLOBAL u32_u*)(bf + ((row > back ? row - back : 0u) * row_f + off_f));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t row = row_of(i * kSteps + step + j, last);
                    xr[i][j] = *(const MRB_GLOBAL float*)(bx + (row * row_x + off_x));
                    dr[i][kQuad ? 0 : j] = (uint8_t)bf[(row > back ? row - back : 0u) * row_f + off_f];
                }
            }
        }
    };
    auto deposit = [&](int buf, const f32x4 (&xr)[kPer], const uint32_t (&dr)[kPer][kFlags]) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = i * kSteps + step;
            if (kQuad) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s_x[buf][4 * quad + j][k] = xr[i][j];
                    s_f[buf][4 * quad + j][k] = (dr[i][0] >> (8 * j)) & 255u ? scaled_done : scaled_live;
                }
            } else {
                f32x4 f;
#pragma unroll
                for (int j = 0; j < 4; ++j) f[j] = dr[i][kQuad ? 0 : j] ? scaled_done : scaled_live;
                *reinterpret_cast<f32x4*>(&s_x[buf][own][k]) = xr[i];
                *reinterpret_cast<f32x4*>(&s_f[buf][own][k]) = f;
            }
        }
    };
    // A chunk's results, from LDS to registers: of each four steps the recurrence has left the last one's. A mover works the three
    // before it out again, from the result in front of them, for four steps of one column; one that carries a step of four
    // columns hands them to the others that carry these four steps, all in its own wave, through LDS.
    auto take = [&](int buf, f32x4 (&v)[kPer]) {
        if (kAll) {
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                if (!kQuad) v[i] = *reinterpret_cast<const f32x4*>(&s_x[buf][own][i * kSteps + step]);
#pragma unroll
                for (int j = 0; kQuad && j < 4; ++j) v[i][j] = s_x[buf][4 * quad + j][i * kSteps + step];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int of = kQuad ? 4 * quad + (step & 3) : own, at = i * kSteps + (step & ~3);
            const f32x4 f = *reinterpret_cast<const f32x4*>(&s_f[buf][of][at]);
            float last = at % kSpan ? s_x[buf][of][at ? at - 1 : 0] : in_front(buf, of, at);
            v[i] = *reinterpret_cast<const f32x4*>(&s_x[buf][of][at]);
#pragma unroll
            for (int j = 0; j < 3; ++j) v[i][j] = last = v[i][j] + f[j] * last;
            if (kQuad) *reinterpret_cast<f32x4*>(&s_x[buf][of][at]) = v[i];
        }
        if (kQuad) {
            wave_lds_fence();
#pragma unroll
            for (int i = 0; i < kPer; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[i][j] = s_x[buf][4 * quad + j][i * kSteps + step];
        }
        wave_lds_fence();  // (the next chunk goes over what other lanes have read)
    };
    auto store = [&](int64_t c, const f32x4 (&v)[kPer], auto whole, int last) {
        char* const bo = reinterpret_cast<char*>(out + base_of(c) * cols);
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = i * kSteps + step;
            if (kQuad) {
                if (decltype(whole)::value || k <= last) {
                    char* const to = bo + (row_of(k, last) * row_x + off_x);
                    if (kThrough) store_through(to, v[i]);
                    else __builtin_nontemporal_store(v[i], reinterpret_cast<f32x4_u*>(to));
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (decltype(whole)::value || k + j <= last) {
                        char* const to = bo + (row_of(k + j, last) * row_x + off_x);
                        if (kThrough) store_through(to, (float)v[i][j]);
                        else __builtin_nontemporal_store(v[i][j], reinterpret_cast<float*>(to));
                    }
            }
        }
    };
    const int end = last_of(nchunks - 1);  // the last chunk's last step
#pragma unroll
    for (int j = 0; j < kDrAhead; ++j) request(j, xs[j], ds[j]);
    uint32_t end_flags[kFlags];  // the last step's, for the bootstrap value's gradient
    if (kBack) {
        if (kQuad)
            end_flags[0] = *reinterpret_cast<const u32_u*>(done + (timesteps - 1) * batch + off_f);
        else
            end_flags[0] = done[(timesteps - 1) * batch + off_f];
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them now: none behind the wait for the first
    // Chunk k lies in buffer k % 3 and comes through register set k % kDrAhead. Between the recurrence's barriers in the middle
    // of chunks c - 1 and c: take chunk c - 2's results out of its buffer and put chunk c + 1 (past the end: a chunk nobody
    // reads) there, each mover its own places.
    static_assert(kDrAhead == 3 && kDrBuffers == 3, "the sets and buffers below");
    f32x4 v[kPer];
    deposit(0, xs[0], ds[0]);
    request(kDrAhead, xs[0], ds[0]);
    lds_barrier();
    deposit(1, xs[1], ds[1]);
    request(kDrAhead + 1, xs[1], ds[1]);
    lds_barrier();
    deposit(2, xs[2], ds[2]);
    request(kDrAhead + 2, xs[2], ds[2]);
    lds_barrier();
    auto stage = [&](int64_t c, auto nth) {
        constexpr int j = decltype(nth)::value;
        take(j, v);
        deposit(j, xs[j], ds[j]);
        request(c + 1 + kDrAhead, xs[j], ds[j]);
        store(c - 2, v, std::true_type{}, kDrChunk - 1);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);  // (the next chunk's flags are not looked at, that is waited for, before its time)
    };
    int64_t c = 2;
    for (; c + 2 < nchunks; c += 3) {  // (no way out in the middle: what is in flight is counted exactly)
        stage(c, std::integral_constant<int, 0>{});
        stage(c + 1, std::integral_constant<int, 1>{});
        stage(c + 2, std::integral_constant<int, 2>{});
    }
    int buf = 0;
    if (c < nchunks) stage(c, std::integral_constant<int, 0>{}), buf = 1;
    if (c + 1 < nchunks) stage(c + 1, std::integral_constant<int, 1>{}), buf = 2;
    if (nchunks > 1) {
        take(buf, v);
        store(nchunks - 2, v, std::true_type{}, kDrChunk - 1);
        buf = buf == kDrBuffers - 1 ? 0 : buf + 1;
    }
    lds_barrier();
    take(buf, v);
    store(nchunks - 1, v, std::false_type{}, end);
    if (kBack && end_value) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = i * kSteps + step;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool flag = kQuad ? (end_flags[0] >> (8 * j)) & 255u : end_flags[0] != 0;
                if (k + (kQuad ? 0 : j) == end) end_value[col + (kQuad ? j : 0)] = (1.0f - (flag ? 1.0f : 0.0f)) * gamma * v[i][j];
            }
        }
    }
}

// Launches k_discounted_return_tiled with the workgroup shape that fits the number of columns (defined in
// mrb_returns.hip). `end_value`: the bootstrap value in, or (back) the bootstrap value's gradient out (may be NULL).
hipError_t launch_discounted_return_tiled(bool back, const float* x, const uint8_t* done, float* end_value, float* out,
                                          int64_t timesteps, int64_t batch, int64_t inner, float gamma, hipStream_t s);

}  // namespace mrb
