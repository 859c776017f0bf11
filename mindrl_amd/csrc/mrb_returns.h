// The discounted return's tiled kernel and its gradient's (see mrb_discounted_return, mrb_discounted_return_grad; the
// kernel for many columns is k_discounted_return in mrb_kernels.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

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
// their steps in chunks of kDrChunk through three LDS buffers, as a pipeline whose stages run at the same time on
// consecutive chunks:
//   deposit  the movers (four waves, or eight) put chunk s, requested kDrAhead stages ago, into its LDS buffer ...
//   request  ... request chunk s + kDrAhead into the registers just emptied (independent, coalesced loads) ...
//   drain    ... and write chunk s - 2's results from LDS to memory, while ...
//   recur    ... wave 0 runs the recurrence over chunk s - 1 out of LDS (lane = column).
// One LDS barrier per stage (lds_barrier: requests and results stay in flight across it).
//
// What bounds it: for few columns the recurrence, a chain of two dependent operations per step in ONE wave; for many
// the memory. The chain is kept as short as it can be: a column's steps lie one after the other in LDS, so that one
// 16-byte read brings four steps' values (one more their factors, one 16-byte write takes the results), and a batch
// of steps is read while the one before runs (read 15 at a time just before their use, and two LDS accesses a step,
// a step took 54 cycles: [1000, 4096] 22.9 us, now 14.5; [1000, 32] 24 us, now 11.9, of which the chain alone, with the
// movers idle, takes 11.2). kCols is small so that a few thousand columns spread over all
// compute units, several workgroups to each when there are more. The pad of four floats puts the sixteen columns'
// 16-byte reads into different banks, and the movers' scalar writes likewise.
//
// Every mover issues the SAME number of loads and stores in every stage, without a branch around any of them: a step
// past the end of the time axis is replaced by the last one (loaded again, stored again with the same value), a
// column past the last one by a column before it. Only so can the compiler count what is in flight: with a branch per
// element it would wait for EVERYTHING before each deposit.
//   kQuad   a mover carries four neighbouring columns of one step, one 16-byte load and store (4-byte aligned when
//           the number of columns is not a multiple of four) and the four flags as one 4-byte load; needs inner == 1
//           and at least four columns. The last quad is moved back so that it ends with the last column.
//   else    a mover carries four steps of one column.
constexpr int kDrChunk = 64;  // steps
constexpr int kDrAhead = 4;   // chunks on their way from memory at any time
constexpr int kDrPitch = kDrChunk + 4;

typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));      // four floats at any float's address
typedef uint32_t u32_u __attribute__((aligned(1)));                         // four flags at any address

template <bool kBack, bool kQuad, int kCols, int kMovers>
__global__ __launch_bounds__(64 + kMovers) void k_discounted_return_tiled(
    const float* __restrict__ x, const uint8_t* __restrict__ done, float* __restrict__ end_value, float* __restrict__ out,
    int64_t timesteps, int64_t batch, int64_t inner, float gamma) {
    constexpr int kPer = kDrChunk * kCols / 4 / kMovers;  // groups of four elements of a chunk that a mover carries
    constexpr int kSteps = kDrChunk / kPer;                 // steps the movers cover at once
    static_assert(kPer >= 1 && kSteps * kPer == kDrChunk && kSteps % 4 == 0, "the movers share a chunk evenly");
    __shared__ float s_x[3][kCols][kDrPitch];  // a step's value in, its result out
    __shared__ float s_f[3][kCols][kDrPitch];  // its factor (1 - done) * gamma
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

    if (threadIdx.x < 64) {
        // ---- wave 0: the recurrence
        const int q = lane < kCols ? lane : 0;
        const int64_t col = c0 + column_of(q);
        float last = kBack ? 0.0f : end_value[col];
        lds_barrier();
        int buf = 0;
        for (int64_t c = 0; c < nchunks; ++c) {
            if (lane < kCols) {
                float* const vx = s_x[buf][q];
                const float* const vf = s_f[buf][q];
                // sixteen steps at a time, the next sixteen requested before these run (a short last chunk runs its
                // doubled steps too: nobody looks at what they leave)
                f32x4 xa[4], fa[4], xb[4], fb[4];
                auto fetch = [&](int at, f32x4 (&xs)[4], f32x4 (&fs)[4]) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        xs[i] = *reinterpret_cast<const f32x4*>(vx + at + 4 * i);
                        fs[i] = *reinterpret_cast<const f32x4*>(vf + at + 4 * i);
                    }
                };
                auto steps16 = [&](int at, f32x4 (&xs)[4], f32x4 (&fs)[4]) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            last = xs[i][j] + fs[i][j] * last;
                            xs[i][j] = last;
                        }
                        *reinterpret_cast<f32x4*>(vx + at + 4 * i) = xs[i];
                    }
                };
                fetch(0, xa, fa);
#pragma unroll
                for (int at = 0; at < kDrChunk; at += 32) {
                    fetch(at + 16, xb, fb);
                    steps16(at, xa, fa);
                    if (at + 32 < kDrChunk) fetch(at + 32, xa, fa);
                    steps16(at + 16, xb, fb);
                }
                if (kBack && c == nchunks - 1) last = vx[timesteps - 1 - c * kDrChunk];  // step T - 1, not a doubled one
            }
            buf = buf == 2 ? 0 : buf + 1;
            lds_barrier();
        }
        lds_barrier();
        if (kBack && end_value && lane < kCols)
            end_value[col] = (1.0f - (done[(timesteps - 1) * batch + col / inner] ? 1.0f : 0.0f)) * gamma * last;
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
    auto request = [&](int64_t c, f32x4 (&xr)[kPer], uint32_t (&dr)[kPer][kFlags]) {
        const int last = last_of(c);
        const int64_t t0 = base_of(c);
        const char* const bx = reinterpret_cast<const char*>(x + t0 * cols);
        const uint8_t* const bf = done + (kBack && t0 > 0 ? t0 - 1 : t0) * batch;
        const uint32_t back = kBack && t0 == 0 ? 1u : 0u;  // the first chunk's flags start a row late: step 0 takes any
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (kQuad) {
                const uint32_t row = row_of(i * kSteps + step, last);
                xr[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_u*>(bx + (row * row_x + off_x)));
                dr[i][0] = *reinterpret_cast<const u32_u*>(bf + ((row > back ? row - back : 0u) * row_f + off_f));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t row = row_of(i * kSteps + step + j, last);
                    xr[i][j] = __builtin_nontemporal_load(reinterpret_cast<const float*>(bx + (row * row_x + off_x)));
                    dr[i][kQuad ? 0 : j] = bf[(row > back ? row - back : 0u) * row_f + off_f];
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
    auto drain = [&](int64_t c, int buf) {
        const int last = last_of(c);
        char* const bo = reinterpret_cast<char*>(out + base_of(c) * cols);
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (kQuad) {
                const int k = i * kSteps + step < last ? i * kSteps + step : last;
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = s_x[buf][4 * quad + j][k];
                __builtin_nontemporal_store(v, reinterpret_cast<f32x4_u*>(bo + (row_of(k, last) * row_x + off_x)));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = i * kSteps + step + j < last ? i * kSteps + step + j : last;
                    __builtin_nontemporal_store(s_x[buf][own][k], reinterpret_cast<float*>(bo + (row_of(k, last) * row_x + off_x)));
                }
            }
        }
    };
#pragma unroll
    for (int j = 0; j < kDrAhead; ++j) request(j, xs[j], ds[j]);
    static_assert(kDrAhead >= 3, "the two stages without a drain use the first two register sets");
    deposit(0, xs[0], ds[0]);
    request(kDrAhead, xs[0], ds[0]);
    lds_barrier();
    deposit(1, xs[1], ds[1]);
    request(kDrAhead + 1, xs[1], ds[1]);
    lds_barrier();
    // stage s, s = 2 .. nchunks + 1: deposit chunk s (past the end: a chunk nobody reads, into a buffer nobody uses),
    // drain chunk s - 2. Buffers: chunk c lies in buffer c % 3.
    int put = 2, take = 0;
    for (int64_t s = 2; s < nchunks + 2; s += kDrAhead) {
#pragma unroll
        for (int j = 0; j < kDrAhead; ++j) {
            if (s + j >= nchunks + 2) break;  // (uniform; nothing is requested or stored after the loop)
            const int set = (2 + j) % kDrAhead;  // = (s + j) % kDrAhead, known when the loop is unrolled
            deposit(put, xs[set], ds[set]);
            request(s + j + kDrAhead, xs[set], ds[set]);
            drain(s + j - 2, take);
            put = put == 2 ? 0 : put + 1;
            take = take == 2 ? 0 : take + 1;
            lds_barrier();
        }
    }
}

// Launches k_discounted_return_tiled with the workgroup shape that fits the number of columns (defined in
// mrb_returns.hip). `end_value`: the bootstrap value in, or (back) the bootstrap value's gradient out (may be NULL).
hipError_t launch_discounted_return_tiled(bool back, const float* x, const uint8_t* done, float* end_value, float* out,
                                          int64_t timesteps, int64_t batch, int64_t inner, float gamma, hipStream_t s);

}  // namespace mrb
