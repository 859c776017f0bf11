// The tiled kernel of the discounted return and its gradient (mrb_returns.h) on the CPU, against the recurrence. Prints what went
// wrong, and returns how much did.
#include "mrb_returns.h"

using namespace mrb;

int wrong = 0;

template <bool kBack, bool kQuad, int kCols, int kMovers, bool kThrough>
void check(int64_t timesteps, int64_t batch, int64_t inner) {
    const int64_t cols = batch * inner;
    const float gamma = 0.97f;
    std::vector<float> x(timesteps * cols), end(cols), out(timesteps * cols, -1.0f), want(timesteps * cols), want_end(cols);
    std::vector<uint8_t> done(timesteps * batch + 4);  // (flags are read four at a time)
    for (auto& v : x) v = (float)(sim::g_rng() % 2001) / 1000.0f - 1.0f;
    for (auto& v : end) v = (float)(sim::g_rng() % 2001) / 1000.0f - 1.0f;
    for (auto& v : done) v = sim::g_rng() % 16 == 0;
    for (int64_t c = 0; c < cols; ++c) {
        float last = kBack ? 0.0f : end[c];
        for (int64_t s = 0; s < timesteps; ++s) {
            const int64_t t = kBack ? s : timesteps - 1 - s, f = kBack ? s - 1 : t;
            const float factor = (1.0f - (f >= 0 && done[f * batch + c / inner] ? 1.0f : 0.0f)) * gamma;
            last = x[t * cols + c] + factor * last;
            want[t * cols + c] = last;
        }
        want_end[c] = (1.0f - (done[(timesteps - 1) * batch + c / inner] ? 1.0f : 0.0f)) * gamma * last;
    }
    g_through = 0;
    for (uint32_t g = 0; g < (uint32_t)((cols + kCols - 1) / kCols); ++g) {
        const bool ended = sim::run(g, 64 + kMovers, [&] {
            k_discounted_return_tiled<kBack, kQuad, kCols, kMovers, kThrough>(x.data(), done.data(), end.data(), out.data(), timesteps, batch, inner, gamma);
        });
        if (!ended) ++wrong, printf("lanes wait at different places\n");
    }
    int64_t differ = 0;
    for (int64_t i = 0; i < timesteps * cols; ++i) differ += memcmp(&out[i], &want[i], 4) != 0;
    for (int64_t c = 0; kBack && c < cols; ++c) differ += memcmp(&end[c], &want_end[c], 4) != 0;
    // (the last group's columns are moved back, so some results are stored twice)
    if (kThrough ? g_through < timesteps * cols : g_through != 0) ++wrong, printf("%lld columns by %d: %lld stored through\n", (long long)cols, kCols, (long long)g_through);
    if (differ) ++wrong, printf("back %d quad %d columns %d: %lld x %lld x %lld: %lld differ\n", kBack, kQuad, kCols, (long long)timesteps, (long long)batch, (long long)inner, (long long)differ);
}

template <bool kQuad, int kCols, int kMovers>
void both(int64_t batch, int64_t inner) {
    for (const int64_t timesteps : {1, 16, 33, 64, 65, 128, 150, 193, 256, 321}) {
        check<false, kQuad, kCols, kMovers, false>(timesteps, batch, inner);
        check<true, kQuad, kCols, kMovers, false>(timesteps, batch, inner);
        if (kCols == 64) continue;
        check<false, kQuad, kCols, kMovers, kCols != 64>(timesteps, batch, inner);
        check<true, kQuad, kCols, kMovers, kCols != 64>(timesteps, batch, inner);
    }
}

// Which calls store their results through the L2.
void rule(bool want, int64_t timesteps, int64_t cols, int group) {
    if (returns_through(timesteps, cols, group) != want) ++wrong, printf("%lld x %lld by %d: %d\n", (long long)timesteps, (long long)cols, group, !want);
}

int main(int argc, char** argv) {
    for (const int group : {16, 32}) {
        for (const int64_t timesteps : {1, 20, 2000, 1000000}) rule(false, timesteps, 1, group), rule(false, timesteps, group, group);
        rule(true, 1, group + 1, group), rule(true, 2000, group + 1, group);
        rule(true, kDrThrough / 1024, 1024, group), rule(false, kDrThrough / 1024, 1025, group);
    }
    rule(false, 1, 65, 64), rule(false, 100, 16384, 64);
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "quads") both<true, 16, 256>(23, 1), both<true, 16, 256>(5, 1);
    else if (what == "columns") both<false, 16, 256>(7, 3), both<false, 16, 256>(3, 1);
    else if (what == "wide") both<true, 32, 256>(37, 1), both<false, 32, 512>(13, 3), both<false, 64, 512>(70, 1);
    else return 2;
    printf("%d wrong\n", wrong);
    return wrong != 0;
}
