// The meeting of a launch's workgroups (mrb_meet.h) on the CPU: a launch is a wave per workgroup that changes its root. Prints what
// went wrong, and returns how much did.
#include "../../mindrl_amd/csrc/mrb_meet.h"

#include <stdio.h>
#include <stdlib.h>

#include <set>

using namespace mrb;

struct Buffer {
    struct { uint32_t err[16]; float maxp[16]; Meet meet; } words;
    float roots_s[256], roots_m[256];
    Buffer() { memset((void*)this, 0, sizeof(*this)); }
    float* maxp() { return words.maxp; }
};

int wrong = 0;
#define CHECK(x, ...) do { if (!(x)) { ++wrong; printf("%s:%d: %s: ", __FILE__, __LINE__, #x); printf(__VA_ARGS__); printf("\n"); } } while (0)

// A launch in which `runs` change their roots, all of them counted but `missing` (its workgroup never comes). Returns the
// workgroups that took the roots.
int launch(Buffer& b, const std::set<uint32_t>& runs, int salt, int missing = -1, uint64_t most = 3000000) {
    std::vector<sim::Wave> waves;
    float new_s[256], new_m[256];
    memcpy(new_s, b.roots_s, sizeof(new_s));
    memcpy(new_m, b.roots_m, sizeof(new_m));
    int takers = 0;
    auto value = [&](uint32_t r) { return (float)(r * 1000 + salt); };
    float got_s[256], got_m[256];
    for (const uint32_t r : runs)
        if ((int)r != missing) {
            sim::Wave w;
            w.body = [&, r](uint32_t lane) {
                const uint32_t turn = meet_turn(b.maxp());
                uint32_t changed = 0;
                for (uint32_t c = 0; c < 4; ++c) changed |= (uint32_t)runs.count(4 * lane + c) << c;
                float4 vs = make_float4(b.roots_s[4 * lane], b.roots_s[4 * lane + 1], b.roots_s[4 * lane + 2], b.roots_s[4 * lane + 3]);
                float4 vm = make_float4(b.roots_m[4 * lane], b.roots_m[4 * lane + 1], b.roots_m[4 * lane + 2], b.roots_m[4 * lane + 3]);
                const MeetPlan plan = meet_plan(changed, r, lane);
                if (!meet(b.maxp(), b.words.err, turn, r, value(r), -value(r), lane, plan, vs, vm)) return;
                takers += lane == 0;
                const float s[4] = {vs.x, vs.y, vs.z, vs.w}, t[4] = {vm.x, vm.y, vm.z, vm.w};
                for (int c = 0; c < 4; ++c) got_s[4 * lane + c] = s[c], got_m[4 * lane + c] = t[c];
            };
            waves.push_back(std::move(w));
        }
    if (!sim::run(waves, most)) {
        ++wrong;
        printf("%zu runs: not ended after %llu turns\n", runs.size(), (unsigned long long)most);
        exit(1);
    }
    for (const uint32_t r : runs)
        if ((int)r != missing) new_s[r] = value(r), new_m[r] = -value(r);
    CHECK(takers > 0, "%zu runs: nobody took the roots", runs.size());
    if (takers) CHECK(!memcmp(got_s, new_s, sizeof(new_s)) && !memcmp(got_m, new_m, sizeof(new_m)), "%zu runs: other roots", runs.size());
    memcpy(b.roots_s, new_s, sizeof(new_s));
    memcpy(b.roots_m, new_m, sizeof(new_m));
    return takers;
}

std::set<uint32_t> some(uint32_t n) {
    std::set<uint32_t> r;
    while (r.size() < n) r.insert((uint32_t)sim::g_rng() % 256);
    return r;
}

bool at_rest(const Meet& m) {
    bool zero = m.arrived == 0;
    for (auto& g : m.group) zero = zero && g[0] == 0;
    return zero;
}

void launches() {
    Buffer b;
    uint32_t k = 0;
    for (const uint32_t n : {1, 2, 3, 16, 95, 96, 97, 98, 150, 255, 256, 1, 256, 97, 40}) {
        CHECK(launch(b, some(n), (int)n) == 1, "%u runs", n);
        CHECK(at_rest(b.words.meet) && b.words.meet.turn == ++k && b.words.err[0] == 0, "%u runs", n);
    }
}

// Whatever the counters hold, the launch has a workgroup that takes all the roots; ordinary launches follow.
void any_count() {
    for (const uint32_t n : {2, 96, 97, 256})
        for (const uint32_t count : {1u, n - 1, n, 100000u})
            for (int where = 0; where < 2; ++where) {
                Buffer b;
                launch(b, some(n), 1);
                if (where == 0) b.words.meet.arrived = count;
                else for (auto& g : b.words.meet.group) g[0] = count;
                for (int k = 2; k < 4; ++k) launch(b, some(n), k);
                CHECK(b.words.err[0] == 0, "%u runs, %u counted", n, count);
            }
}

// A root that never comes: the wait ends, the root stays as it was, the buffer is flagged and the next launch is an ordinary one.
void missing_root() {
    for (const uint32_t n : {2, 100}) {
        Buffer b;
        launch(b, some(256), 1);
        const auto runs = some(n);
        const uint32_t gone = *runs.begin();
        b.words.meet.arrived = 1;
        if (n > kMeetDirect) b.words.meet.group[gone / kMeetGroup][0] = 1, b.words.meet.arrived = 0;
        CHECK(launch(b, runs, 2, (int)gone, 100000000) > 0, "%u runs", n);
        CHECK(b.words.err[0] == MRB_DERR_OVERLAP, "%u runs: flags %u", n, b.words.err[0]);
        b.words.err[0] = 0;
        launch(b, some(n), 3);
        CHECK(b.words.err[0] == 0, "%u runs", n);
    }
}

// Launches around the last of the 2^32 numbers, on words that the lap before left: none holds a later launch's number.
void last_number() {
    for (int lap = 0; lap < 40; ++lap) {
        Buffer b;
        b.words.meet.turn = 0xfffffffdu;
        if (lap % 2)
            for (uint32_t r = 0; r < 256; ++r) b.words.meet.root[r][0] = b.words.meet.root[r][1] = b.words.meet.largest[r] = (uint64_t)(1 + r % 4) << 32;
        for (int k = 1; k < 8; ++k) CHECK(launch(b, some(k < 6 ? 2 + (uint32_t)lap : 120), k) == 1, "launch %d", k);
        CHECK(at_rest(b.words.meet) && b.words.err[0] == 0, "lap %d", lap);
    }
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "launches") launches();
    else if (what == "any_count") any_count();
    else if (what == "missing_root") missing_root();
    else if (what == "last_number") last_number();
    else return 2;
    printf("%d wrong\n", wrong);
    return wrong != 0;
}
