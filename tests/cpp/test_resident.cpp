// The memory the workgroups of a resident solve share (csrc/rt_resident.h),
// run on the host: the workgroups are coroutines that give way before every
// access, and a seeded scheduler takes them in random order, one far behind
// the others as well.  Prints OK.
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <memory>
#include <random>
#include <vector>

#include "rt_resident.h"

using namespace rt;

#define CHECK(c, ...)                                          \
    do {                                                       \
        if (!(c)) {                                            \
            std::printf("FAILED %s: ", #c);                    \
            std::printf(__VA_ARGS__);                          \
            std::printf("\n");                                 \
            std::exit(1);                                      \
        }                                                      \
    } while (0)

struct Sched {
    struct Co {
        ucontext_t ctx;
        std::vector<char> stack = std::vector<char>(64 << 10);
        std::function<void()> fn;
        bool done = false;
    };
    std::vector<std::unique_ptr<Co>> cos;
    ucontext_t main;
    int cur = -1;
    std::mt19937_64 rng;
    static Sched* self;
    static void entry() {
        Co& c = *self->cos[self->cur];
        c.fn();
        c.done = true;
        swapcontext(&c.ctx, &self->main);
    }
    void spawn(std::function<void()> fn) {
        cos.emplace_back(new Co);
        Co& c = *cos.back();
        c.fn = std::move(fn);
        getcontext(&c.ctx);
        c.ctx.uc_stack.ss_sp = c.stack.data();
        c.ctx.uc_stack.ss_size = c.stack.size();
        c.ctx.uc_link = &main;
        makecontext(&c.ctx, &Sched::entry, 0);
    }
    void yield() { swapcontext(&cos[cur]->ctx, &main); }
    // slow: a coroutine taken sixteen times less often than the others, -1: none
    void run(uint64_t seed, int slow) {
        self = this;
        rng.seed(seed);
        for (;;) {
            std::vector<int> live;
            for (int i = 0; i < (int)cos.size(); ++i)
                if (!cos[i]->done) live.push_back(i);
            if (live.empty()) return;
            int i = live[rng() % live.size()];
            if (i == slow && live.size() > 1 && rng() % 16) continue;
            cur = i;
            swapcontext(&main, &cos[i]->ctx);
        }
    }
};
Sched* Sched::self = nullptr;

// The partial sums: random runs of sweeps and rounds in the plans' order, with a
// barrier that only orders.  Every workgroup reads what every workgroup wrote in
// the same reduction.
static void partial_sums(uint64_t seed) {
    std::mt19937_64 rng(seed);
    const int P = 2 + (int)(rng() % 5), G = P + (int)(rng() % 2);
    const ResPlan plan = rng() % 2 ? RES_PLAN_STAB : RES_PLAN_BICG;
    std::vector<ResSlot> seq;
    for (int k = 0; k < 4; ++k) {
        if (rng() % 2) seq.push_back(RES_SWEEP_SLOT);
        for (int i = 0; i < plan.n; ++i) seq.push_back(plan.slot[i]);
    }
    std::vector<int> words((size_t)RES_SUMS * G, -1);
    std::vector<int> arrived(seq.size(), 0);
    Sched s;
    for (int p = 0; p < P; ++p)
        s.spawn([&, p] {
            for (int k = 0; k < (int)seq.size(); ++k) {
                const int nq = RES_SLOT_SUMS[seq[k]];
                int* w = words.data() + (size_t)RES_SLOT_BEGIN[seq[k]] * G;
                for (int q = 0; q < nq; q += 3) {
                    s.yield();
                    w[p * nq + q] = k;
                }
                ++arrived[k];
                while (arrived[k] < P) s.yield();
                for (int b = 0; b < P; ++b)
                    for (int q = 0; q < nq; q += 3) {
                        s.yield();
                        CHECK(w[b * nq + q] == k, "reduction %d of slot %d: workgroup %d reads reduction %d's word of %d",
                              k, (int)seq[k], p, w[b * nq + q], b);
                    }
            }
        });
    s.run(seed, rng() % 2 ? (int)(rng() % P) : -1);
}

// The barrier: workgroups on one to three XCDs meet a few times, over the same
// words launch after launch, some with so few polls that waits give up.
struct At {
    static Sched* s;
    template <ResScope>
    static uint32_t add(uint32_t* p, uint32_t v) {
        s->yield();
        const uint32_t o = *p;
        *p += v;
        return o;
    }
    template <ResScope>
    static uint32_t or_(uint32_t* p, uint32_t v) {
        s->yield();
        const uint32_t o = *p;
        *p |= v;
        return o;
    }
    template <ResScope>
    static uint32_t swap(uint32_t* p, uint32_t v) {
        s->yield();
        const uint32_t o = *p;
        *p = v;
        return o;
    }
    static uint32_t get(const uint32_t* p) {
        s->yield();
        return *p;
    }
    static void set(uint32_t* p, uint32_t v) {
        s->yield();
        *p = v;
    }
    static void sleep() { s->yield(); }
    static void release() {}
    static void acquire() {}
};
Sched* At::s = nullptr;

static int gaveUp = 0, finished = 0, finalAll = 0;
static void barrier(uint64_t seed) {
    std::mt19937_64 rng(seed);
    uint32_t bar[32] = {0}, barL2[RES_XCDS][32] = {{0}};
    for (int launch = 0; launch < 3; ++launch) {
        const int P = 2 + (int)(rng() % 6), nx = 1 + (int)(rng() % 3), K = 1 + (int)(rng() % 4);
        const uint32_t polls = rng() % 2 ? 1000000u : 1u + (uint32_t)(rng() % 60);
        std::vector<int> arrived(K + 1, 0);
        int failed = 0, passed = 0;
        Sched s;
        At::s = &s;
        for (int p = 0; p < P; ++p)
            s.spawn([&, p] {
                const uint32_t x = (uint32_t)(p % nx);
                ResBar B{bar, barL2, P, 1, P, nullptr, polls, 0, 1};
                ++arrived[0];
                if (res_enter_wait<At>(B, x)) {
                    ++failed;
                    return;
                }
                res_enter_place<At>(B, x);
                for (int k = 0;; ++k) {
                    CHECK(arrived[k] == P, "workgroup %d passed barrier %d with %d of %d there", p, k, arrived[k], P);
                    if (k == K) break;
                    s.yield();
                    ++arrived[k + 1];
                    ++B.ph;
                    if (res_wait<At>(B)) {
                        ++failed;
                        return;
                    }
                }
                ++passed;
                res_depart<At>(B);
            });
        s.run(seed * 7 + launch, rng() % 2 ? (int)(rng() % P) : -1);
        bool clean = true;
        for (uint32_t w : bar) clean = clean && w == 0;
        for (auto& l : barL2)
            for (uint32_t w : l) clean = clean && w == 0;
        CHECK(clean || failed, "counters left set with no workgroup to say so");
        if (failed) {  // as the host does
            for (uint32_t& w : bar) w = 0;
            for (auto& l : barL2)
                for (uint32_t& w : l) w = 0;
        }
        CHECK(polls < 1000000u || !failed, "a wait gave up on workgroups that all run");
        (failed == 0 ? finished : passed ? finalAll : gaveUp)++;
    }
}

// The budget: launches and groups come and go in random order.  No XCD is ever
// promised more than it has, every member of a group has all its workgroups in one
// launch on the XCDs counted, and what is held together ends: workgroups placed on
// any CU with room, in any order, do not leave two launches waiting for each other.
static void budget(uint64_t seed) {
    std::mt19937_64 rng(seed);
    const int cus = 2 + (int)(rng() % 6), cap = 2 * cus;
    struct Job {  // one launch under way: workgroups per XCD, in `unit` half CUs
        std::unique_ptr<ResHold> hold;
        int unit;
        std::vector<std::array<int, RES_XCDS>> launches;  // one after another
        int placed[RES_XCDS] = {0};
        std::vector<std::pair<int, int>> on;  // (XCD, CU) of its placed workgroups
        int lane = 0;                         // jobs of a lane run in their order
    };
    ResBudget B;
    std::vector<std::shared_ptr<ResLane>> lanes(3);
    for (auto& l : lanes) l.reset(new ResLane);
    std::vector<Job> jobs;
    for (int i = 0; i < 6; ++i) {
        Job j;
        j.hold.reset(new ResHold);
        j.unit = 1 + (int)(rng() % 2);
        j.lane = (int)(rng() % lanes.size());
        if (rng() % 2) {
            const int P = 2 + (int)(rng() % (RES_XCDS * cus));
            const int x = B.take(P, j.unit, cap, (int)(rng() % RES_XCDS), lanes[j.lane], *j.hold);
            if (x == RES_FULL) continue;
            std::array<int, RES_XCDS> n{};
            for (int p = 0; p < P; ++p) ++n[x == RES_SPREAD ? p % RES_XCDS : x];
            j.launches.push_back(n);
        } else {
            std::vector<ResMember> ms;
            for (int k = 0; k < 1 + (int)(rng() % 9); ++k)
                ms.push_back({1 + (int)(rng() % (rng() % 3 ? 2 * cus : RES_XCDS * cus)), (int)(rng() % 2)});
            std::vector<int> left;
            const std::vector<ResLaunch> ls = B.group(ms, j.unit, cap, lanes[j.lane], *j.hold, left);
            std::vector<int> seen(ms.size(), 0), at(ms.size(), -1);
            bool alone = true;  // no other lane holds anything
            for (const Job& o : jobs) alone = alone && o.lane == j.lane;
            CHECK(!alone || left.empty(), "a lane alone on the device leaves a member out");
            for (int i : left) seen[i] = ms[i].P;
            for (size_t l = 0; l < ls.size(); ++l) {
                std::array<int, RES_XCDS> n{};
                for (size_t b = 0; b < ls[l].map.size(); ++b) {
                    const int m = ls[l].map[b][0];
                    if (m < 0) continue;
                    CHECK(ms[m].form == ls[l].form && (at[m] == -1 || at[m] == (int)l), "member %d in two launches", m);
                    at[m] = (int)l;
                    CHECK(ls[l].map[b][1] < ms[m].P, "member %d has a workgroup too many", m);
                    ++seen[m];
                    ++n[b % RES_XCDS];
                }
                j.launches.push_back(n);
            }
            for (size_t m = 0; m < ms.size(); ++m) CHECK(seen[m] == ms[m].P, "member %d: %d of %d workgroups", (int)m, seen[m], ms[m].P);
        }
        for (const auto& n : j.launches)
            for (int x = 0; x < RES_XCDS; ++x) CHECK(n[x] * j.unit <= j.hold->n[x], "XCD %d: more than is held", x);
        jobs.push_back(std::move(j));
    }
    for (int x = 0; x < RES_XCDS; ++x) {
        int sum = 0;
        for (int l = 0; l < (int)lanes.size(); ++l) {
            int most = 0;
            for (const Job& j : jobs)
                if (j.lane == l) most = std::max(most, j.hold->n[x]);
            CHECK(lanes[l]->n[x] == most, "lane %d takes %d, its launches %d", l, lanes[l]->n[x], most);
            sum += most;
        }
        CHECK(sum <= cap, "XCD %d: %d of %d half CUs promised", x, sum, cap);
    }
    // placement: used[x][c] half CUs; a launch ends once all its workgroups are placed
    std::vector<std::vector<int>> used(RES_XCDS, std::vector<int>(cus, 0));
    while (!jobs.empty()) {
        std::vector<std::array<int, 3>> moves;  // job, XCD, CU
        for (int k = 0; k < (int)jobs.size(); ++k) {
            Job& j = jobs[k];
            bool waits = false;  // for an earlier launch of its stream
            for (int e = 0; e < k; ++e) waits = waits || jobs[e].lane == j.lane;
            if (waits) continue;
            if (j.launches.empty()) {
                moves.push_back({k, -1, -1});
                continue;
            }
            bool all = true;
            for (int x = 0; x < RES_XCDS; ++x)
                if (j.placed[x] < j.launches[0][x]) {
                    all = false;
                    for (int c = 0; c < cus; ++c)
                        if (used[x][c] + j.unit <= 2) moves.push_back({k, x, c});
                }
            if (all) moves.push_back({k, -1, -1});
        }
        CHECK(!moves.empty(), "launches wait for each other");
        const auto mv = moves[rng() % moves.size()];
        Job& j = jobs[mv[0]];
        if (mv[1] >= 0) {
            used[mv[1]][mv[2]] += j.unit;
            ++j.placed[mv[1]];
            j.on.push_back({mv[1], mv[2]});
            continue;
        }
        for (auto& o : j.on) used[o.first][o.second] -= j.unit;
        j.on.clear();
        std::fill(j.placed, j.placed + RES_XCDS, 0);
        if (!j.launches.empty()) j.launches.erase(j.launches.begin());
        if (j.launches.empty()) {
            j.hold->release();
            jobs.erase(jobs.begin() + mv[0]);
        }
    }
    ResHold h;
    CHECK(B.take(RES_XCDS * cus, 2, cap, 3, lanes[0], h) == RES_SPREAD, "not everything was given back");
}

int main() {
    for (uint64_t seed = 1; seed <= 2000; ++seed) budget(seed);
    for (uint64_t seed = 1; seed <= 500; ++seed) partial_sums(seed);
    for (uint64_t seed = 1; seed <= 5000; ++seed) barrier(seed);
    std::printf("launches finished %d, gave up %d, gave up behind the last barrier %d\n", finished, gaveUp, finalAll);
    CHECK(finished > 1000 && gaveUp > 1000 && finalAll > 10, "the schedules miss an outcome");
    std::printf("OK\n");
}
