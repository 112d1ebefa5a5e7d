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

int main() {
    for (uint64_t seed = 1; seed <= 500; ++seed) partial_sums(seed);
    for (uint64_t seed = 1; seed <= 5000; ++seed) barrier(seed);
    std::printf("launches finished %d, gave up %d, gave up behind the last barrier %d\n", finished, gaveUp, finalAll);
    CHECK(finished > 1000 && gaveUp > 1000 && finalAll > 10, "the schedules miss an outcome");
    std::printf("OK\n");
}
