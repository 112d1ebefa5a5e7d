// rt_resident.h -- the memory the workgroups of a resident solve share between
// its barriers.  Plain C++: the host tests run these rules against every
// interleaving the kernels allow.
#pragma once
#include <algorithm>
#include <array>
#include <cstdint>
#include <memory>
#include <mutex>
#include <vector>

#ifdef __HIP__
#define RES_FN __device__ __forceinline__
#else
#define RES_FN inline
#endif

namespace rt {

// Partial sums.  Every reduction of a resident solve is: each workgroup writes
// its sums, a barrier, each workgroup reads the sums of all.  Nothing orders a
// workgroup that has read them, and goes on, against one that has not yet, up
// to the next barrier.  So two reductions that follow each other never use the
// same slot: a slot's next use is then at least one whole reduction away, and
// that reduction's barrier is one every workgroup reaches only after its reads
// of the slot.  In words per row-kernel workgroup:
//   RS_T  the t pass and the sweep's residual (18 sums)
//   RS_V  the v pass, PBiCG's w pass (6)
//   RS_X  the x/r passes (12)
enum ResSlot { RS_T, RS_V, RS_X };
constexpr int RES_SLOT_BEGIN[] = {0, 18, 24};
constexpr int RES_SLOT_SUMS[] = {18, 6, 12};
constexpr int RES_SUMS = 36;  // of all slots

// the reductions of one round, in order; a refinement sweep (RES_SWEEP_SLOT)
// stands between rounds and never follows another sweep without a round between
struct ResPlan {
    int n;
    ResSlot slot[3];
};
constexpr ResPlan RES_PLAN_STAB{3, {RS_V, RS_T, RS_X}};  // v, t, x/r
constexpr ResPlan RES_PLAN_BICG{2, {RS_V, RS_X}};        // w, x/r
constexpr ResSlot RES_SWEEP_SLOT = RS_T;

constexpr bool resPlanHolds(const ResPlan& p) {
    for (int i = 0; i < p.n; ++i)
        if (p.slot[i] == p.slot[(i + 1) % p.n]) return false;
    return p.slot[0] != RES_SWEEP_SLOT && p.slot[p.n - 1] != RES_SWEEP_SLOT;
}
static_assert(resPlanHolds(RES_PLAN_STAB) && resPlanHolds(RES_PLAN_BICG), "consecutive reductions share a slot");
static_assert(RES_SLOT_BEGIN[RS_T] + RES_SLOT_SUMS[RS_T] <= RES_SLOT_BEGIN[RS_V] &&
                  RES_SLOT_BEGIN[RS_V] + RES_SLOT_SUMS[RS_V] <= RES_SLOT_BEGIN[RS_X] &&
                  RES_SLOT_BEGIN[RS_X] + RES_SLOT_SUMS[RS_X] <= RES_SUMS,
              "partial-sum slots overlap");

// The barrier's words (SolveState::bar and ::barL2).  Every workgroup arrives on
// its XCD's counter here[0].  On one XCD all wait there.  On several, the last
// arrival of an XCD arrives on bar[2], waits for the other XCDs' and then counts
// the barrier on here[1], where the rest of its XCD waits.
//
// A wait that polls maxPolls times sets RES_FAIL, the top bit of the word it
// waits on.  The bit is only ever set with an or and never cleared before the
// host does: added instead, two of them carry out of the word and leave a count
// that reads as a passed barrier.  Counts stay below it.  So a workgroup that
// passes a barrier knows that every workgroup had arrived at it, whoever gave up.
// At: the memory's operations on a word (add, or_, swap give the old value).
constexpr uint32_t RES_FAIL = 0x80000000u;
constexpr int RES_XCDS = 8;
enum ResScope { RES_XCD, RES_CHIP };  // executed in the XCD's L2; seen by the whole chip

struct ResBar {
    uint32_t* bar;         // [0] entered, [1] left, [2] the XCDs' barrier, [8 + x] workgroups on XCD x
    uint32_t (*barL2)[32];  // [x]: XCD x's arrivals, barriers, departures
    int P, nXcd, nHere;    // workgroups; XCDs they are on; workgroups on this one
    uint32_t* here;        // barL2 of this XCD
    uint32_t maxPolls, ph, one;  // ph: barriers so far; one: 1, unknown to the compiler
};

// Polls *p (an atomic add of 0: L2 executes it, no L1 copy is read) until its low
// bits reach target; returns with RES_FAIL set if a wait gave up, this or another
template <class At, ResScope S>
RES_FN uint32_t res_poll(uint32_t* p, uint32_t v, uint32_t target, const ResBar& B) {
    for (uint32_t n = 0; v < target;) {
        if (++n > B.maxPolls) return At::template or_<S>(p, RES_FAIL) | RES_FAIL;
        At::sleep();
        v = At::template add<S>(p, B.one - 1u);
    }
    return v;
}
// Before the first pass, one thread of a workgroup on XCD x: counts the workgroups
// on each XCD and waits for all of them, with a counter of its own and every
// workgroup fencing.  True: a wait gave up.
template <class At>
RES_FN bool res_enter_wait(const ResBar& B, uint32_t x) {
    At::template add<RES_CHIP>(&B.bar[8 + x], 1u);
    At::release();
    const uint32_t v = res_poll<At, RES_CHIP>(B.bar, At::template add<RES_CHIP>(B.bar, 1u) + 1u, (uint32_t)B.P, B);
    At::acquire();
    return ((v | At::template add<RES_CHIP>(B.bar, B.one - 1u)) & RES_FAIL) != 0;
}
// all threads, behind it: where the workgroups are
template <class At>
RES_FN void res_enter_place(ResBar& B, uint32_t x) {
    B.nXcd = 0;
    for (int i = 0; i < RES_XCDS; ++i) B.nXcd += At::get(&B.bar[8 + i]) != 0;
    B.nHere = (int)At::get(&B.bar[8 + x]);
    B.here = B.barL2[x];
}
// Barrier B.ph, one thread, the workgroup's stores done.  True: a wait gave up.
template <class At>
RES_FN bool res_wait(const ResBar& B) {
    uint32_t v = At::template add<RES_XCD>(&B.here[0], B.one) + 1u;
    const uint32_t full = B.ph * (uint32_t)B.nHere;
    if (B.nXcd == 1) {
        v = res_poll<At, RES_XCD>(&B.here[0], v, full, B);
    } else if (v == full) {
        At::release();
        uint32_t* g = &B.bar[2];
        v = res_poll<At, RES_CHIP>(g, At::template add<RES_CHIP>(g, 1u) + 1u, B.ph * (uint32_t)B.nXcd, B);
        At::acquire();
        v |= At::template add<RES_CHIP>(g, B.one - 1u);
        if (v & RES_FAIL) At::template or_<RES_XCD>(&B.here[1], RES_FAIL);
        v = At::template add<RES_XCD>(&B.here[1], B.one) | (v & RES_FAIL);
    } else {
        v = res_poll<At, RES_XCD>(&B.here[1], At::template add<RES_XCD>(&B.here[1], B.one - 1u), B.ph, B);
    }
    At::acquire();
    v |= At::template add<RES_XCD>(&B.here[B.nXcd == 1 ? 0 : 1], B.one - 1u);
    return (v & RES_FAIL) != 0;
}
// Past the last barrier, one thread: the last workgroup of an XCD, and the last of
// all, leave their counters at zero for the next launch.
template <class At>
RES_FN void res_depart(const ResBar& B) {
    if (At::template add<RES_XCD>(&B.here[2], B.one) + 1u == (uint32_t)B.nHere)
        for (int i = 0; i < 3; ++i) At::template swap<RES_XCD>(&B.here[i], 0u);
    if (At::template add<RES_CHIP>(&B.bar[1], 1u) + 1u == (uint32_t)B.P)
        for (int i = 0; i < 8 + RES_XCDS; ++i) At::set(&B.bar[i], 0u);
}

// ------------------------------------------------------------------ host side
// A barrier needs its workgroups on the chip together.  Two launches that each
// got part of their workgroups placed wait for each other until their polls run
// out, so the resident launches of a process take their CUs from one budget per
// device: per XCD, in half CUs (an FP32 solve's workgroup takes half a CU's
// registers, an FP64 one's a whole CU's).  What is held together always fits:
// FP32 workgroups can share every CU that no FP64 one is on, and once they end,
// which they do, the FP64 ones have a CU each.  Other kernels end by themselves.
// Another process's launches are not counted: there the bounded wait remains.
// Launches of one stream run one after another, so a stream (ResLane) takes the
// most that any of its launches under way holds.
class ResBudget;
struct ResHold;
struct ResLane {
    int n[RES_XCDS] = {0};    // the most of its holds
    ResHold* first = nullptr;  // its holds
};
struct ResHold {  // what a launch holds, given back once it has ended
    ResBudget* from = nullptr;
    std::shared_ptr<ResLane> lane;
    ResHold* next = nullptr;
    int n[RES_XCDS] = {0};
    ResHold() = default;
    ResHold(const ResHold&) = delete;
    ResHold& operator=(const ResHold&) = delete;
    ~ResHold() { release(); }
    inline void release();
};

// one launch of a group: workgroup b of the grid (on XCD b % RES_XCDS) is
// {member, its workgroup}, {-1, 0} for none
struct ResLaunch {
    int form = 0;
    int load[RES_XCDS] = {0};
    std::vector<std::array<int32_t, 2>> map;
};
struct ResMember {
    int P, form;
};
constexpr int RES_SPREAD = -1, RES_FULL = -2;

class ResBudget {
    std::mutex mu;
    int held[RES_XCDS] = {0};  // of all lanes
    static int share(int P, int x) { return (P - x + RES_XCDS - 1) / RES_XCDS; }  // of P dealt over all XCDs
    int others(const ResLane& l, int x) const { return held[x] - l.n[x]; }
    void settle(ResLane& l) {
        for (int x = 0; x < RES_XCDS; ++x) {
            int most = 0;
            for (const ResHold* h = l.first; h; h = h->next) most = std::max(most, h->n[x]);
            held[x] += most - l.n[x];
            l.n[x] = most;
        }
    }
    void give(const std::shared_ptr<ResLane>& l, ResHold& h) {
        h.from = this;
        h.lane = l;
        h.next = l->first;
        l->first = &h;
        settle(*l);
    }

   public:
    // A launch of P workgroups of `unit` half CUs each; cap: half CUs of an XCD.
    // The XCD (of those with room the one with most, from `first` on) that takes
    // them all, RES_SPREAD: dealt over all, or RES_FULL
    int take(int P, int unit, int cap, int first, const std::shared_ptr<ResLane>& lane, ResHold& h) {
        std::lock_guard<std::mutex> lk(mu);
        int best = RES_FULL;
        for (int i = 0; i < RES_XCDS; ++i) {
            const int x = (first + i) % RES_XCDS;
            if (others(*lane, x) + P * unit <= cap && (best < 0 || others(*lane, x) < others(*lane, best))) best = x;
        }
        if (best >= 0) {
            h.n[best] = P * unit;
        } else {
            for (int x = 0; x < RES_XCDS; ++x)
                if (others(*lane, x) + share(P, x) * unit > cap) return RES_FULL;
            for (int x = 0; x < RES_XCDS; ++x) h.n[x] = share(P, x) * unit;
            best = RES_SPREAD;
        }
        give(lane, h);
        return best;
    }
    // The launches, one after another on a stream, of a group of solves: a member
    // goes to the XCD with the most room left, one that no XCD can take over all
    // of them (the largest members first would pack tighter; a queue's order keeps
    // its latency).  Holds the most any launch places on an XCD; left: the members
    // no launch can take beside what others hold.
    std::vector<ResLaunch> group(const std::vector<ResMember>& ms, int unit, int cap,
                                 const std::shared_ptr<ResLane>& lane, ResHold& h, std::vector<int>& left) {
        std::lock_guard<std::mutex> lk(mu);
        int room[RES_XCDS];  // workgroups
        for (int x = 0; x < RES_XCDS; ++x) room[x] = std::max(0, cap - others(*lane, x)) / unit;
        std::vector<ResLaunch> out;
        const ResLaunch none;
        auto freest = [&](const ResLaunch& L) {
            int b = 0;
            for (int x = 1; x < RES_XCDS; ++x)
                if (room[x] - L.load[x] > room[b] - L.load[b]) b = x;
            return b;
        };
        auto spreads = [&](const ResLaunch& L, int P) {
            for (int x = 0; x < RES_XCDS; ++x)
                if (L.load[x] + share(P, x) > room[x]) return false;
            return true;
        };
        for (int i = 0; i < (int)ms.size(); ++i) {
            const int P = ms[i].P;
            const bool one = room[freest(none)] >= P;
            if (!one && !spreads(none, P)) {
                left.push_back(i);
                continue;
            }
            const bool open = !out.empty() && out.back().form == ms[i].form;
            if (!open || !(one ? room[freest(out.back())] - out.back().load[freest(out.back())] >= P : spreads(out.back(), P))) {
                out.emplace_back();
                out.back().form = ms[i].form;
            }
            ResLaunch& L = out.back();
            const int on = one ? freest(L) : RES_SPREAD;
            for (int p = 0; p < P; ++p) {
                const int x = one ? on : p % RES_XCDS;
                const size_t b = (size_t)RES_XCDS * L.load[x]++ + x;
                if (L.map.size() <= b) L.map.resize(b + 1, {-1, 0});
                L.map[b] = {i, p};
            }
        }
        for (int x = 0; x < RES_XCDS; ++x) {
            h.n[x] = 0;
            for (const ResLaunch& L : out) h.n[x] = std::max(h.n[x], L.load[x] * unit);
        }
        give(lane, h);
        return out;
    }
    void takeBack(ResHold& h) {
        std::lock_guard<std::mutex> lk(mu);
        ResHold** p = &h.lane->first;
        while (*p != &h) p = &(*p)->next;
        *p = h.next;
        settle(*h.lane);
    }
};

// A wait that gave up cost the time of all its polls (about 0.1 s) and a step by
// launches.  What kept the workgroups apart, another process's work, is likely to
// be there at the next step too, so the context's next solves run by launches: 64
// after the first, twice as many after each further one, until as many resident
// solves as that have finished again.
struct ResBackoff {
    uint32_t pause = 0, span = 0, good = 0;
    bool skip() { return pause > 0 && pause-- > 0; }  // of a solve that would run resident
    void gaveUp() {
        span = std::min(std::max(2 * span, 64u), 65536u);
        pause = span;
        good = 0;
    }
    void finished() {
        if (span > 0 && ++good >= span) span = 0;
    }
};

inline void ResHold::release() {
    if (!from) return;
    from->takeBack(*this);
    from = nullptr;
    lane.reset();
    next = nullptr;
    for (int& v : n) v = 0;
}

}  // namespace rt
