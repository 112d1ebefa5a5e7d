// rt_resident.h -- the memory the workgroups of a resident solve share between
// its barriers.  Plain C++: the host tests run these rules against every
// interleaving the kernels allow.
#pragma once
#include <cstdint>

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

}  // namespace rt
