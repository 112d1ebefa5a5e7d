// rt_resident.h -- the memory the workgroups of a resident solve share between
// its barriers.  Plain C++: the host tests run these rules against every
// interleaving the kernels allow.
#pragma once
#include <cstdint>

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

}  // namespace rt
