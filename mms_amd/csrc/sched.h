// How the wavefronts of a workgroup share its items in a scheduled launch (sim_mixed.hip, sim_lanes.hip).
#pragma once

#include "mmsim_internal.h"

namespace mmsim {
namespace {

// Schedule state of one workgroup (in LDS behind the latency table): one word per item, twice the segment
// the item is at, plus one while a wavefront is simulating that segment.  A wavefront takes an item by
// compare-and-swap on its word and hands it back with a plain atomic store, so there is no lock to hold.
struct SchedLds {
    uint32_t item[kMaxGroupItems];
};
static_assert(sizeof(SchedLds) <= kSchedLdsBytes, "schedule state outgrew its LDS reservation");

// Takes the item of this workgroup that is furthest behind among those that fit this wavefront's LDS
// region and that nobody is simulating right now (ties: the largest, so that the large regions serve
// the large items).  One lane looks and claims the item with a compare-and-swap; if another
// wavefront was faster it looks again.  -1: nothing left for this wavefront.  -2: what is left is being simulated by
// others right now; wait a little for a segment to end and look again (a wavefront that has waited long leaves: no item
// depends on it, an item is either being simulated or was just handed back by a wavefront that is about to look for
// work itself).
__device__ __forceinline__ int sched_claim(SchedLds *sched, const MixedArgs &a, int item0, int n_items, int part_bytes, int lane) {
    int got = -1;
    if (lane == 0) {
        for (int tries = 0; tries < 64; ++tries) {
            int best = -1, best_bytes = -1;
            uint32_t best_word = 0xFFFFFFFFu;
            bool pending = false;
            for (int k = 0; k < n_items; ++k) {
                const uint32_t w = __hip_atomic_load(&sched->item[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                const int sg = (int)(w >> 1), nsg = a.item_nseg[item0 + k];
                const int bytes = a.item_bytes[item0 + k];
                if (sg >= nsg || bytes > part_bytes) continue;
                if (w & 1u) {  // worth waiting for only if a segment follows the one being simulated
                    if (sg + 1 < nsg) pending = true;
                    continue;
                }
                if (w < best_word || (w == best_word && bytes > best_bytes)) {
                    best = k;
                    best_word = w;
                    best_bytes = bytes;
                }
            }
            if (best < 0) {
                got = pending ? -2 : -1;
                break;
            }
            uint32_t expect = best_word;
            if (__hip_atomic_compare_exchange_strong(&sched->item[best], &expect, best_word | 1u, __ATOMIC_ACQUIRE,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) {
                got = best;
                break;
            }
            got = -2;  // lost the race for that item: look again (or, after many losses, sleep first)
        }
    }
    return __builtin_amdgcn_readfirstlane(got);
}

// The segment that a claimed item is at; afterwards the state that another wavefront parked for it can be read.
__device__ __forceinline__ int sched_segment(SchedLds *sched, int item_k) {
    const int seg = __builtin_amdgcn_readfirstlane(
        (int)(__hip_atomic_load(&sched->item[item_k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> 1));
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return seg;
}

// Hands the item back: its parked state must be visible to whichever wavefront takes its next segment.
__device__ __forceinline__ void sched_hand_back(SchedLds *sched, const MixedArgs &a, int item_k, int seg, bool last_seg, int lane) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (lane == 0) {
        __hip_atomic_store(&sched->item[item_k], (uint32_t)(seg + 1) << 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (last_seg) atomicAdd(a.error + 1, 1);  // items completed: the host checks that none is missing
    }
}

}  // namespace
}  // namespace mmsim
