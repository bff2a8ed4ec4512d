// A simulation of a long stream cut into runs that are simulated at the same time (sim_window.hip says how): what the kernels
// that do so share.  Device code.
#pragma once
#include "mmsim_internal.h"

namespace mmsim {
namespace {

// What wavefronts of different workgroups tell one another while the kernel runs: stores and loads that all of the device sees.
// A mark is told, the wavefront waits until its stores have been carried out, and only then tells that the mark is there; who is told so
// asks for the mark afterwards.  (The waits are instructions of this hardware.  A release and an acquire at device scope would say the same in the
// language's terms, but write back and throw away caches at every mark: 179 placements of 25094 requests 0.335 -> 0.557 ms, 79 of 98901 0.87 -> 1.20.)
__device__ __forceinline__ void tell(uint64_t *p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void tell(uint32_t *p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint64_t told(const uint64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t told(const uint32_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The arguments as they lie in memory, for what is done rarely: asked for there, and not kept in scalar registers, which the loop over blocks
// has none to spare of (71 of its instructions, of 930 a block, moved them to and fro).
template <class Args>
__device__ __forceinline__ const __attribute__((address_space(4))) Args *cold_args() {
    const __attribute__((address_space(4))) Args *p = (const __attribute__((address_space(4))) Args *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

struct Runs {  // what a run goes by (scalars; blocks of 64 requests)
    int own;         // the run, or -1: one that is taken up again
    int in, mark;    // the span of the next mark, and which of that span's it is
    uint32_t since;  // where the run left its own span
    uint32_t next;   // block before which something happens
    bool looked;     // another run's mark: what to compare with is on its way (asked for a block ahead)
    bool met;        // the run of span `in` at that mark

    // known to be what the simulation does: the first run, or one taken up again
    __device__ __forceinline__ bool true_one() const { return own <= 0; }
    template <class A>
    __device__ __forceinline__ uint32_t limit(A *a) const {
        return true_one() ? 0xFFFFFFFFu : (uint32_t)((own + 1) * a->span_blocks + a->ext_blocks);
    }
    template <class A>
    __device__ __forceinline__ void start(A *a, int span) {
        own = in = span;
        mark = 0;
        looked = met = false;
        since = (uint32_t)((own + 1) * a->span_blocks);
        next = (uint32_t)(own * a->span_blocks + span_mark(0));  // (within the span: it has more than eight blocks)
    }
    template <class A>
    __device__ __forceinline__ void resume(A *a, uint32_t at) {
        own = -1;
        in = (int)(at / (uint32_t)a->span_blocks);
        mark = -1;
        met = false;
        since = at;
        go_on(a, at);
    }
    // From block `at` to the next mark: of its own span all, of others those that are further by an eighth of how far the run has come on
    // its own (a run that meets nobody looks fifty times or so, not at every mark of the stream).
    template <class A>
    __device__ __forceinline__ void go_on(A *a, uint32_t at) {
        const int span = a->span_blocks;
        const uint32_t least = at < since ? 0u : at + 2u + (at - since) / 8u;
        uint32_t m;
        do {
            mark += 1;
            if (span_mark(mark) >= span) {
                in += 1;
                mark = 0;
            }
            m = (uint32_t)(in * span + span_mark(mark));
        } while (m < least);
        looked = false;
        next = in != own ? m - 1u : m;
        next = next < limit(a) ? next : limit(a);
    }
};

}  // namespace
}  // namespace mmsim
