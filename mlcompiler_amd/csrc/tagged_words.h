// Words that workgroups of one launch leave each other in memory: {value, tag}, written and read whole (64-bit relaxed
// atomics at device scope: the store is written through to memory, the load bypasses the per-XCD L2 caches).  The tag is
// the launch's, never seen in the buffer before, so every word says by itself whether it has been written in this
// launch: no order among the stores, no acknowledgement, no arrival counter, nothing to clear until the tags start over
// (renew_tags).  A word gets from one workgroup to another in 0.5 us, on the same XCD or not; in 2 us
// where thousands of waves poll words of the same few lines.
//
// Why every wait ends.  Each XCD starts its workgroups of a launch in the launch's order, but the XCDs run ahead of each
// other, and who shares words with whom need not be on one XCD nor running at the same time.
//   * K slices of a matmul: only workgroups of the last slice wait, and they are the last of the launch.  While a workgroup
//     of another slice has yet to start on some XCD, no waiting one has started there, and the others end by themselves.
//   * Partials of the decode attention: a workgroup waits for workgroups with lower numbers only, after it has published
//     its own part.  Take the lowest number that has not published: whatever has started before it on its XCD waits for
//     lower numbers at most, which all have, and ends.
//   * Two matmuls in one launch: the second one's workgroups, the last of the launch, wait for the first one's, which wait for
//     each other's slices at most.  None of the second's has started on an XCD where one of the first's has yet to start.
// That holds for one such launch at a time (scratch_follow orders those of a process across streams), beside launches that
// end by themselves.  Two processes on a GPU are not ordered.  K slices of up to 64 requests end even then: who waits has its
// partners on its own XCD.  So do two matmuls in one launch: a workgroup that waits may have a CU to itself (1024 threads of up to
// 128 registers), but those of one launch leave a CU of every XCD to others (launch_chain): room for the first matmuls' workgroups, and
// for what the other process has yet to start.  With a third process they need not end, nor the decode launches
// of two processes beside each other, nor K slices of many tokens: each may hold the place that the other waits for.  The
// waits are bounded all the same: a pass then fails instead of hanging.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlc_hip {

__device__ __forceinline__ void st_tagged(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ld_tagged(const uint64_t* p) {
    return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The tag of a launch: its own number, and in a captured pass, whose arguments are the same at every replay, the replay
// word on top.  Never zero, which is what untouched memory holds.
__device__ __forceinline__ uint32_t launch_tag(uint32_t tag, uint32_t replay_word) {
    const uint32_t sum = tag + replay_word;
    return sum ? sum : 0x9E3779B9u;
}

// Tells the host that a wait for such words was given up.
__device__ __forceinline__ void report_fault(uint32_t* fault) {
    __hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What a launch needs to know for it.
struct TagArgs {
    const uint32_t* tag_dev;    // null, or a device word that is added to `tag` (captured passes)
    uint32_t* fault;            // host-visible word, set when a wait was given up
    uint32_t tag;               // this launch's tag: differs from that of every earlier launch whose words may still lie there
    uint32_t spin_limit;        // rounds a wait polls before it gives up
    uint32_t test_flags;        // bit 0: words are not published (tests of the give-up path)
};

}  // namespace mlc_hip
