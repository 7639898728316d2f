// Words that many workgroups fold a maximum into.
//
// Atomics on one address are served one at a time (about 12 ns each on this part), so a workgroup whose maximum no longer
// raises the word must not queue up for it: of the thousands of chunks of a large tensor only the first few and a
// logarithmic number of later ones raise a maximum.  Ten tensors of 17 to 50 M elements (24 704 chunks of 16 Ki elements,
// three maxima each) spent 0.83 of the 1.27 ms of their first AdamW pass in that queue.
//
// Where the word as it is now is looked at matters: a load at the end of a workgroup waits for the workgroup's stores as
// well (one counter tracks both), which cost a kernel that writes its outputs more than the queue (32 gradients of
// 4 M elements: 66 us with one atomic per chunk, 155 us with such a load in front).  So a kernel that stores looks at
// the word when it starts (`seen`, an older and therefore lower value: some needless atomics, never a missing one), and a
// kernel that only reads looks again at the end.
#pragma once
#include "common.cuh"

namespace msamp {

__device__ __forceinline__ uint32_t seen_word(const uint32_t* word) {
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void raise_max(uint32_t* word, uint32_t v, uint32_t seen) {
    if (v > seen) __hip_atomic_fetch_max(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}    // namespace msamp
