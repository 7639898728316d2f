// Words that many workgroups fold a maximum into, where the tensors can be so large that the atomics queue up.
//
// Atomics on one address are served one at a time (some 30 ns each with 2000 workgroups at it), and a workgroup whose
// maximum no longer raises the word need not queue up for it: of the thousands of chunks of a large tensor only the first
// few and a logarithmic number of later ones raise a maximum.  But the workgroup has to wait for a look at the word, and with
// it for its stores (one counter, in order), where an atomic without a result is sent and forgotten.  So a kernel looks for
// tensors of more chunks than a line measured for it, and always at its end: in front of the loads the look held up the
// first data of every workgroup, and the words it left in registers through the loop cost fused_spec_kernel the fourth
// wavefront of a SIMD; between the last loads and the last stores it was slower than either for tensors of 256 chunks.
// us per step of 240 M parameters in tensors of so many chunks of 16 Ki elements, without and with a look at the end:
//   chunks                                                 256       384       512       768      1024       1536       2048
//   fused_amax_kernel (stores nothing, three maxima)    675, 730  684, 708  683, 710  716, 700  763, 702   957, 690  1195, 724
//   fused_spec_kernel (stores, three maxima)            463, 474  464, 463  483, 457  500, 454  566, 454  1000, 445  1295, 471
// (Few tensors by themselves gain from smaller sizes on, and so the line of the first lies below its row above: eight of 256
// chunks 100, 99, of 384 141, 137, of 512 201, 198.)
// plain_amax_kernel (two maxima, 120 M parameters) is within 1 % either way up to 1536 chunks, and bucket_amax_kernel (one)
// loses up to there (120 M elements, 256 chunks: 69, 148; 1536: 86, 96): they never look.
#pragma once
#include "common.cuh"

namespace msamp {

__device__ __forceinline__ uint32_t seen_word(const uint32_t* word) {
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void raise_max(uint32_t* word, uint32_t v) {
    if (v) __hip_atomic_fetch_max(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// words[0..2] at once, the three looks together
__device__ __forceinline__ void raise_max3(uint32_t* words, uint32_t a, uint32_t b, uint32_t c, bool look) {
    uint32_t sa = 0, sb = 0, sc = 0;
    if (look) sa = seen_word(words), sb = seen_word(words + 1), sc = seen_word(words + 2);
    if (a > sa) raise_max(words, a);
    if (b > sb) raise_max(words + 1, b);
    if (c > sc) raise_max(words + 2, c);
}

}    // namespace msamp
