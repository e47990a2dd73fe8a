// Workgroups of the Stage-2 forward walk long sequences in step.
//
// Past some length the block images of one KV head exceed an XCD's 4 MiB of L2 many times over, and what a token walks on its own is
// fetched from the fabric behind it.  Every row is walked in ascending order at the same pace, so workgroups that start
// together pass a key block at about the same time and share its fetch; started whenever a CU becomes free, they are spread
// over the whole sequence.  A wavefront therefore sets itself up and then waits until the workgroups of its XCD that belong to earlier
// generations (a generation is what an XCD runs at once: a workgroup on each of its 32 CUs) have finished their walks, by their first wavefronts' word.
//
// The wait is a matter of speed only: nothing depends on which workgroups run at once, a workgroup of an earlier generation never
// waits for a later one, and a wait ends after kInStepPolls looks whatever the counters hold.
//
// With the device shared a generation is more than an XCD runs at once, and CUs that become free wait for its second half.  What sharing fetches gives is still
// more than that costs; forward in ms, in step | not, 2 KV heads, 64 blocks selected, as many as keep both streams busy: 65 536 tokens alone 6.9 | 9.5, two such forwards on two
// streams (time of both) 19.5 | 25.0, beside products of 8192^3 14.8 | 16.7, beside copies of 0.5 GiB 14.1 | 15.5, beside products of 64 rows 10.7 | 10.7; 131 072: 19.2 | 24.7,
// 50.2 | 57.6, 38.2 | 41.1, 32.9 | 37.0, 21.5 | 25.6; 40 000: 3.6 | 3.8, 9.4 | 12.4, 7.5 | 7.7, 6.5 | 6.8, 5.4 | 5.4.
//
// Which launches: at 30 000 tokens a whole prefill gained 1 % and at 32 768 it gained or lost less (L2 serves 91 % of the requests
// there and the wait for a generation's slowest workgroup costs 2 %); at 40 000 it gained 7 %, at 49 152 14, at 65 536 22 (10.9 -> 8.5 ms,
// two KV heads), at 98 304 20, at 131 072 17 (31.3 -> 25.9).  Only wavefronts whose row has blocks of its own in
// several mask words wait: with window masks everything is shared (60 000 tokens, 6 blocks: 473 us without all this, 478 with the counters and no waits).  Letting up to 8 workgroups of a
// generation start early gave back a quarter of the gain; more meeting points during the walk, or walking every other
// generation downwards, gave nothing more.  The dQ kernel walks the same way but is not bound by its fetches: waiting cost it 2 %
// of its time at 40 000 tokens and gained nothing at 64 000.
#pragma once
#include "common.h"

namespace IV2_NS {

constexpr int kGeneration = 32;
constexpr int kInStepKeys = 32768;                             // sequences with more keys than this
constexpr int kInStepWords = 4;                                // and rows with blocks of their own in at least so many mask words
constexpr int kInStepPolls = 256;                              // of about a microsecond each
constexpr int kInStepPitch = 32;                               // the XCDs' counters lie 128 bytes apart
constexpr size_t kInStepBytes = 8 * kInStepPitch * sizeof(unsigned);

// counter: of the workgroup's XCD, how many workgroups have finished their walk; order: the workgroup's number on its XCD
__device__ __forceinline__ void in_step_finished(unsigned* counter) {
    __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void in_step_wait(const unsigned* counter, int order) {
    const unsigned before = static_cast<unsigned>(order / kGeneration) * static_cast<unsigned>(kGeneration);
    for (int poll = 0; poll < kInStepPolls; ++poll) {
        if (__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= before) return;
        __builtin_amdgcn_s_sleep(4);
    }
}

}  // namespace IV2_NS
