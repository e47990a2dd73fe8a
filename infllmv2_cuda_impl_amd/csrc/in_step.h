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
// Started together is not enough: a row's own blocks lie where they lie, and after as many of them two rows are up to a fifth of the sequence apart (131 072
// tokens, 31 blocks of a row's own: standard deviation 9 % in the middle, 180 blocks of 32 KiB), while L2 holds 128 blocks.  So the walk is paced too: the blocks that a group of 8
// tokens walks together, in lock step, are its clock.  Behind each of them come kPacedSteps steps for a block of a wavefront's own, and a wavefront takes its next block in a
// step only if the block lies before a front that crosses the group's keys evenly in the steps there are - or if it has a block left for every
// step left, so that no row ends later for it, wherever its blocks lie.  With two steps to a common block a row has twice as many as blocks of its own, is rarely
// held up, and passes a block when the others do.  The rule looks at the group's rows alone: the order in which a row's blocks are added up,
// and with it the result's bits, are the same in every launch.  131 072 tokens, 64 blocks: L2 serves 80 % of the requests instead of 57, 60 GB come from behind it instead of 125,
// forward 19.4 -> 14.1 ms, whole prefill 26.0 -> 20.9; 65 536: 8.8 -> 7.95; 40 000: 4.5 -> 4.4.  One step to a common block 24.9, 8.6, 4.5, three 20.9, 8.0, 4.4.
// Groups that end behind block 384: 20.8, 7.9, 4.4; 768: 21.2, 8.2, 4.6.  Below 32 768 keys, waiting and paced or not: within 1 % either way.
// That is with a row's own blocks anywhere.  Forward in ms, in step | paced too (and five of eight rows in the ring), a window of 32 blocks and 32 blocks that lie, 131 072 tokens with
// one KV head; 65 536 with two: anywhere 9.5 | 6.7; 6.5 | 5.8.  In four runs of eight 13.0 | 10.3; 9.5 | 7.4.  In one run 15.1 | 15.2; 11.3 | 11.2.  Half of them anywhere, half the same
// for 64 tokens 7.0 | 5.8; 5.8 | 5.3.  Within one block of the same for 8 tokens 6.13 | 6.08; 5.58 | 5.61, for 64 5.58 | 5.71; 5.36 | 5.40, for 512 5.55 | 5.60; 5.29 | 5.33.  In the first
// tenth 5.29 | 5.23; 4.72 | 4.60, in the 64 blocks before the window 5.18 | 5.17; 5.04 | 5.04, between 80 and 95 % of the way 5.27 | 5.40; 4.62 | 4.68: where L2 has the blocks
// anyway the pace costs up to 2 %, where it has not it gives up to 30.
//
// With the device shared a generation is more than an XCD runs at once, and CUs that become free wait for its second half.  What sharing fetches gives is still
// more than that costs; forward in ms, in step and paced | in step | neither, 2 KV heads, 64 blocks selected (the first, a window of 32, the rest anywhere), as many as keep both
// streams busy: 131 072 tokens alone 13.2 | 18.4 | 24.9, two such forwards on two streams (time of one) 40.7 | 49.7 | 60.5, beside products of 8192^3 45.7 | 51.3 | 53.4, beside
// copies of 0.5 GiB 29.9 | 31.6 | 35.9, beside products of 64 rows 24.0 | 26.8 | 29.7; 40 000: 3.3 | 3.4 | 3.6, 8.1 | 8.9 | 11.8, 10.4 | 10.7 | 11.4, 7.4 | 7.4 | 7.2, 4.9 | 5.1 | 5.6.
//
// Which launches (measured before there was a pace): at 30 000 tokens a whole prefill gained 1 % and at 32 768 it gained or lost less (L2 serves 91 % of the requests
// there and the wait for a generation's slowest workgroup costs 2 %); at 40 000 it gained 7 %, at 49 152 14, at 65 536 22 (10.9 -> 8.5 ms,
// two KV heads), at 98 304 20, at 131 072 17 (31.3 -> 25.9).  Only wavefronts whose row has blocks of its own in
// several mask words wait: with window masks everything is shared (60 000 tokens, 6 blocks: 473 us without all this, 478 with the counters and no waits).  Letting up to 2 | 4 | 8 workgroups of a
// generation start early: 131 072 tokens 14.05 -> 14.85 | 15.7 | 17.8 ms.  Meeting again 1 | 3 | 7 times during the walk: 13.95 | 14.7 | 16.8, 65 536 tokens 6.05 -> 6.2 | 6.6 | 7.4.  Walking
// every other generation downwards gave nothing (before there was a pace).  The dQ kernel walks the same way but is not bound by its fetches: waiting cost it 2 %
// of its time at 40 000 tokens and gained nothing at 64 000.
#pragma once
#include "common.h"
#include "infllmv2_hip.h"

namespace IV2_NS {

constexpr int kGeneration = 32;
constexpr int kInStepKeys = INFLLMV2_IN_STEP_KEYS;             // sequences with more keys than this: 32 768
constexpr int kInStepWords = 4;                                // and rows with blocks of their own in at least so many mask words
constexpr int kPacedBlocks = kInStepKeys / kBlockN;            // groups that reach beyond so many blocks are paced, in every launch that can hold such a group
constexpr int kPacedSteps = 2;
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
