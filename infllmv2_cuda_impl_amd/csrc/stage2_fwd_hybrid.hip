// Stage-2 forward, workgroup-hybrid kernel (gfx950).
//
// Same mathematics and register layout as stage2_fwd_kernel (stage2_fwd.hip: one wavefront owns
// one token, S^T = K Q^T, O^T = V^T P^T, online softmax); what changes is who fetches K/V.
// A workgroup of 8 wavefronts owns 8 consecutive tokens of one sequence and KV head and splits
// each token's mask row in two:
//
//   * the blocks that five or more of the 8 rows select (for InfLLM-V2 masks: the initial block, the local
//     window, and what neighbouring tokens share beyond) are walked in lock step: every such block is
//     copied once, by LDS-DMA, from its fragment-major image into a 4-tile LDS ring (two blocks in
//     use, the next two in flight: one workgroup barrier per two blocks), and each wavefront whose row selects it
//     reads its MFMA operands with conflict-free ds_read_b128;
//     Five: a block of the ring costs the vector memory path one fetch and the LDS pipe, twice as wide, one for every row that selects it, a block outside
//     it the former one for every such row.  From all eight down to six | five | four | three, whole passes in us: one prompt of 2048 tokens with 16 blocks
//     80.3 -> 79.3 | 77.2 | 77.4 | 80.0; four ragged prompts 1032 -> 1037 | 1023 | 1001 | 1013; training on four short samples 617 -> 614 | 612 | 612 | 617;
//     2049 queries behind 17962 keys 321.5 -> 322.3 | 322.8 | 328.9 | 330.7; 32768 tokens the same | the same | 1 % more | 9 % more: where rows share
//     little, wavefronts wait for the few that want a ring block.
//   * the remaining blocks of a row are walked by its wavefront alone, operands straight from
//     global memory into registers, as in stage2_fwd_kernel;
//   * the two walks are interleaved, common, own, common, own per turn: the first is bound by
//     the matrix pipeline and the VALU, the second by the vector memory path.  A row with few blocks more than the ring
//     walks them beside ring blocks that are not its own (kOwnBeside in block_walker.h).
//
// A per-token kernel is bound by what the vector memory path can deliver (32 KiB of operands per
// 512 MFMA cycles); the shared walk takes the common half of the work off that path.  Online
// softmax is order-independent, so the split changes nothing in the result.
//
// Workgroups are numbered so that each of the 8 XCDs takes shares of consecutive token
// groups of one KV head (their L2 sees one head's images and neighbouring local windows), and
// the longest causal prefixes are scheduled first (group_order.h).
// Long sequences are walked in step with the other workgroups of the XCD, at a given pace (in_step.h).
#include "common.h"
#include "kv_image.h"
#include "block_walker.h"
#include "group_order.h"
#include "lds_dma.h"
#include "in_step.h"
#include "stage2_fwd.h"
#include <math.h>
#include <type_traits>

namespace IV2_NS {

constexpr int kHybTokens = 8;                                  // tokens (= wavefronts) per workgroup
constexpr int kRingTiles = 4;
constexpr int kTileBytes = 32768;                              // K image | V image of one block
constexpr int kMaxMaskWords = 256;                             // LDS copies of the mask rows hold at most this many words each: 16384 key blocks

struct HybridExtra {
    int groups_per_seq;                                        // ceil(max_seqlen_q / kHybTokens)
    GroupOrder order;                                          // of all groups, or of all but the late ones
    int total_groups;                                          // places
    int late;                                                  // short groups that go last: num_heads_k * batch, or 0
    int mask_words;                                            // words per LDS mask row: what max_seqlen_k needs, not the maximum
    unsigned* finished;                                        // the XCDs' counters of in_step.h, or null: no workgroup waits
};

__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Online-softmax update with one 16 x 64 score tile (s: S^T accumulators); returns P as the B operand of P.V.
//
// m is the REFERENCE exponent of the lane's head (log2 units, the same in the four lanes that share a head), not
// necessarily its running maximum: P = exp2(scale s - m), l and O are all kept relative to m, and out = O / l and
// LSE = m ln2 + log l hold for any finite m.  So the common path takes m as it is - no row maximum, no cross-lane
// exchange, no rescale of O - and only checks afterwards that its sixteen P values stayed small (their sum is needed
// anyway): a lane whose sum exceeds 2^kLazyBits, or whose head has no reference yet, sends the wavefront through the
// exact path, which moves m to the true running maximum and rescales.  P is rounded to the element type relative to
// m: its relative rounding error does not depend on the offset, and fp32 l and O have room for 2^kLazyBits many times over.
constexpr float kLazyLimit = 64.f;                             // 2^6

__device__ __forceinline__ void softmax_step(floatx4 (&s)[4], float& m, float& l, floatx4 (&o)[8], elem8 (&pf)[2],
                                             int lim, int g, float scale_log2) {
    if (lim < kBlockN - 1) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (16 * kt + 4 * g + e > lim) s[kt][e] = -INFINITY;
    }
    floatx4 pv[4];
    float rs = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            pv[kt][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][e], scale_log2, -m));   // m = -inf (no reference yet): +inf or NaN, caught below
            rs += pv[kt][e];
        }
    if (__ballot(!(rs <= kLazyLimit)) != 0ull) {               // rare after a row's first blocks; also catches NaN
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[kt][e]);
        mx = wave_max_over_g(mx);
        const float m_new = fmaxf(m, mx * scale_log2);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);  // 0 when there was no reference
        rs = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pv[kt][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][e], scale_log2, -m_use));
                rs += pv[kt][e];
            }
        l *= alpha;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt] *= alpha;
    }
    l += rs;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            pf[cc][e] = static_cast<elem_t>(pv[2 * cc][e]);
            pf[cc][4 + e] = static_cast<elem_t>(pv[2 * cc + 1][e]);
        }
}

// kLong: sequences long enough for in_step.h, its counters and its pacing; a variant of its own, because a workgroup has its CU to itself and pays for all
// set-up (the counting alone took 2.6 % where rows are short: 30000 tokens with a window of 9 blocks 536 -> 550 us)
// kParts: so many workgroups share a group, each with some of its tokens.  All of them choose the blocks walked together from the group's eight rows and bring them
// through their rings; a wavefront of another part's token only helps with that.  A row is added up in the same order for any kParts.
template <bool kCausal, bool kLong, int kParts>
__global__ __launch_bounds__(512)
void stage2_fwd_hybrid_kernel(const FwdParams p, const HybridExtra x) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    uint4* ring = reinterpret_cast<uint4*>(smem_raw);                               // [kRingTiles][2048]: K units 0..1023, V units 1024..2047
    unsigned long long* com = reinterpret_cast<unsigned long long*>(smem_raw + kRingTiles * kTileBytes);   // [mask_words]
    unsigned long long* rows = com + x.mask_words;                                  // [kHybTokens][mask_words]

    // ---- which tokens: in the XCDs' shares, heaviest first (x.late: but the last group of every sequence at the end) ----
    const int bid = blockIdx.x;
    // (few groups are few chunks: two parts to an XCD fill its CUs, the next two go to another)
    const int xcd = (kParts <= 2 ? bid : bid - 16 / kParts * (static_cast<int>(blockIdx.y) >> 1)) & 7, sidx = bid >> 3;
    const int G = place_from_end(x.order, xcd, sidx);
    if (G >= x.total_groups) return;                                                // uniform per workgroup
    int grp, h, b;
    bool there = true;
    if (kParts == 1 && G >= x.total_groups - x.late) {
        grp = x.groups_per_seq - 1;
        const int hb = G - (x.total_groups - x.late);
        b = hb % x.order.batch;
        h = hb / x.order.batch;
    } else {
        there = group_at(x.order, x.total_groups - x.late - 1 - G, grp, h, b);
    }

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int q0 = p.cu_seqlens_q[b];
    const int Sq = p.cu_seqlens_q[b + 1] - q0;
    const int i0 = grp * kHybTokens;
    const int Sk = p.cu_seqlens_k[b + 1] - p.cu_seqlens_k[b];
    const int64_t slot0 = static_cast<int64_t>(h) * p.n_slots + image_slot0(p.cu_seqlens_k, b);
    // (All of these are read before the first atomic: behind it the compiler loads them into vector registers, 0.5 us per workgroup.)
    unsigned* finished = x.finished + xcd * kInStepPitch;
    if (i0 >= Sq || !there) {                                                            // uniform per workgroup
        if (kLong && tid == 0 && x.finished) in_step_finished(finished);
        return;
    }

    // A group at the end of a sequence that has four tokens or fewer: 2, 4 or 8 wavefronts share a token's blocks (every so-manyth column
    // of its mask row each) and merge at the end.  With one wavefront per token such a group took as long as a full one, and where a
    // launch has few groups per CU the last of them decides (2049 queries behind 17962 keys, 514 groups: 254 -> 236 us).
    const int in_group = Sq - i0 < kHybTokens ? Sq - i0 : kHybTokens;
    const int share_log2 = in_group > 4 ? 0 : in_group > 2 ? 1 : in_group > 1 ? 2 : 3;
    const int slots = kHybTokens >> share_log2;                                     // wavefronts of one share
    const int part = wave >> (3 - share_log2);
    const int i = i0 + (wave & (slots - 1));                                        // this wavefront's token
    const bool live = i < Sq;
    const int slots_of_part = slots > kParts ? slots / kParts : 1;
    const bool walks = live && (kParts == 1 || (wave & (slots - 1)) / slots_of_part == static_cast<int>(blockIdx.y));
    if (kParts > 1 && static_cast<int>(blockIdx.y) * slots_of_part >= in_group) return;    // uniform: none of the part's tokens is there
    int last_key = kCausal ? (i + Sk - Sq) : (Sk - 1);                              // largest allowed key index
    if (last_key > Sk - 1) last_key = Sk - 1;
    if (!live) last_key = -1;
    const int last_blk = last_key < 0 ? -1 : (last_key >> 6);
    const int64_t tok = static_cast<int64_t>(q0) + (live ? i : i0);
    const uint64_t* mrow = p.mask ? p.mask + (static_cast<int64_t>(h) * p.total_q + tok) * p.n64 : nullptr;

    // ---- the row words, and which blocks the group walks together ----
    int nw;                                                                          // words that can hold an allowed block of any token
    {
        const int i_last = (i0 + kHybTokens - 1 < Sq) ? i0 + kHybTokens - 1 : Sq - 1;
        int lk = kCausal ? (i_last + Sk - Sq) : (Sk - 1);
        if (lk > Sk - 1) lk = Sk - 1;
        nw = lk < 0 ? 0 : (lk >> 12) + 1;
        if (mrow && nw > p.n64) nw = p.n64;
        if (nw > x.mask_words) nw = x.mask_words;                                    // a sequence longer than the announced max_seqlen_k
    }
    unsigned long long* own = rows + wave * x.mask_words;                           // this token's row
    auto row_word = [&](int w) { return w < nw && last_blk >= 0 && w <= (last_blk >> 6) ? (mrow ? mrow[w] : ~0ull) : 0ull; };
    uint64_t word = row_word(lane);
    // ---- Q operand, on its way while the words are looked at (requested behind them, kernel in us: 2048 tokens 52.3 -> 51.9, 3941 (16 blocks) 104.0 -> 101.2, 6741 in four
    //      sequences 141.5 -> 138.0, 32 768 2809 -> 2794) ----
    elem8 qf[4];
    {
        const int nq = n < p.group ? n : p.group - 1;
        const elem_bits* qp = p.q + tok * p.q_tok_stride + h * p.q_kvh_stride + nq * p.q_grp_stride + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const elem8*>(qp + 32 * c);
    }
    for (int w = lane; w < nw; w += 64) {
        if (w == (last_blk >> 6)) {
            const int tb = last_blk & 63;
            word &= (tb == 63) ? ~0ull : ((1ull << (tb + 1)) - 1ull);
        }
        own[w] = word;
        word = row_word(w + 64);
    }
    __syncthreads();
    for (int w = tid; w < nw; w += 512) com[w] = share_log2 == 0 ? walked_together(rows + w, x.mask_words, in_group) : 0ull;   // shared out: no lock step
    __syncthreads();
    int beside = own_beside(own, com, nw, lane);
    const uint64_t columns = (share_log2 == 0 ? ~0ull : share_log2 == 1 ? 0x5555555555555555ull
                              : share_log2 == 2 ? 0x1111111111111111ull : 0x0101010101010101ull) << part;

    float m = -INFINITY, l = 0.f;
    floatx4 o[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};

    // ---- the walk: one turn = two common blocks (lock step, operands from the LDS ring) alternating with two own
    //      blocks (operands from global memory into registers).  The own blocks' loads keep the vector memory path
    //      busy while the matrix pipeline works on a common block, and the other way round. ----
    const uint4* src_lane = (wave < 4 ? reinterpret_cast<const uint4*>(p.kimg) + slot0 * 1024 + wave * 256
                                      : reinterpret_cast<const uint4*>(p.vimg) + slot0 * 1024 + (wave - 4) * 256) + lane;
    const uint32_t ring_base = __builtin_amdgcn_readfirstlane(lds_address_of(ring) + wave * 4096);
    auto issue = [&](int jj, int tile) { dma_copy_4k(src_lane + static_cast<int64_t>(jj) * 1024, ring_base + tile * kTileBytes); };
    int cw = -1, ow = -1;
    uint64_t cbits = 0ull, crow = 0ull, obits = 0ull, cfilled = 0ull, ofilled = 0ull;
    auto next_common = [&](bool& mine) -> int {
        while (cbits == 0ull) {
            if constexpr (kLong) cw = next_filled_word(cw, nw, cfilled, [&](int w) { return com[w]; });
            else ++cw;
            if (cw >= nw) return -1;
            cbits = uniform_u64(com[cw]);
            crow = uniform_u64(own[cw]);
        }
        const int bit = __builtin_ctzll(cbits);
        mine = (kParts == 1 || walks) && ((crow >> bit) & 1ull);
        cbits &= cbits - 1ull;
        return cw * 64 + bit;
    };
    auto next_own = [&]() -> int {
        while (obits == 0ull) {
            if constexpr (kLong) ow = next_filled_word(ow, nw, ofilled, [&](int w) { return own[w] & ~com[w] & columns; });
            else ++ow;
            if (ow >= nw) return -1;
            obits = uniform_u64(own[ow] & ~com[ow] & columns);
        }
        const int bit = __builtin_ctzll(obits);
        obits &= obits - 1ull;
        return ow * 64 + bit;
    };
    const elem_bits* kimg = p.kimg + slot0 * kImageElems + lane * 8;
    const elem_bits* vimg = p.vimg + slot0 * kImageElems + lane * 8;
    elem8 kreg[16], vreg[16];
    int jp = walks ? next_own() : -1;                           // own block of this turn; its K fragments are loaded a turn ahead
    if (jp >= 0) {
        const elem_bits* src = kimg + static_cast<int64_t>(jp) * kImageElems;
#pragma unroll
        for (int f = 0; f < 16; ++f) kreg[f] = *reinterpret_cast<const elem8*>(src + f * 512);
    }
    // Pacing (in_step.h): steps for own blocks per common block, the steps and own blocks that are left, and the block the walk may reach by now
    // in 1/256.  With these values there is none: own_left and steps_left count down together.
    int steps = 1, steps_left = 0, own_left = 0, front = 0, front_step = 0;
    if constexpr (kLong) {
        int last = i0 + kHybTokens - 1 < Sq ? i0 + kHybTokens - 1 : Sq - 1;    // the group's last key block
        last = (kCausal && last + Sk - Sq < Sk - 1 ? last + Sk - Sq : Sk - 1) >> 6;
        if (last >= kPacedBlocks && jp >= 0) {                 // uniform per wavefront; a row without own blocks has nothing to pace (window of 6 blocks in 60 000 tokens: 427 -> 422 us)
            int count = 0;                                     // blocks walked together << 16 | this row's own
            for (int w = lane; w < nw; w += 64) count += (__builtin_popcountll(com[w]) << 16) + __builtin_popcountll(own[w] & ~com[w]);
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) count += __shfl_xor(count, d);
            count = __builtin_amdgcn_readfirstlane(count);
            if (count >> 16) {
                steps = kPacedSteps;
                steps_left = (count >> 16) * kPacedSteps;
                own_left = count & 0xffff;
                front_step = ((last + 1) << 8) / steps_left;
                front = front_step;
            }
        }
        if (Sk > kInStepKeys && x.finished) {                  // uniform
            int words = 0;                                     // with blocks of this row's own
            for (int w = 0; w < nw; w += 64) words += __builtin_popcountll(__builtin_amdgcn_ballot_w64(w + lane < nw && (own[w + lane] & ~com[w + lane]) != 0ull));
            if (words >= kInStepWords) in_step_wait(finished, sidx);
        }
    }
    // All ordinary loads so far (Q, mask words, first K fragments) land before the first LDS-DMA.  From here on the
    // compiler's wait counts know nothing of the DMA loads; they stay correct because loads complete in order (an
    // unknown younger load only makes a wait stricter), and the waits written by hand below count the ordinary
    // loads that may be younger than the DMA they wait for.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[c]));
#pragma unroll
    for (int f = 0; f < 16; ++f) asm volatile("" : "+v"(kreg[f]));
    // The common blocks go through the ring in pairs: tiles {0, 1} and {2, 3} alternate, the pair after the current
    // one is in flight, and one workgroup barrier serves two blocks.
    bool mine0 = false, mine1 = false;                         // whether this row selects them
    int c0 = next_common(mine0);
    int c1 = c0 >= 0 ? next_common(mine1) : -1;
    if (c0 >= 0) issue(c0, 0);
    if (c1 >= 0) issue(c1, 1);
    int half = 0;
    bool k_ready = jp >= 0;                                    // the coming own block's K fragments are in registers or on their way
    bool k_ahead = false;                                      // ... and were requested after the last DMA
    auto common_part = [&](int j0, int tile) {
        // all 16 fragments of a tile are fetched before the MFMAs that use them (vreg is free between own
        // blocks), and the MFMAs run over independent accumulators first
        const uint4* kb = ring + tile * 2048 + lane;
        const uint4* vb = kb + 1024;
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            const uint4 raw = kb[f * 64];
            __builtin_memcpy(&vreg[f], &raw, 16);
        }
        floatx4 s[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) s[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
                s[kt] = IV2_MFMA(vreg[kt * 4 + c], qf[c], s[kt], 0, 0, 0);
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            const uint4 raw = vb[f * 64];
            __builtin_memcpy(&vreg[f], &raw, 16);
        }
        elem8 pf[2];
        softmax_step(s, m, l, o, pf, (j0 == last_blk) ? last_key - j0 * kBlockN : kBlockN, g, p.scale_log2);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
                o[dt] = IV2_MFMA(vreg[dt * 2 + cc], pf[cc], o[dt], 0, 0, 0);
    };
    auto own_part = [&]() {
        if (!kLong || k_ready) {
            const elem_bits* src = vimg + static_cast<int64_t>(jp) * kImageElems;
#pragma unroll
            for (int f = 0; f < 16; ++f) vreg[f] = *reinterpret_cast<const elem8*>(src + f * 512);
            floatx4 s[4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) s[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
                    s[kt] = IV2_MFMA(kreg[kt * 4 + c], qf[c], s[kt], 0, 0, 0);
            elem8 pf[2];
            softmax_step(s, m, l, o, pf, (jp == last_blk) ? last_key - jp * kBlockN : kBlockN, g, p.scale_log2);
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                for (int dt = 0; dt < 8; ++dt)
                    o[dt] = IV2_MFMA(vreg[dt * 2 + cc], pf[cc], o[dt], 0, 0, 0);
            jp = next_own();
            k_ready = k_ahead = false;
            if constexpr (kLong) --own_left;
        }
        if constexpr (kLong) {
            if (steps_left > 0) front += front_step;           // (no overflow: a walk may go on for long after its last step)
            --steps_left;
        }
        if (jp >= 0 && (!kLong || jp < (front >> 8) || own_left >= steps_left)) {   // K fragments of the next own block
            const elem_bits* src = kimg + static_cast<int64_t>(jp) * kImageElems;
#pragma unroll
            for (int f = 0; f < 16; ++f) kreg[f] = *reinterpret_cast<const elem8*>(src + f * 512);
            k_ready = k_ahead = true;
        }
    };
    // a ring block, and what of its own a row walks beside it
    auto slot = [&](int c, bool mine, int tile) {
        if (mine) common_part(c, tile);
        int blocks = mine ? 0 : 1;
        if (mine && beside > 0) { blocks = 1; --beside; }
        if (kLong && steps == kPacedSteps) blocks = kPacedSteps;
        if constexpr (kLong) {
#pragma unroll 1
            for (; blocks > 0 && jp >= 0; --blocks) own_part();
        } else if (blocks > 0 && jp >= 0) own_part();
    };
    while (c0 >= 0) {                                          // uniform over the workgroup
        // younger than this wavefront's DMA loads of the pair: the 16 K loads of the coming own block
        if (k_ahead) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                       // the pair is in LDS for everyone; the other two tiles are free
        bool next_mine0 = false, next_mine1 = false;
        const int n0 = c1 >= 0 ? next_common(next_mine0) : -1;
        const int n1 = n0 >= 0 ? next_common(next_mine1) : -1;
        if (n0 >= 0) issue(n0, 2 - 2 * half);
        if (n1 >= 0) issue(n1, 3 - 2 * half);
        k_ahead = false;
        slot(c0, mine0, 2 * half);
        if (c1 >= 0) slot(c1, mine1, 2 * half + 1);
        c0 = n0;
        c1 = n1;
        mine0 = next_mine0;
        mine1 = next_mine1;
        half ^= 1;
    }
    while (jp >= 0) own_part();
    if (kLong && tid == 0 && x.finished) in_step_finished(finished);       // the first wavefront for its workgroup: its row is one of eight neighbours
    if (share_log2 != 0) {                                     // uniform per workgroup
        // the ring was not used: 34 floats of every lane, lane by lane
        float* mine = reinterpret_cast<float*>(smem_raw) + wave * (34 * 64) + lane;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[(4 * dt + e) * 64] = o[dt][e];
        mine[32 * 64] = m;
        mine[33 * 64] = l;
        __syncthreads();
        if (part != 0 || !walks) return;
        for (int other = 1; other < (1 << share_log2); ++other) {
            const float* theirs = mine + other * slots * (34 * 64);
            const float m2 = theirs[32 * 64], m_new = fmaxf(m, m2);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;                 // neither has a key
            const float a1 = __builtin_amdgcn_exp2f(m - m_use), a2 = __builtin_amdgcn_exp2f(m2 - m_use);
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[dt][e] = o[dt][e] * a1 + theirs[(4 * dt + e) * 64] * a2;
            l = l * a1 + theirs[33 * 64] * a2;
            m = m_new;
        }
    }
    if (!walks) return;

    // ---- epilogue ----
    const float l_tot = wave_sum_over_g(l);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (n >= p.group) return;                                  // rows that only fill the MFMA tile
    elem_bits* op = p.out + tok * p.o_tok_stride + h * p.o_kvh_stride + n * p.o_grp_stride + 4 * g;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
        uint2 wv;
        wv.x = pack_elem2(o[dt][0] * inv, o[dt][1] * inv);
        wv.y = pack_elem2(o[dt][2] * inv, o[dt][3] * inv);
        *reinterpret_cast<uint2*>(op + 16 * dt) = wv;
    }
    if (g == 0) {
        const float lse = l_tot > 0.f ? m * 0.69314718055994530942f + logf(l_tot) : INFINITY;
        p.lse[h * p.lse_kvh_stride + tok * p.lse_tok_stride + n * p.lse_grp_stride] = lse;
    }
}

static int launch_groups(hipStream_t st, const FwdParams& p, int batch, int num_heads_k, int max_seqlen_q, int max_seqlen_k, bool causal, int most_selected, unsigned* in_step) {
    HybridExtra x{};
    x.groups_per_seq = (max_seqlen_q + kHybTokens - 1) / kHybTokens;
    const int64_t groups = static_cast<int64_t>(num_heads_k) * x.groups_per_seq * batch;
    const int parts = groups * 2 > 256 ? 1 : groups * 4 > 256 ? 2 : groups * 8 > 256 ? 4 : 8;
    x.order = group_order(batch, num_heads_k, x.groups_per_seq, parts > 1);
    const int64_t of_sequence = x.order.per_seq;
    int64_t total = x.order.places();
    const int64_t most = max_workgroups(512) - 8 * kLargestShare;
    if (total > most) {                                        // more than a dispatch holds (thousands of sequences beside a long one): some sequences at a time
        const int fit = static_cast<int>(most / of_sequence);
        IV2_CHECK(fit > 0, "varlen_fwd: too many token groups");
        for (int b = 0; b < batch; b += fit) {
            FwdParams some = p;
            some.cu_seqlens_q += b;
            some.cu_seqlens_k += b;
            some.kimg += static_cast<int64_t>(b) * kImageElems;               // a sequence's first image: image_slot0
            some.vimg += static_cast<int64_t>(b) * kImageElems;
            if (int rc = launch_groups(st, some, batch - b < fit ? batch - b : fit, num_heads_k, max_seqlen_q, max_seqlen_k, causal, most_selected, in_step)) return rc;
        }
        return 0;
    }
    x.mask_words = ((max_seqlen_k + kBlockN - 1) / kBlockN + 63) / 64;
    if (x.mask_words < 1) x.mask_words = 1;
    const size_t lds = kRingTiles * kTileBytes + static_cast<size_t>(1 + kHybTokens) * x.mask_words * 8;
    const bool far = max_seqlen_k > kInStepKeys;
    // As many parts as give every workgroup a CU of its own (256).  A group's turn is bound by what its eight rows fetch through one CU's vector memory path (256 KiB for
    // a block of their own each, 1.6 us) and read from its LDS; its parts have a CU each for that, at the price of a ring each.  Kernel in us, one part ->
    // two: 512 tokens behind 20011 with 2 KV heads and 96 blocks 88 -> 60, 300 behind 60000 with one head 105 -> 67, 1024 of them 104 -> 78; four: 256
    // tokens behind 20011 88 -> 51 (two 60), 256 of 3000 52 -> 41; eight: 64 behind 20011 95 -> 50 (four 54), 8 each of 8 sequences with 9000 keys
    // 101 -> 55 (four 64).  Parts by columns of V, which repeat the products with K: 70 for the four and the eight, 76 for the two.  More workgroups than CUs run in two rounds
    // and gain nothing: 700 tokens behind 20011, 176 groups, take 102 whole.
    // So few groups run all at once: they neither count nor wait (in_step.h).  They keep the pace: it gives the order in which a row's blocks are added up, which must not
    // depend on the number of parts.
    x.finished = parts > 1 ? nullptr : in_step;
    // Heaviest first is also longest prefix first, which puts the one short group of a chunk of queries in front.  Where the chunk's groups are alike, with at least
    // twice as many blocks behind the first of them as a row selects, it holds up a CU that then has as many whole groups to walk as the others, and goes last instead.
    // Forward with the images in us, first | last, 2 KV heads:
    //   2049 queries, 64 blocks: behind 8192 keys 215 | 208, 17 962 234 | 212 (2048 of them 197), 40 960 312 | 238; 32 blocks behind 4096 114 | 114, 12 288 133 | 121;
    //   16 behind 2048 68.6 | 69.0, 10 240 81.2 | 78.0; 4097 queries, 64 blocks, behind 15 914 432 | 391.
    //   Where the groups do not fill whole rounds, 1412 to 3500 queries, the same within 0.6 %.
    //   With fewer blocks behind them last is slower: 64 blocks behind 4096 175 | 187, behind none 332 | 359 (6145 queries).
    const int over = max_seqlen_q % kHybTokens;
    const int64_t held = static_cast<int64_t>(max_seqlen_k) - max_seqlen_q, selected = most_selected < 0 ? -static_cast<int64_t>(most_selected) : most_selected;
    if (parts == 1 && over > 0 && over <= 4 && x.groups_per_seq > 1 && selected > 0 && held >= 2 * kBlockN * selected) {
        x.late = num_heads_k * batch;
        x.order = group_order(batch, num_heads_k, x.groups_per_seq - 1);
        total = x.order.places() + x.late;
    }
    x.total_groups = static_cast<int>(total);
    const int64_t per_round = 8 << x.order.share_log2;
    const int64_t grid = (total + per_round - 1) / per_round * per_round;
    auto pick = [&](auto n) {
        constexpr int kParts = decltype(n)::value;
        return causal ? (far ? stage2_fwd_hybrid_kernel<true, true, kParts> : stage2_fwd_hybrid_kernel<true, false, kParts>)
                      : (far ? stage2_fwd_hybrid_kernel<false, true, kParts> : stage2_fwd_hybrid_kernel<false, false, kParts>);
    };
    auto kernel = parts == 8 ? pick(std::integral_constant<int, 8>{}) : parts == 4 ? pick(std::integral_constant<int, 4>{}) : parts == 2 ? pick(std::integral_constant<int, 2>{}) : pick(std::integral_constant<int, 1>{});
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    IV2_CHECK(e == hipSuccess, "varlen_fwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid), parts), dim3(512), lds, st, p, x);
    IV2_LAUNCH_CHECK();
    return 0;
}

int launch_stage2_fwd_hybrid(hipStream_t st, const FwdParams& p, int batch, int num_heads_k, int max_seqlen_q,
                             int max_seqlen_k, bool causal, int most_selected, unsigned* in_step) {
    IV2_CHECK((max_seqlen_k + kBlockN - 1) / kBlockN <= kMaxMaskWords * 64, "varlen_fwd: more than %d key blocks per sequence", kMaxMaskWords * 64);
    const bool tiles = p.mask == nullptr
        ? dense_tiles_pay(batch, num_heads_k, p.group, p.total_q, p.total_k, max_seqlen_q, max_seqlen_k, causal)
        : masked_by_tiles(most_selected);
    return tiles ? launch_stage2_fwd_tile(st, p, batch, num_heads_k, max_seqlen_q, max_seqlen_k, causal)
                 : launch_groups(st, p, batch, num_heads_k, max_seqlen_q, max_seqlen_k, causal, most_selected, in_step);
}

}  // namespace IV2_NS
