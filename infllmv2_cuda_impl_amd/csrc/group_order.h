// The order of the token groups of a launch of the row-parallel kernels, and which XCD takes which.
#pragma once
#include <cstdint>

namespace IV2_NS {

// The kernels take the groups from the end of the order.  One (head, sequence) after the other, its longest prefixes first; or, in launches of up to kGroupsByTurns
// groups, one sequence after the other and in it a chunk of groups of a head, the same ones of the next head, and so on, so that the longest prefixes of all heads
// come first and the shortest last.  Head by head the second head's longest groups were begun half-way.
//
// Workgroups go round the 8 XCDs, each of which runs 32 at once; an XCD takes a share of consecutive places, its neighbour the next.  Small shares come out
// even, in ragged batches too, where the places behind a short sequence are nobody's; large ones keep neighbours, whose windows overlap, in one L2.  Shares of 4 up to kGroupsInFour
// groups, of 8 up to kGroupsByTurns, of 16 beyond and where all groups run at once.  With shares of 4 a chunk is as long as makes an XCD meet the same
// head every time (four heads, 2100 tokens 97.9 -> 96.1 us).
//
// A head's last chunk is as long as its groups in short sequences; else it is rounded up, with shares of 4 to a share, beyond to a chunk, for what lies behind it to begin
// with one (16 001 tokens, two heads, 2001 groups: as they come 1417 us, rounded 1300; training on 2500 + 700 + 2900, 16 blocks, shares of 8, to a share 565, to a chunk 552), but not if that
// gives a CU a second group (rounded up to 16, 656 queries each behind three prompts, one head, 246 groups: 152 us instead of 96).  In short sequences it would be a large part of
// them, and of the same XCDs (16 blocks, one head, rounded up to 16 | this: 128 sequences of 136 tokens 99 | 61, 20 of 900 175 | 118).
//
// Forward in us: head by head in shares of 16 | by turns, chunks and shares of 16, chunks rounded up | this.  KV heads, blocks selected:
//   1160 tokens, 4, 64                          47.3 | 41.4 | 43.0        487 + 1295 + 909, 1, 32                    39.1 | 40.0 | 29.6
//   2100, 4, 64                                  116 |   95 |   96        440 + 254 + 846 + 634 + 354, 1, 16         21.7 | 24.0 | 22.0
//   2185, 2, 64                                 69.0 | 62.5 | 59.6        1739 + 1117 + 1273 + 1022 + 2282, 2, 16     140 |  144 |  133
//   3849, 1, 64                                 83.8 | 82.6 |   72        984 + 3512 + 3164, 2, 64                    251 |  227 |  231
//   8192, 2, 64                                  514 |  495 |  487        1839 + 584 + 1225, 2, 32                   82.9 | 68.9 | 73.2
//   8191, 4, 64                                 1009 |  960 |  959        1288 + 1099 + 1098, 4 of 8 heads, 32        104 |  100 |  104
//   1024, 4, 64                                 47.4 | 34.5 | 32.4        2048, 2, 64                                 59.7 | 52.7 | 46.1
//   1038, 4, 64 (520 groups: a third round)     46.8 | 35.4 | 38.3        2100, 2, 64 (526)                           60.0 | 52.5 | 55.2
//   701 queries behind three prompts, 1, 16     65.4 | 73.9 | 75.1        2435 + 1905, 4, 32                          192 |  203 |  196
// Shares of 4 beyond kGroupsInFour cost L2 hits: 8191 tokens, 4, 16 420 | 441 with them, training on 1023 + 3001 + 517 + 2200, 2, 16, forward 151 | 156.
// Shares of 16 there instead of 8: that training pass 564 us instead of 570, on 1739 + 1117 + 1273 + 1022 + 2282 606 instead of 579, on 2435 + 1905, 4, 32 897 instead of 885.
struct GroupOrder {
    int batch, heads, groups;                                  // groups: of the longest sequence and a head
    int chunk_log2;                                            // by turns, groups of a head in a row; < 0: head by head
    int share_log2;                                            // places in a row that are one XCD's
    int rest;                                                  // by turns, places of a head in its last chunk, where that is not a whole one
    int64_t per_seq;                                           // places of a sequence
    int64_t places() const { return batch * per_seq; }
};
constexpr int64_t kGroupsByTurns = 4096, kGroupsInFour = 2048, kGroupsAtOnce = 256;
constexpr int kLargestShare = 16;
constexpr int kShortSequence = 256;                            // groups; shorter ones are not rounded up
// in_parts: so few groups that several workgroups take one; the kernel spreads them over the XCDs in shares of 16
inline GroupOrder group_order(int batch, int heads, int groups, bool in_parts = false) {
    const int64_t all = static_cast<int64_t>(batch) * heads * groups;
    if (in_parts || all > kGroupsByTurns) return {batch, heads, groups, -1, 4, 0, static_cast<int64_t>(heads) * groups};
    const bool at_once = all <= kGroupsAtOnce;
    const int share = at_once ? 4 : all <= kGroupsInFour ? 2 : 3, most = share != 2 || heads <= 2 ? 4 : heads <= 4 ? 3 : 2;
    int log2 = 0;
    while (log2 < most && (1 << log2) < groups) ++log2;
    const int whole = (groups >> log2) << log2;
    int round = !at_once && groups < kShortSequence ? 1 : share == 2 ? 4 : 1 << log2;
    if (at_once && static_cast<int64_t>(batch) * heads * ((groups + round - 1) / round * round) > kGroupsAtOnce) round = 1;
    const int rest = (groups - whole + round - 1) / round * round;
    return {batch, heads, groups, log2, share, rest, static_cast<int64_t>(heads) * (whole + rest)};
}
// The place, counted from the end, of an XCD's turn-th workgroup.
__device__ __forceinline__ int place_from_end(const GroupOrder& o, int xcd, int turn) {
    const int within = turn & ((1 << o.share_log2) - 1);
    return ((((turn >> o.share_log2) << 3) + xcd) << o.share_log2) + within;
}
// The group at a place; false: nobody's.
__device__ __forceinline__ bool group_at(const GroupOrder& o, int at, int& grp, int& h, int& b) {
    if (o.chunk_log2 < 0) {                                    // uniform
        const int hb = at / o.groups;
        grp = at - hb * o.groups;
        h = hb / o.batch;
        b = hb - h * o.batch;
        return true;
    }
    b = 0;
    if (o.batch > 1) {
        const int per_seq = static_cast<int>(o.per_seq);
        b = at / per_seq;
        at -= b * per_seq;
    }
    const int whole = (o.groups >> o.chunk_log2) << o.chunk_log2;
    if (at < whole * o.heads) {
        const int chunk = at >> o.chunk_log2, level = chunk / o.heads;
        h = chunk - level * o.heads;
        grp = (level << o.chunk_log2) + (at & ((1 << o.chunk_log2) - 1));
        return true;
    }
    at -= whole * o.heads;
    h = at / o.rest;
    grp = whole + at - h * o.rest;
    return grp < o.groups;
}

}  // namespace IV2_NS
