// Mask-row iteration and small cross-lane helpers shared by the Stage-2 kernels.
#pragma once
#include "common.h"

namespace IV2_NS {

// Walks the set bits of one mask row in ascending block order, clipped to [0, last_blk].
struct BlockWalker {
    const uint64_t* row;
    int n_words;                    // words that can hold an allowed block
    int last_blk;
    int w;
    uint64_t bits;

    __device__ __forceinline__ uint64_t load_word(int word) const {
        uint64_t v = row ? row[word] : ~0ull;
        if (word == (last_blk >> 6)) {
            const int t = last_blk & 63;
            v &= (t == 63) ? ~0ull : ((1ull << (t + 1)) - 1ull);
        }
        // the row is shared by the whole wavefront: keep the loop control in scalar registers
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
        return (static_cast<uint64_t>(hi) << 32) | lo;
    }
    __device__ __forceinline__ void init(const uint64_t* r, int words_in_row, int last) {
        row = r;
        last_blk = last;
        n_words = last < 0 ? 0 : (last >> 6) + 1;
        if (row && n_words > words_in_row) n_words = words_in_row;
        w = 0;
        bits = n_words > 0 ? load_word(0) : 0ull;
    }
    __device__ __forceinline__ int next() {
        while (bits == 0ull) {
            if (++w >= n_words) return -1;
            bits = load_word(w);
        }
        const int bit = __builtin_ctzll(bits);
        bits &= bits - 1ull;
        return w * 64 + bit;
    }
};

// The word after `at` (at first -1) that is not zero, for a walk over words in LDS, or `words`; `filled` (at first 0) is the walk's.  For long rows: words without
// blocks are passed over 64 at a time.  One by one, a trip to LDS each, they took 0.03 us a word of a group's set-up (window of 6 blocks in 60 000 tokens, 15 words: 422 -> 410 us).
template <typename Word>
__device__ __forceinline__ int next_filled_word(int at, int words, uint64_t& filled, Word word) {
    int from = at & ~63;
    while (filled == 0ull) {
        from += 64;
        if (from >= words) return words;
        const int w = from + static_cast<int>(__lane_id());
        filled = __builtin_amdgcn_ballot_w64(w < words && word(w) != 0ull);
    }
    const int w = from + __builtin_ctzll(filled);
    filled &= filled - 1ull;
    return w;
}

// A word of the mask rows of a group of up to eight tokens, `pitch` words apart: the blocks that the group walks together, which is those that five or
// more of eight rows select, or all rows of a smaller group.  The row-parallel kernels say what that measured.  Rows that are all alike, as under a window or without a
// mask, have nothing from it and are found first: the count is 50 vector instructions of one wavefront for which the others wait.  Forward in us, blocks of all eight
// rows | counted | counted where rows differ: 30 000 tokens, 2 KV heads, groups of 8, 34 blocks 1110 | 1126 | 1109; 2000, 33 blocks 60.7 | 61.5 | 60.7; 30 x 600,
// 7 blocks 197.4 | 196.5 | 194.3; without a mask 3800, one KV head 83.9 | 85.2 | 84.1.
__device__ __forceinline__ uint64_t walked_together(const unsigned long long* words, int pitch, int tokens) {
    if (tokens < 8) {
        uint64_t all = words[0];
        for (int t = 1; t < tokens; ++t) all &= words[t * pitch];
        return all;
    }
    // how many of the rows select a block, a binary digit to a word
    uint64_t r[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) r[t] = words[t * pitch];
    const uint64_t all = r[0] & r[1] & r[2] & r[3] & r[4] & r[5] & r[6] & r[7], any = r[0] | r[1] | r[2] | r[3] | r[4] | r[5] | r[6] | r[7];
    if (__builtin_amdgcn_ballot_w64(all != any) == 0ull) return all;
    auto sum3 = [](uint64_t a, uint64_t b, uint64_t c, uint64_t& carry) { carry = (a & b) | (c & (a | b)); return a ^ b ^ c; };
    uint64_t t0, t1, t2, f0;
    const uint64_t s0 = sum3(r[0], r[1], r[2], t0), s1 = sum3(r[3], r[4], r[5], t1), s2 = sum3(r[6], r[7], s0, t2);
    const uint64_t ones = s1 ^ s2, t3 = s1 & s2, u = sum3(t0, t1, t2, f0), twos = u ^ t3, f1 = u & t3, fours = f0 ^ f1, eights = f0 & f1;
    return eights | (fours & (twos | ones));
}

// How many of the ring's blocks that a row selects have one of its own walked beside them (beside those it does not select there always is one).
// A row that has its own blocks beside every ring block until they run out waits, from then on, at ring blocks that are not its own; with so many fewer beside the
// others it has one for each of those.  That is its blocks less the ring's: negative, none, with few blocks to choose from.  Rows with more than kOwnBeside over take
// one every time: their own blocks outnumber the ring's that are not theirs.  A rule on the group's rows alone, which gives the order in which they are added up.
//   all balanced: four packed sequences (71 552 tokens), forward and dQ, 5625 | 7320 -> 5740 | 7450 us
//   whole passes, every time -> balanced: 2048 tokens with 16 blocks 65.0 -> 63.5, four ragged prompts 931 -> 922, training on four short samples 588 -> 585;
//   32 768 tokens and chunks as before
//   two over instead of kOwnBeside: forward of 9934 + 3083 tokens, 32 blocks, 591 -> 599, of 11 878 + 8202, 64 blocks, 706 -> 711, of 49 other inputs within 1 % on average
//   two beside a ring block that is not the row's, too, as long as there are enough: 64.1, 942, 584, and 32 768 tokens 3164 -> 3212
constexpr int kOwnBeside = 8;
__device__ __forceinline__ int own_beside(const unsigned long long* row, const unsigned long long* together, int words, int lane) {
    int over = 0;
    for (int w = lane; w < words; w += 64) over += __builtin_popcountll(row[w]) - __builtin_popcountll(together[w]);
    over = __builtin_amdgcn_readlane(scan_lanes(over), 63);
    return over > kOwnBeside ? 1 << 30 : over;
}

// Cross-row exchanges with gfx950's v_permlane16_swap / v_permlane32_swap (VALU speed; a ds_bpermute takes a trip
// through the LDS crossbar): swapping a register with itself hands every lane its own row's value and the partner
// row's value.
__device__ __forceinline__ void row_pair_xor16(float x, float& mine, float& other) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    mine = __uint_as_float(r[0]);
    other = __uint_as_float(r[1]);
}
__device__ __forceinline__ void row_pair_xor32(float x, float& mine, float& other) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    mine = __uint_as_float(r[0]);
    other = __uint_as_float(r[1]);
}
// reductions over the four 16-lane groups g of a wavefront (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float wave_max_over_g(float x) {
    float a, b;
    row_pair_xor16(x, a, b);
    x = fmaxf(a, b);
    row_pair_xor32(x, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float wave_sum_over_g(float x) {
    float a, b;
    row_pair_xor16(x, a, b);
    x = a + b;
    row_pair_xor32(x, a, b);
    return a + b;
}

}  // namespace IV2_NS
