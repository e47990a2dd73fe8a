// Tiles of 256 query rows that walk the key blocks any of their tokens selected: what the forward and the dQ kernel share.
#pragma once
#include "common.h"
#include "block_walker.h"
#include <math.h>

namespace IV2_NS {

constexpr int kTileWaves = 4;
constexpr int kTileRows = 64 * kTileWaves;                     // query rows of a workgroup, 64 per wavefront in two halves
constexpr int kSlotBytes = 2 * kBlockN * kHeadDim * 2;         // of an LDS ring: K image | V image of a block
constexpr int kMostTokens = 8;                                 // of a wavefront: groups of 8

// A token takes 16 rows, 8 in groups of 8.
inline int tile_row_shift(int group) { return group == 8 ? 3 : 4; }
inline int tiles_per_sequence(int group, int max_seqlen_q) {
    const int tokens = kTileRows >> tile_row_shift(group);
    return (max_seqlen_q + tokens - 1) / tokens;
}

struct TileExtra {
    int tiles_per_seq;                                         // ceil(max_seqlen_q / tokens of a tile)
    int batch;
    int heads_k;
    int sequences;                                             // heads_k * batch
    int max_blocks;                                            // what the images hold of a sequence
    int row_shift;                                             // log2 of the MFMA rows a token takes: 3 for groups of 8, else 4
};

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
#ifdef IV2_F16
#define IV2_MFMA32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0)
#else
#define IV2_MFMA32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)
#endif

// the two lanes of a row
__device__ __forceinline__ float half_max(float x) {
    float a, b;
    row_pair_xor32(x, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float half_sum(float x) {
    float a, b;
    row_pair_xor32(x, a, b);
    return a + b;
}

// The key blocks of a tile in ascending order: those that any of its tokens selected (all of them without a mask) and that do not begin behind that token's
// last key.  A tile that straddles the beginning of a block walks it for the tokens behind; those before it must not count as having selected it, whatever their
// mask says, or what the block holds would reach them as 0 x inf.  Everything here is uniform over the wavefront; the blocks are the same in all
// wavefronts of a workgroup.
constexpr int kTokenBits = 20;
__device__ __forceinline__ uint64_t lowest_bits(int n) { return n >= 64 ? ~0ull : n <= 0 ? 0ull : (1ull << n) - 1ull; }
template <bool kCausal>
struct TileWalk {
    const uint64_t* rows;           // mask row of the tile's first token, or null
    int n64, tokens;                // words of a row; tokens of the tile that exist
    int mine;                       // first token of this wavefront inside the tile
    int per_wave;
    int last_key;                   // of the tile's first token (negative: it has none); causal: the next ones see a key more each
    int blocks;                     // blocks at or behind this one are not walked
    int w;
    uint64_t bits;                  // of word w: what is left of the union
    int chosen;                     // lane b: which of this wavefront's tokens selected block b of word w, a bit each

    __device__ __forceinline__ int seen(int t) const { return ((last_key + (kCausal ? t : 0)) >> 6) + 1; }     // blocks of the tile's token t
    __device__ __forceinline__ void load() {
        const int left = blocks - w * 64, lane = __lane_id();
        if (rows == nullptr) {
            bits = ~0ull;
            const int live = tokens - mine < per_wave ? tokens - mine : per_wave;
            chosen = live > 0 ? (1 << live) - 1 : 0;
            const int blind = (w * 64 + lane) * kBlockN - last_key - (kCausal ? mine : 0);       // this wavefront's tokens that end before the block
            if (blind > 0) chosen &= kCausal && blind < kMostTokens ? ~0 << blind : 0;
        } else {
            // lane t holds the word of the tile's token t
            uint32_t lo = 0u, hi = 0u;
            if (lane < tokens) {
                const uint64_t row = rows[static_cast<int64_t>(lane) * n64 + w] & lowest_bits(seen(lane) - w * 64);
                lo = static_cast<uint32_t>(row);
                hi = static_cast<uint32_t>(row >> 32);
            }
            chosen = 0;
#pragma unroll
            for (int t = 0; t < kMostTokens; ++t) {
                const int from = mine + t < 64 ? mine + t : 63;
                const uint32_t a = __builtin_amdgcn_readlane(lo, from), b = __builtin_amdgcn_readlane(hi, from);
                if (t < per_wave) chosen |= static_cast<int>(((lane < 32 ? a : b) >> (lane & 31)) & 1u) << t;
            }
#pragma unroll
            for (int hop = 16; hop > 0; hop >>= 1) {           // a tile has at most 32 tokens
                lo |= __shfl_xor(lo, hop);
                hi |= __shfl_xor(hi, hop);
            }
            bits = static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(hi))) << 32 | static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(lo));
        }
        bits &= lowest_bits(left);
    }
    __device__ __forceinline__ void init() {
        if (rows != nullptr && blocks > n64 * 64) blocks = n64 * 64;
        w = 0;
        bits = 0ull;
        chosen = 0;
        if (blocks > 0) load();
    }
    // Behind an empty word: to the last one before the next that any token has blocks in.  Eight words to a round of loads; one at a time, a window at the end of
    // 110000 tokens cost 11 us per tile, a microsecond each.
    __device__ __forceinline__ void skip() {
        const int last = (blocks - 1) >> 6, lane = __lane_id(), t = lane & 31;
        while (w < last) {
            uint64_t words = 0ull;                             // bit i: word w + 1 + i
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int at = w + 1 + 2 * u + (lane >> 5);
                const uint64_t filled = __builtin_amdgcn_ballot_w64(t < tokens && at <= last && rows[static_cast<int64_t>(t) * n64 + at] != 0ull);
                words |= static_cast<uint64_t>((filled & 0xffffffffull) != 0ull) << (2 * u) | static_cast<uint64_t>((filled >> 32) != 0ull) << (2 * u + 1);
            }
            if (words != 0ull) {
                w += __builtin_ctzll(words);
                return;
            }
            w = w + 8 < last ? w + 8 : last;
        }
    }
    // the next block and, from kTokenBits up, which of this wavefront's tokens selected it; or -1
    __device__ __forceinline__ int next() {
        while (bits == 0ull) {
            if ((w + 1) * 64 >= blocks) return -1;
            ++w;
            load();
            if (bits == 0ull && rows != nullptr) skip();
        }
        const int bit = __builtin_ctzll(bits);
        bits &= bits - 1ull;
        return w * 64 + bit | __builtin_amdgcn_readlane(chosen, bit) << kTokenBits;
    }
    __device__ __forceinline__ static int index(int block) { return block & ((1 << kTokenBits) - 1); }
};

// Time of a launch whose workgroups take `tokens` tokens each, one workgroup per CU at a time, where a workgroup whose last token sees b key blocks
// takes cost(b), in microseconds but for what all launches share: as long as the longest walk, or as the work of all on 256 CUs with a last round
// that is `partial` of one more; workgroups behind the end of a sequence, which return at once, 1.7 ns each.  The host knows the longest sequence
// and the totals: the others are taken to be of equal length.
template <typename Cost>
static double walk_time(int tokens, Cost cost, double partial, int batch, int num_heads_k, int64_t total_q, int64_t total_k, int max_seqlen_q,
                        int max_seqlen_k, bool causal) {
    auto mean = [&](double q, double k) {                      // over the workgroups of a sequence
        const double first = causal ? (k > q ? k - q : 0.) : k;
        if (q <= tokens) return cost(ceil(k / kBlockN));
        double sum = 0.;
        for (int i = 0; i < 16; ++i) sum += cost((first + (k - first) * (i + 0.5) / 16) / kBlockN + 0.5);
        return sum / 16;
    };
    const int others = batch - 1;
    const double q = others > 0 && total_q > max_seqlen_q ? static_cast<double>(total_q - max_seqlen_q) / others : 0.;
    const double k = others > 0 && total_k > max_seqlen_k ? static_cast<double>(total_k - max_seqlen_k) / others : 0.;
    const double of_longest = ceil(static_cast<double>(max_seqlen_q) / tokens), of_others = others * ceil(q / tokens);
    const double rounds = num_heads_k * (of_longest + of_others) / 256.;
    const double each = (of_longest * mean(max_seqlen_q, max_seqlen_k) + (of_others > 0. ? of_others * mean(q, k) : 0.)) / (of_longest + of_others);
    const double chain = cost(ceil(static_cast<double>(max_seqlen_k) / kBlockN));
    const double all = each * (rounds + (rounds > 1. ? partial : 0.));
    return (chain > all ? chain : all) + 0.0017 * num_heads_k * batch * of_longest;
}

}  // namespace IV2_NS
