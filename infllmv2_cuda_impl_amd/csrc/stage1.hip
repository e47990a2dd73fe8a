// Stage-1 scoring for gfx950: softmax-like scores of the 16 grouped query heads against the
// compressed keys, normalised by a log-sum-exp taken over a (usually coarser) second key set,
// summed over the 16 heads.
//
// Semantics follow compute_attn_1rowblock_splitkv_stage1
// (csrc/flash_attn/src/flash_fwd_kernel.h:1203-1744), Mask::apply_mask_stage1
// (csrc/flash_attn/src/mask.h:225-319), softmax_rescale_simple / softmax_rescale_gt
// (csrc/flash_attn/src/softmax.h:94-121,198-237) and hdim16_reduce (flash_fwd_kernel.h:53-112):
//   vis_s(i) = min(L, max(0, (i+1)/s - 1 + L - (Sq - s + 1)/s))     (C++ truncating divisions)
//   lse_g(i) = log sum_{c < vis_c(i)} exp(scale * q_g . kc_c),  s = 64, or 16 when Lc == Lk
//   score[h, i, j] = bf16( sum_g exp(scale * q_g . kf_j - lse_g(i)) )   for j < vis_16(i), else 0
//   rows with vis_c(i) == 0 are all zero (the reference's early exit leaves its zero fill).
//
// Design: S = Q.K^T with the 16 heads of one token as the 16 MFMA rows and 16 compressed keys as
// the columns, so a lane owns four heads of one key column; the per-head running max/sum of
// pass 1 stay lane-local until one 16-lane butterfly at the end, and the sum over the 16 heads
// in pass 2 is an in-lane add of four values plus two cross-lane adds.  A workgroup is 8
// wavefronts x 2 consecutive tokens; each 64-key tile of compressed keys is staged once in LDS
// (LDS-DMA, straight into MFMA-operand order, read back with conflict-free ds_read_b128) and reused
// by all 16 tokens, and inside a wavefront one operand read feeds two MFMAs.
//
// Bound by vector instructions (the vector pipe was 80 % busy, the matrix pipe 42 %) and by power: what is saved in instructions is half lost to a lower
// clock.  Tiles without a test, offsets in scalar registers, DPP maxima spelled out and results stored a tile later took them from 202 to 184 per 64
// fine keys, 16 coarse ones and two tokens (counted, beside 40 MFMAs); pooled, two KV heads, us: 131 072 tokens 5800 -> 5580, 32 768 428 -> 415, 9173 62 -> 60; 2049 queries against 20 011
// keys 60.3 -> 58.5.  Launches of one or two tiles pay 0.1 to 0.25 us for the set-up (500 tokens, scores 7.9 -> 8.0, pooled 8.2 -> 8.45).
// With 32-row MFMAs and plain sums in pass 1: 5470, 407, 59, 54, but sums in another order round some scores to the neighbouring 16-bit value, and
// single rows then attend another block.
#include "common.h"
#include "block_walker.h"
#include "infllmv2_hip.h"
#include <math.h>
#include <type_traits>

namespace IV2_NS {

struct Stage1Params {
    const elem_bits* q;
    const elem_bits* k;              // fine compressed keys   (sum Lk, Hk, d)
    const elem_bits* c;              // coarse compressed keys (sum Lc, Hk, d)
    elem_bits* score;                // (Hk, total_q, row_stride); pooled output: (Hk, total_q, pool_len), dense
    const int* cu_seqlens_q;
    const int* cu_seqlens_k;
    const int* cu_seqlens_c;
    int64_t q_tok_stride, q_grp_stride, q_kvh_stride;
    int64_t k_row_stride, k_head_stride, c_row_stride, c_head_stride;
    int64_t score_head_stride, score_row_stride;
    int score_cols;                  // columns to define in every row (max_seqlen_k)
    float scale_log2;
    int causal;
    int splits;                      // workgroups that share a block of tokens, each with a run of its fine tiles
    int group;                       // query heads per KV head, 1..16: MFMA rows >= group repeat head group - 1 and add nothing
    // pooled output only
    const int* cache_lens;           // per sequence, or null: cache_len for all
    int cache_len;
    int pool_len;                    // key blocks per output row
    int local_blocks, init_blocks;
    // selection only
    uint64_t* mask;                  // (Hk, total_q, mask_words)
    int64_t total_q;
    int mask_words, topk;
};

// 8 wavefronts x 2 tokens: 112 registers, so four wavefronts share a SIMD and the exp-heavy VALU work of one hides
// behind the MFMAs of another (4 x 4 at two wavefronts per SIMD measures 6 % slower, 8 x 1 2 to 10 % slower where the launch fills the chip; where it does not: launch_stage1)
constexpr int kTokPerWave = 2;
constexpr int kWavesS1 = 8;
constexpr int kWavesPerSimdS1 = 4;
constexpr int kTokPerBlock = kTokPerWave * kWavesS1;   // 16
// 8 x 1 takes 60 registers: eight wavefronts to a SIMD, four workgroups to a CU, or three where LDS ends it (512 blocks of 16 tokens pooled).  Held to four wavefronts
// like 8 x 2, a third workgroup waited for one of the first two: scores of 2048 | 2049 queries against 20 011 keys 36.2 | 49.3 us, now 36.4 | 42.2.
constexpr int waves_per_simd(int tok, int items, int pack) { return tok > 1 ? kWavesPerSimdS1 : items * pack >= 16 ? 6 : 8; }
constexpr int kKeysPerBlock = 4;                       // compressed keys (stride 16) per 64-token key block

__device__ __forceinline__ int trunc_div(int a, int b) { return a / b; }   // C++ semantics on purpose

__device__ __forceinline__ int stage1_visible(int i, int s, int L, int Sq, bool causal) {
    if (!causal) return L;
    const int cq = trunc_div(Sq - s + 1, s);
    int v = (i + 1) / s - 1 + L - cq;
    v = v < 0 ? 0 : v;
    return v < L ? v : L;
}

// A (64 keys x 128 d) tile goes from global memory to LDS by LDS-DMA, in MFMA-operand order: 16-byte unit
// u = (kt*4 + c)*64 + 16*g + n holds K[16*kt + n][32*c + 8*g ..].  Wavefront w of the workgroup moves the 64-unit groups
// grp = w, w + 8 (key tile grp / 4, chunk grp % 4 of its 16 keys): lane l's unit lands at lds_base + 16 l, which is exactly operand order, so the operand reads are linear and free of bank conflicts.
// A lane's offset inside a tile is the same in every whole tile (first_off) and the tile's own goes into the scalar base: no vector instruction.
// Keys beyond the last one are read from the last row (finite values that every consumer masks).
// The compiler's wait counts do not see these loads: the code waits for them by hand before the barrier that
// publishes the tile.
__device__ __forceinline__ uint32_t s1_lds_addr(const void* ptr) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)ptr));
}
__device__ __forceinline__ void s1_dma16(const void* base, uint32_t lane_off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
                 : : "v"(lane_off), "s"(base), "s"(lds_base) : "memory", "m0");
}
__device__ __forceinline__ uint32_t s1_first_off(int row_stride, int wave, int n, int g) {
    return static_cast<uint32_t>((16 * (wave >> 2) + n) * row_stride + 32 * (wave & 3) + 8 * g) * 2u;
}
__device__ __forceinline__ void issue_tile(const elem_bits* base, int row_stride, uint32_t first_off, int key0, int L, uint32_t lds_tile,
                                           int wave, int n, int g) {
    static_assert(kWavesS1 == 8, "first_off: two groups of a wavefront are 32 keys apart");
    if (key0 + 64 <= L) {                                      // uniform
        const elem_bits* tile_base = base + static_cast<int64_t>(key0) * row_stride;
        s1_dma16(tile_base, first_off, lds_tile + wave * 1024);
        s1_dma16(tile_base + 32 * static_cast<int64_t>(row_stride), first_off, lds_tile + (wave + 8) * 1024);
        return;
    }
#pragma unroll
    for (int it = 0; it < 16 / kWavesS1; ++it) {
        const int grp = it * kWavesS1 + wave;                  // (kt, c) = (grp / 4, grp % 4)
        int row = key0 + 16 * (grp >> 2) + n;
        row = row < L ? row : L - 1;
        const uint32_t off = static_cast<uint32_t>(row * row_stride + 32 * (grp & 3) + 8 * g) * 2u;
        s1_dma16(base, off, lds_tile + grp * 1024);
    }
}

// x, y -> (x's even 16-lane rows interleaved with y's even rows, x's odd rows interleaved with y's odd rows), summed:
// row 2r of the result is x.row(2r) + x.row(2r+1), row 2r+1 is y.row(2r) + y.row(2r+1).
__device__ __forceinline__ float fold_rows16(float x, float y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// rows 0,1 of the result are x.row(r) + x.row(r+2), rows 2,3 are y.row(r-2) + y.row(r)
__device__ __forceinline__ float fold_rows32(float x, float y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// the lower halves of x and y, and the upper halves
__device__ __forceinline__ void halves(float x, float y, float& lower, float& upper) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    lower = __uint_as_float(r[0]);
    upper = __uint_as_float(r[1]);
}
// value of lane (n + k) % 16 of the same 16-lane row (DPP row_ror:k)
template <int kRot>
__device__ __forceinline__ float dpp_row_ror(float x) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x120 + kRot, 0xF, 0xF, false));
}
// maximum / sum over the 16 lanes of a row, left in every lane: rotations by 8, 4, 2, 1 each double the covered set
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, dpp_row_ror<8>(x));
    x = fmaxf(x, dpp_row_ror<4>(x));
    x = fmaxf(x, dpp_row_ror<2>(x));
    return fmaxf(x, dpp_row_ror<1>(x));
}
__device__ __forceinline__ float row16_sum(float x) {
    x += dpp_row_ror<8>(x);
    x += dpp_row_ror<4>(x);
    x += dpp_row_ror<2>(x);
    return x + dpp_row_ror<1>(x);
}
// Of every quad's first lane: the maximum of the quad and of the lane before it, for two registers at a time; lane 0's lane before is prev's lane 63.
// Spelled out because the compiler makes three instructions (a move, a canonicalisation, a maximum) of what one can do.  A
// lane read by DPP must have been written three instructions before; the registers are each other's distance.
__device__ __forceinline__ void pool_quads(float a, float b, float prev_a, float prev_b, float& best_a, float& best_b) {
    float x, y;
    asm volatile("s_nop 1\n\t"
                 "v_max_f32_dpp %0, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f32_dpp %1, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 0\n\t"
                 "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f32_dpp %0, %2, %0 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f32_dpp %1, %3, %1 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f32_dpp %0, %4, %0 wave_ror:1 row_mask:0x1 bank_mask:0x1\n\t"
                 "v_max_f32_dpp %1, %5, %1 wave_ror:1 row_mask:0x1 bank_mask:0x1"
                 : "=&v"(x), "=&v"(y) : "v"(a), "v"(b), "v"(prev_a), "v"(prev_b));
    best_a = x;
    best_b = y;
}

// kPool: instead of the score rows, write their 1-D max-pooling onto 64-token key blocks (window of 5 compressed
// keys, stride 4, padding 1, forced blocks +inf, empty windows -inf: the rule of csrc/max_pooling_1d.cuh:12-160
// applied to the scores this kernel would have written, which never reach memory).
// kItems > 0: nor do these; of a row of at most 64 kItems blocks the topk best (larger score first, ties by ascending block: topk.hip) are chosen here, and their
// mask words written.  A wavefront has its tokens' rows in LDS by the end, 64 kItems scores each, and finds the last key that is in bit by bit.
// Bound by the counts, 16 kItems of them to a token, in scalar instructions beside the other wavefronts' exponentials; scores and selection in us, two launches | one, 2 KV heads:
// 2048 tokens 15.9 | 11.9, 4096 27.3 | 21.2, 8192 56.2 | 48.5, 16 384 133 | 125, 20 480 201 | 196, 32 768 443 | 443, 49 152 931 | 944: rows of 512 blocks and no more.  Whole prefill of
// 1000 tokens, 16 blocks selected, 42.0 -> 40.7, of 2048 74.4 -> 70.0, training on 1023 + 3001 + 517 + 2200 606 -> 596.
// kShared: workgroups share a block of tokens (launch_stage1); a variant of its own, because the others paid 0.5 us for the possibility.
// kTok: tiles of 16 rows of a wavefront, a token each: 2 or, in launches of few workgroups (launch_stage1), 1.  kPack == 2: two tokens to a tile, heads 0 to 7 of
// its rows 0 to 7 and 8 to 15.  The head sums then end where the two halves of the rows would have been added.  A token's row is the same bits in every form.
template <bool kCausal, bool kPool, int kItems = 0, bool kShared = false, int kTok = kTokPerWave, int kPack = 1>
__global__ __launch_bounds__(64 * kWavesS1) __attribute__((amdgpu_waves_per_eu(waves_per_simd(kTok, kItems, kPack), kTok == 1 ? 8 : kWavesPerSimdS1)))
void stage1_kernel(const Stage1Params p) {
    constexpr int kMine = kTok * kPack, kTokens = kMine * kWavesS1;                 // tokens of a wavefront and of the workgroup
    __shared__ uint4 tile[2][1024];                            // two 16 KiB operand-ordered key tiles
    __shared__ elem_bits pooled[kItems > 0 ? kTokens : 1][kItems > 0 ? 64 * kItems : 1];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);     // wavefront-uniform: what depends on it alone stays in scalar registers
    const int n = lane & 15, g = lane >> 4;
    const int b = blockIdx.y, h = blockIdx.z;
    const int q0 = p.cu_seqlens_q[b];
    const int Sq = p.cu_seqlens_q[b + 1] - q0;
    // late tokens see the most keys: they go first, so the long workgroups do not form the tail of the launch
    const int splits = kShared ? p.splits : 1;
    const int from_end = blockIdx.x / splits, split = blockIdx.x - from_end * splits;
    const int tok_block0 = (static_cast<int>(gridDim.x) / splits - 1 - from_end) * kTokens;
    if (tok_block0 >= Sq) return;                              // uniform per workgroup
    const int k0 = p.cu_seqlens_k[b], Lk = p.cu_seqlens_k[b + 1] - k0;
    const int c0 = p.cu_seqlens_c[b], Lc = p.cu_seqlens_c[b + 1] - c0;
    const int s1 = (Lk == Lc) ? 16 : 64;                       // flash_fwd_kernel.h:1236-1240

    const int tok0 = tok_block0 + wave * kMine;                // first token of this wavefront
    int vis_f[kMine], vis_c[kMine];
    bool live[kMine];
#pragma unroll
    for (int t = 0; t < kMine; ++t) {
        const int i = tok0 + t;
        live[t] = i < Sq;
        vis_f[t] = live[t] ? stage1_visible(i, 16, Lk, Sq, kCausal) : 0;
        vis_c[t] = live[t] ? stage1_visible(i, s1, Lc, Sq, kCausal) : 0;
        if (vis_c[t] == 0) vis_f[t] = 0;                       // early exit of flash_fwd_kernel.h:1271-1276
        if (kPool && vis_f[t] > p.score_cols) vis_f[t] = p.score_cols;               // the score row the pooling would have read ends there
    }
    // tile counts are taken over the whole workgroup (its last live token sees the most keys)
    const int i_last = (tok_block0 + kTokens - 1 < Sq ? tok_block0 + kTokens - 1 : Sq - 1);
    const int wg_vis_c = stage1_visible(i_last, s1, Lc, Sq, kCausal);
    const int wg_vis_f = wg_vis_c == 0 ? 0 : stage1_visible(i_last, 16, Lk, Sq, kCausal);
    const int tiles_c = (wg_vis_c + 63) >> 6;
    const int tiles_f = (wg_vis_f + 63) >> 6;
    if constexpr (kItems > 0) {
        // Rows that take as many blocks as they can score need no scores: only blocks up to wg_vis_f / 4 hold a visible key, only those up to the token's own
        // are local, initial blocks are the first ones, and of the others, which score 0 or nothing, the first come first; so the row is its first blocks, whatever the scores.
        // The launch in us, with 64 blocks: 8192 tokens 54.5 -> 39.3, 14 848 + 20 480 + 24 320 + 11 904 packed 715 -> 624, 32 768 440 -> 421; a whole prefill of 4096 204 -> 186,
        // of 1000 with 16 blocks 36.0 -> 31.4, of 777 + 5003 + 1291 + 9173 976 -> 945.
        if (wg_vis_f / kKeysPerBlock < p.topk && i_last / kBlockN < p.topk) {                        // uniform per workgroup
            const int taken = p.topk < p.pool_len ? p.topk : p.pool_len;
#pragma unroll
            for (int t = 0; t < kMine; ++t) {
                if (!live[t]) continue;
                uint64_t* row = p.mask + (static_cast<int64_t>(h) * p.total_q + q0 + tok0 + t) * p.mask_words;
                for (int w = lane; w < p.mask_words; w += 64) row[w] = 64 * w + 64 <= taken ? ~0ull : 64 * w < taken ? (1ull << (taken - 64 * w)) - 1ull : 0ull;
            }
            return;
        }
    }
    // this workgroup's fine tiles; pooled, the scores of the tile before them are made too, for its last key
    const int each = (tiles_f + splits - 1) / splits;
    const int first_f = split * each, end_f = first_f + each < tiles_f ? first_f + each : tiles_f;
    if (kShared && split > 0 && first_f >= tiles_f) return;    // uniform per workgroup
    const int begin_f = kShared && kPool && first_f > 0 ? first_f - 1 : first_f;

    const elem_bits* cbase = p.c + static_cast<int64_t>(c0) * p.c_row_stride + h * p.c_head_stride;
    const elem_bits* kbase = p.k + static_cast<int64_t>(k0) * p.k_row_stride + h * p.k_head_stride;
    const uint32_t lds_tiles = __builtin_amdgcn_readfirstlane(s1_lds_addr(tile));
    const int wave_u = wave;
    const int c_stride = static_cast<int>(p.c_row_stride), k_stride = static_cast<int>(p.k_row_stride);
    const uint32_t c_off = s1_first_off(c_stride, wave, n, g), k_off = s1_first_off(k_stride, wave, n, g);
    if (tiles_c > 0) issue_tile(cbase, c_stride, c_off, 0, Lc, lds_tiles, wave_u, n, g);

    // (Waiting for Q before the tile was requested: kernel alone 20.8 us instead of 20.0 at 4096 tokens, 48.6 instead of 47.2 at 8192.  Of 11 us at 2048 tokens
    // this wait is 3: all of Q, 16.8 MB, at once.)
    // Q as the A operand, requested behind the first tile: r = lane % 16 is the head, g the k-group
    elem8 qf[kTok][4];
#pragma unroll
    for (int t = 0; t < kTok; ++t) {
        const int r = kPack == 2 ? n & 7 : n, want = tok0 + t * kPack + (kPack == 2 ? n >> 3 : 0), i = want < Sq ? want : Sq - 1;
        const elem_bits* qp = p.q + (static_cast<int64_t>(q0) + i) * p.q_tok_stride + h * p.q_kvh_stride + (r < p.group ? r : p.group - 1) * p.q_grp_stride + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[t][c] = *reinterpret_cast<const elem8*>(qp + 32 * c);
    }

    // both have landed from here on: the compiler's wait counts know nothing of the DMA loads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int t = 0; t < kTok; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[t][c]));
    __syncthreads();

    // ---------------- pass 1: per-head log-sum-exp over the coarse keys ----------------
    float m[kTok][4], l[kTok][4];                              // lane-local over keys == n (mod 16); head 4g+e
#pragma unroll
    for (int t = 0; t < kTok; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) { m[t][e] = -INFINITY; l[t][e] = 0.f; }

    int vis_here[kTok];                                        // of the token whose heads this lane holds
#pragma unroll
    for (int t = 0; t < kTok; ++t) vis_here[t] = vis_c[t * kPack] + (g >= 2 ? vis_c[t * kPack + kPack - 1] - vis_c[t * kPack] : 0);      // (a choice of two elements put the array in LDS)
    auto next_coarse = [&](int ti) {
        if (ti + 1 < tiles_c) issue_tile(cbase, c_stride, c_off, (ti + 1) * 64, Lc, lds_tiles + ((ti + 1) & 1) * 16384, wave_u, n, g);
    };
    auto coarse_tile = [&](int ti, floatx4 (&s)[kTok][4]) {
        const uint4* cur = tile[ti & 1];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int t = 0; t < kTok; ++t) s[t][kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint4 raw = cur[(kt * 4 + c) * 64 + lane];
                elem8 kf;
                __builtin_memcpy(&kf, &raw, 16);
#pragma unroll
                for (int t = 0; t < kTok; ++t)
                    s[t][kt] = IV2_MFMA(qf[t][c], kf, s[t][kt], 0, 0, 0);
            }
        }
    };
    auto tile_done = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // this wavefront's share of the next tile has landed
        __syncthreads();
    };
    // Two loops, as many rounds in all for every wavefront of the workgroup.  In the first every key of the tile is visible to all of its
    // tokens: the maximum is finite, no key test, and the scale rides in the multiply-add that feeds exp2, which rounds otherwise: which tiles these are is
    // decided by the first of four tokens, however many of them a wavefront has, so that a row does not depend on that.
    const int seen_c = live[0] ? stage1_visible(tok0 & ~3, s1, Lc, Sq, kCausal) : 0;
    const int whole_c = seen_c >> 6 < tiles_c ? seen_c >> 6 : tiles_c;
    for (int ti = 0; ti < whole_c; ++ti) {
        next_coarse(ti);
        floatx4 s[kTok][4];
        coarse_tile(ti, s);
#pragma unroll
        for (int t = 0; t < kTok; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // (fmaxf quiets its operands first, an instruction each: 131 072 tokens 5380 -> 5300 us)
                const float mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(s[t][0][e], s[t][1][e]), __builtin_elementwise_maximum(s[t][2][e], s[t][3][e]));
                const float m_new = __builtin_elementwise_maximum(m[t][e], mx * p.scale_log2);
                float acc = l[t][e] * __builtin_amdgcn_exp2f(m[t][e] - m_new);
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) acc += __builtin_amdgcn_exp2f(s[t][kt][e] * p.scale_log2 - m_new);
                l[t][e] = acc;
                m[t][e] = m_new;
            }
        }
        tile_done();
    }
    for (int ti = whole_c; ti < tiles_c; ++ti) {               // the tiles that hold a token's last visible key
        next_coarse(ti);
        if (kTok == 1 && !live[0]) {                           // uniform: a wavefront without a token only brings its share of the tiles
            tile_done();
            continue;
        }
        floatx4 s[kTok][4];
        coarse_tile(ti, s);
#pragma unroll
        for (int t = 0; t < kTok; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v[4];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
                    v[kt] = (ti * 64 + kt * 16 + n < vis_here[t]) ? s[t][kt][e] * p.scale_log2 : -INFINITY;
                const float mx = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
                const float m_new = fmaxf(m[t][e], mx);
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
                float acc = l[t][e] * __builtin_amdgcn_exp2f(m[t][e] - m_use);
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) acc += __builtin_amdgcn_exp2f(v[kt] - m_use);
                l[t][e] = acc;
                m[t][e] = m_new;
            }
        }
        tile_done();
    }
    // merge the 16 key-column lanes of each head: lse2 = m + log2(l) in log2 units
    float lse2[kTok][4];
#pragma unroll
    for (int t = 0; t < kTok; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            // the row's maximum first, then every lane's sum rescaled to it once, then the sum of those
            const float mm = row16_max(m[t][e]);
            const float mu = (mm == -INFINITY) ? 0.f : mm;
            const float ll = row16_sum(l[t][e] * __builtin_amdgcn_exp2f(m[t][e] - mu));
            lse2[t][e] = mm + __builtin_amdgcn_logf(ll);        // v_log_f32 is log2
            if ((kPack == 2 ? 4 * (g & 1) : 4 * g) + e >= p.group) lse2[t][e] = INFINITY;    // a row that only fills the tile: exp2(x - inf) = 0 in the head sum
        }

    // ---------------- pass 2: scores over the fine keys ----------------
    if (begin_f < end_f) issue_tile(kbase, k_stride, k_off, begin_f * 64, Lk, lds_tiles + (begin_f & 1) * 16384, wave_u, n, g);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    static_assert(kMine == 1 || kMine % 2 == 0, "pool_quads takes two tokens");
    elem_bits* out_rows[kMine];
    int bq[kMine];                                             // pooled output: the key block the token itself sits in
    float prev[kMine];                                         // pooled output: scores of the previous tile, for its last key
    int plain_first = 0, plain_end;                            // tiles that need no test, below
    {
        const int cache_len = kPool ? (p.cache_lens ? p.cache_lens[b] : p.cache_len) : 0;
        int seen = 0x7fffffff, before_local = 0x7fffffff;
#pragma unroll
        for (int t = 0; t < kMine; ++t) {
            const int64_t row = static_cast<int64_t>(q0) + tok0 + t;
            out_rows[t] = kPool ? p.score + (static_cast<int64_t>(h) * p.score_head_stride + row * p.pool_len)
                                : p.score + h * p.score_head_stride + row * p.score_row_stride;
            bq[t] = (tok0 + t + cache_len) / kBlockN;
            prev[t] = 0.f;
            seen = vis_f[t] < seen ? vis_f[t] : seen;          // 0: no such token
            before_local = bq[t] - p.local_blocks < before_local ? bq[t] - p.local_blocks : before_local;
        }
        // most tiles lie inside the visible keys and the output row, and pooled wholly before the tokens' local windows and after the
        // initial blocks: no key of theirs is hidden, no block forced or empty
        if (seen > p.score_cols) seen = p.score_cols;
        plain_end = seen >> 6;
        if (kPool) {
            before_local = before_local < p.pool_len ? before_local : p.pool_len;
            plain_end = before_local < 0 ? 0 : (before_local >> 4) < plain_end ? before_local >> 4 : plain_end;
            plain_first = (p.init_blocks >> 4) + ((p.init_blocks & 15) != 0 ? 1 : 0);      // (rounded up without a sum that could overflow)
        }
    }
    // value of a pooled entry that no visible key reaches
    auto pool_rest = [&](int kb, int bq_t, float reached) -> elem_bits {
        const bool forced = (kb < p.init_blocks) || (bq_t >= kb && bq_t <= kb + p.local_blocks);
        const int first = kb * kKeysPerBlock - 1;              // first key of the window (before clipping at 0)
        const bool empty = (first < 0 ? 0 : first) >= (Lk < p.score_cols ? Lk : p.score_cols);
        return forced ? kElemPosInf : (empty ? kElemNegInf : f32_to_elem_hw(reached));
    };

    // A plain tile's results are stored when the next tile begins: the wait at a tile's end counts stores too, and one just
    // issued would add its round trip to every tile.
    float held[kMine] = {};
    bool pending = false;
    auto store = [&](int t, uint32_t at, elem_bits value) {
        if constexpr (kItems > 0) pooled[wave * kMine + t][at] = value;
        else out_rows[t][at] = value;
    };
    auto store_held = [&](int ti) {
        const uint32_t at = static_cast<uint32_t>(kPool ? ti * 16 + (lane >> 2) : ti * 64 + lane);
        if (!kPool || (lane & 3) == 0) {
#pragma unroll
            for (int t = 0; t < kMine; ++t) store(t, at, f32_to_elem_hw(held[t]));
        }
    };
    for (int ti = begin_f; ti < end_f; ++ti) {
        if (pending) store_held(ti - 1);                       // uniform per wavefront
        if (ti + 1 < end_f) issue_tile(kbase, k_stride, k_off, (ti + 1) * 64, Lk, lds_tiles + ((ti + 1) & 1) * 16384, wave_u, n, g);
        if (kTok == 1 && !live[0]) {
            tile_done();
            continue;
        }
        const uint4* cur = tile[ti & 1];
        float part[kTok][4];                                   // [t][kt]: this lane's four heads summed, key 16 kt + n
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            floatx4 s[kTok];
#pragma unroll
            for (int t = 0; t < kTok; ++t) s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint4 raw = cur[(kt * 4 + c) * 64 + lane];
                elem8 kf;
                __builtin_memcpy(&kf, &raw, 16);
#pragma unroll
                for (int t = 0; t < kTok; ++t)
                    s[t] = IV2_MFMA(qf[t][c], kf, s[t], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < kTok; ++t) {
                float sum = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) sum += __builtin_amdgcn_exp2f(s[t][e] * p.scale_log2 - lse2[t][e]);
                part[t][kt] = sum;
            }
        }
        // sum over the four 16-lane rows (the head groups) and hand row kt the total of key tile kt, in three
        // exchanges: (row0 + row1 | row2 + row3) of tiles 0/1 and of tiles 2/3, then the two halves.  lane = 16*g + n  <->  key 16*g + n of this tile
        float mine[kMine];
#pragma unroll
        for (int t = 0; t < kTok; ++t) {
            const float even = fold_rows16(part[t][0], part[t][1]), odd = fold_rows16(part[t][2], part[t][3]);
            if constexpr (kPack == 1) mine[t] = fold_rows32(even, odd);
            else halves(even, odd, mine[2 * t], mine[2 * t + 1]);
        }
        const bool mine_too = !kShared || !kPool || ti >= first_f;                   // not the tile before
        pending = ti >= plain_first && ti < plain_end && mine_too;
        const int col = ti * 64 + lane;
        if (!pending) {
#pragma unroll
            for (int t = 0; t < kMine; ++t) mine[t] = col < vis_f[t] ? mine[t] : 0.f;     // keys the token may not see score 0
        }
        if (!kPool) {
#pragma unroll
            for (int t = 0; t < kMine; ++t) {
                held[t] = mine[t];
                if (!pending && live[t] && col < p.score_cols) out_rows[t][col] = f32_to_elem_hw(mine[t]);
            }
        } else {
            // block kb = col / 4 pools keys 4 kb - 1 .. 4 kb + 3: its quad and the last key of the quad before
            if constexpr (kMine == 1) {
                float same;
                pool_quads(mine[0], mine[0], prev[0], prev[0], held[0], same);
            } else {
#pragma unroll
                for (int t = 0; t < kMine; t += 2) pool_quads(mine[t], mine[t + 1], prev[t], prev[t + 1], held[t], held[t + 1]);
            }
            const int kb = col >> 2;
#pragma unroll
            for (int t = 0; t < kMine; ++t) {
                prev[t] = mine[t];
                if (!pending && mine_too && live[t] && (lane & 3) == 0 && kb < p.pool_len) store(t, kb, pool_rest(kb, bq[t], held[t]));
            }
        }
        tile_done();
    }
    if (pending) store_held(end_f - 1);
    if (kShared && end_f < tiles_f) return;                // uniform per workgroup; the rest is the last one's
    // columns no tile covered
#pragma unroll
    for (int t = 0; t < kMine; ++t) {
        if (!live[t]) continue;
        if (!kPool) {
            for (int col = tiles_f * 64 + lane; col < p.score_cols; col += 64) out_rows[t][col] = 0;
        } else {
            // the first of them still sees the last key of the last tile
            const float last_score = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(prev[t]), 63));
            for (int kb = tiles_f * 16 + lane; kb < p.pool_len; kb += 64)
                store(t, kb, pool_rest(kb, bq[t], kb == tiles_f * 16 ? last_score : 0.f));
        }
    }
    if constexpr (kItems > 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        uint32_t key[kMine][kItems];                           // 0: no column
        const int take_at_most = p.topk < p.pool_len ? p.topk : p.pool_len;
#pragma unroll
        for (int t = 0; t < kMine; ++t)
#pragma unroll
            for (int e = 0; e < kItems; ++e) {
                const int kb = 64 * e + lane;
                key[t][e] = kb < p.pool_len ? sortable16(pooled[wave * kMine + t][kb]) : 0u;
            }
        auto count = [&](int t, auto&& in) {
            int c = 0;
#pragma unroll
            for (int e = 0; e < kItems; ++e) c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(in(key[t][e])));
            return c;
        };
        uint32_t thr[kMine];                                   // the largest key that so many keys reach
#pragma unroll
        for (int t = 0; t < kMine; ++t) thr[t] = 0;
#pragma unroll
        for (int bit = 15; bit >= 0; --bit)
#pragma unroll
            for (int t = 0; t < kMine; ++t) {
                const uint32_t next = thr[t] | (1u << bit);
                thr[t] = count(t, [&](uint32_t x) { return x >= next; }) >= take_at_most ? next : thr[t];
            }
#pragma unroll
        for (int t = 0; t < kMine; ++t) {
            if (!live[t]) continue;
            int ties = take_at_most - count(t, [&](uint32_t x) { return x > thr[t]; });          // of the keys equal to it
            uint64_t words = 0ull;                             // lane w: word w
#pragma unroll
            for (int e = 0; e < kItems; ++e) {
                const uint64_t equal = __builtin_amdgcn_ballot_w64(key[t][e] == thr[t]);
                const int rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(equal >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(equal), 0));
                const uint64_t taken = __builtin_amdgcn_ballot_w64(key[t][e] > thr[t] || (key[t][e] == thr[t] && rank < ties));
                words = lane == e ? taken : words;
                ties -= __builtin_popcountll(equal);
            }
            uint64_t* row = p.mask + (static_cast<int64_t>(h) * p.total_q + q0 + tok0 + t) * p.mask_words;
            for (int w = lane; w < p.mask_words; w += 64) row[w] = w < kItems ? words : 0ull;
        }
    }
}

}  // namespace IV2_NS

using namespace IV2_NS;

namespace {

struct Stage1Pool {                  // pooled-output mode of the launch below
    const int32_t* cache_lens;
    int cache_len, pool_len, local_blocks, init_blocks;
    uint64_t* mask = nullptr;        // not null: the selection instead
    int mask_words = 0, topk = 0;
};

int launch_stage1(const char* who, void* stream, const void* q, const void* k, const void* v, void* out,
                  const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, const int32_t* cu_seqlens_v, int batch,
                  int64_t total_q, int num_heads, int num_heads_k, int head_dim, int max_seqlen_q, int max_seqlen_k,
                  const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                  int64_t out_head_stride, int64_t out_row_stride, float softmax_scale, int is_causal,
                  const Stage1Pool* pool) {
    IV2_CHECK(head_dim == kHeadDim, "%s: this build only supports head_dim 128 (got %d)", who, head_dim);
    IV2_CHECK(valid_group(num_heads, num_heads_k),
              "%s: requires num_heads == g * num_heads_k with g in {1, 2, 4, 8, 16} (got %d and %d)", who, num_heads, num_heads_k);
    IV2_CHECK(batch > 0 && total_q >= 0 && max_seqlen_q >= 0 && max_seqlen_k >= 0, "%s: bad sizes", who);
    IV2_CHECK(q && k && v && (out || (pool && pool->mask)) && cu_seqlens_q && cu_seqlens_k && cu_seqlens_v, "%s: null pointer", who);
    IV2_CHECK(num_heads_k <= 65535 && batch <= 65535, "%s: batch and num_heads_k must not exceed 65535", who);
    IV2_CHECK(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(v) % 16 == 0, "%s: q, k, v must be 16-byte aligned", who);
    for (int s = 0; s < 3; ++s) IV2_CHECK(q_strides[s] % 8 == 0, "%s: q strides must be multiples of 8 elements", who);
    IV2_CHECK(k_strides[0] % 8 == 0 && k_strides[1] % 8 == 0 && v_strides[0] % 8 == 0 && v_strides[1] % 8 == 0,
              "%s: k/v strides must be multiples of 8 elements", who);
    // a lane's byte offset from its sequence's first compressed key is a 32-bit LDS-DMA operand
    IV2_CHECK(k_strides[0] > 0 && v_strides[0] > 0 &&
              (static_cast<int64_t>(max_seqlen_k) + 64) * k_strides[0] < (1ll << 30) &&
              (static_cast<int64_t>(max_seqlen_k) + 64) * v_strides[0] < (1ll << 30),
              "%s: compressed-key rows too far apart (row stride x max_seqlen_k must stay below 2^30 elements)", who);
    if (total_q == 0 || max_seqlen_q == 0) return 0;
    Stage1Params p{};
    p.q = static_cast<const elem_bits*>(q);
    p.k = static_cast<const elem_bits*>(k);
    p.c = static_cast<const elem_bits*>(v);
    p.score = static_cast<elem_bits*>(out);
    p.cu_seqlens_q = cu_seqlens_q; p.cu_seqlens_k = cu_seqlens_k; p.cu_seqlens_c = cu_seqlens_v;
    p.q_tok_stride = q_strides[0]; p.q_grp_stride = q_strides[1]; p.q_kvh_stride = q_strides[2];
    p.k_row_stride = k_strides[0]; p.k_head_stride = k_strides[1];
    p.c_row_stride = v_strides[0]; p.c_head_stride = v_strides[1];
    p.score_head_stride = out_head_stride; p.score_row_stride = out_row_stride;
    p.score_cols = max_seqlen_k;
    p.group = num_heads / num_heads_k;
    p.scale_log2 = softmax_scale * 1.44269504088896340736f;
    p.causal = is_causal;
    if (pool) {
        p.cache_lens = pool->cache_lens; p.cache_len = pool->cache_len; p.pool_len = pool->pool_len;
        p.local_blocks = pool->local_blocks; p.init_blocks = pool->init_blocks;
        p.mask = pool->mask; p.total_q = total_q; p.mask_words = pool->mask_words; p.topk = pool->topk;
    }
    // Few workgroups leave CUs idle while each walks all tiles, so they share the fine ones (every one walks the coarse tiles, a quarter as many): as many sharers as
    // give each CU a workgroup, with four tiles each at least.  Kernel alone, us, 2 KV heads, 20 011 keys: 16 queries 34.8 -> 19.3, 256 35.4 -> 20.1, 512 34.8 -> 21.2, 700 35.2 ->
    // 25.6, 1024 35.5 -> 27.2; 60 000 keys, one KV head, 300 queries 90.4 -> 36.1; a whole chunk of 512 queries behind 19 499 keys 154.7 -> 139.9.  Two workgroups to a
    // CU: 700 queries 31.0, 1500 36.1 -> 39.5; two tiles each at least: 256 queries 26.7.
    // Groups of 8 heads and fewer: two tokens share the 16 rows of a product, of which half were spare.  us, groups of 8, 2 KV heads, one | two tokens:
    //   scores of 256 queries against 20 011 keys 13.6 | 13.6, 2049 51.1 | 36.5, 8000 92 | 63; selecting prefill of 2048 tokens 15.7 | 15.0, 32 768 391 | 257;
    //   scores of 65 536, one KV head, with the top-k launch 733 | 453.
    const int pack = p.group <= 8 ? 2 : 1;
    const int64_t wgs = static_cast<int64_t>((max_seqlen_q + kTokPerBlock * pack - 1) / (kTokPerBlock * pack)) * batch * num_heads_k;
    const int64_t fill = wgs > 0 ? 256 / wgs : 1, most = max_seqlen_k / 256;
    p.splits = p.mask != nullptr || fill < 2 || most < 2 ? 1 : static_cast<int>(fill < most ? fill : most);
    // One token to a wavefront (two, where two share the rows), twice the workgroups, up to 384 of the others: three to a CU.  The time is then that of the CU with the
    // most, half a workgroup finer, and of the chain of one tile (one wavefront's products and exponentials behind the other's on a SIMD), which is shorter.
    // Scores alone, us, two tokens | one:
    //   2 KV heads, 20 011 keys: 17 queries 18.8 | 12.5, 256 19.3 | 13.3, 512 20.1 | 20.6, 1100 35.1 | 32.9, 2049 54.0 | 42.2, 3000 (376 workgroups) 56.1 | 49.4;
    //   3100 (388) 55.3 | 58.8, 4096 60.0 | 63.6; 131 072 keys: 2049 344 | 244, 3100 313 | 362; selecting prefill of 1000 tokens 15.2 | 12.4;
    //   whole sequences, whose workgroups walk from one tile to all: 1160 tokens, 4 KV heads, 13.6 | 11.0, 2185, 2 heads, 14.5 | 11.2, 3849, one head, 12.8 | 10.7,
    //   487 + 1295 + 909, one head, 11.0 | 9.6.
    // Selecting, a workgroup walks what its own tokens see, from one tile to all of them, and smaller ones end together: always where two tokens share the rows, else up to
    // 10 240 tokens; longer, the keys' second trip from L2 costs more.  Selection in us, two tokens | one, 2 KV heads, 16 blocks:
    //   6000 tokens 39.1 | 38.0, 10 000 71.6 | 66.5, 777 + 5003 + 1291 + 9173 92.2 | 83.1, 5000 x 4 80.6 | 77.5, 8000 x 3 115.8 | 115.9;
    //   left to two: 11 300 79.3 | 74.4, 12 000 82.6 | 77.5, 11 000 with 4 heads and 32 blocks 125 | 120, 11 300 + 11 800 + 11 000 + 10 000 249 | 244;
    //   12 000 x 4 300 | 317, 16 000 129 | 130.5, 24 000 251.5 | 264.5; groups of 8: 8192 42.1 | 37.9, 20 000 138.6 | 126.8, 24 000 171.5 | 166.2.
    // Workgroups whose rows take every block return at once and do not count (selecting prefill of 5000 tokens, 64 blocks, 22.9 | 19.8, of 8192 with one KV head 26.2 | 23.8).
    constexpr int64_t kOneTokenWorkgroups = 384, kOneTokenLength = 10240;
    const int64_t scored = p.mask ? static_cast<int64_t>(max_seqlen_q) - static_cast<int64_t>(kBlockN) * p.topk : max_seqlen_q;
    const bool one = (p.mask && (pack == 2 || max_seqlen_q <= kOneTokenLength)) ||
                     (scored + kTokPerBlock * pack - 1) / (kTokPerBlock * pack) * batch * num_heads_k <= kOneTokenWorkgroups;
    const int tokens = (one ? kWavesS1 : kTokPerBlock) * pack;
    const dim3 grid((max_seqlen_q + tokens - 1) / tokens * p.splits, batch, num_heads_k);
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto pick = [&](auto tok, auto packed) {
        constexpr int kTok = decltype(tok)::value, kPack = decltype(packed)::value;
        if constexpr (kTok == 1 || kPack == 1) {               // selecting, two tokens that share their rows are all a wavefront takes
            if (p.mask) return p.pool_len <= 64 ? stage1_kernel<true, true, 1, false, kTok, kPack> : p.pool_len <= 128 ? stage1_kernel<true, true, 2, false, kTok, kPack>
                             : p.pool_len <= 256 ? stage1_kernel<true, true, 4, false, kTok, kPack> : stage1_kernel<true, true, 8, false, kTok, kPack>;
        }
        static_assert(kOneTokenWorkgroups >= 128, "launches that share tokens have at most so many workgroups");
        if constexpr (kTok == 1) {
            if (p.splits > 1) return pool ? (is_causal ? stage1_kernel<true, true, 0, true, kTok, kPack> : stage1_kernel<false, true, 0, true, kTok, kPack>)
                                          : (is_causal ? stage1_kernel<true, false, 0, true, kTok, kPack> : stage1_kernel<false, false, 0, true, kTok, kPack>);
        }
        return pool ? (is_causal ? stage1_kernel<true, true, 0, false, kTok, kPack> : stage1_kernel<false, true, 0, false, kTok, kPack>)
                    : (is_causal ? stage1_kernel<true, false, 0, false, kTok, kPack> : stage1_kernel<false, false, 0, false, kTok, kPack>);
    };
    constexpr std::integral_constant<int, 1> k1{};
    constexpr std::integral_constant<int, 2> k2{};
    static_assert(kTokPerWave == 2, "k2");
    auto kernel = one ? (pack == 2 ? pick(k1, k2) : pick(k1, k1)) : (pack == 2 ? pick(k2, k2) : pick(k2, k1));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * kWavesS1), 0, st, p);
    IV2_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int IV2_ENTRY(infllmv2_varlen_fwd_stage1)(void* stream, const void* q, const void* k, const void* v, void* score,
                                          const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                          const int32_t* cu_seqlens_v, int batch, int64_t total_q, int num_heads,
                                          int num_heads_k, int head_dim, int max_seqlen_q, int max_seqlen_k,
                                          const int64_t* q_strides, const int64_t* k_strides,
                                          const int64_t* v_strides, int64_t score_head_stride,
                                          int64_t score_row_stride, float softmax_scale, int is_causal) {
    IV2_CHECK(score_row_stride >= max_seqlen_k, "varlen_fwd_stage1: score row stride shorter than max_seqlen_k");
    return launch_stage1("varlen_fwd_stage1", stream, q, k, v, score, cu_seqlens_q, cu_seqlens_k, cu_seqlens_v, batch,
                         total_q, num_heads, num_heads_k, head_dim, max_seqlen_q, max_seqlen_k, q_strides, k_strides,
                         v_strides, score_head_stride, score_row_stride, softmax_scale, is_causal, nullptr);
}

extern "C" int IV2_ENTRY(infllmv2_varlen_fwd_stage1_pooled)(void* stream, const void* q, const void* k, const void* v,
                                                 void* pooled, const int32_t* cu_seqlens_q,
                                                 const int32_t* cu_seqlens_k, const int32_t* cu_seqlens_v,
                                                 const int32_t* cache_lens, int cache_len, int batch,
                                                 int64_t total_q, int num_heads, int num_heads_k, int head_dim,
                                                 int max_seqlen_q, int max_seqlen_k, const int64_t* q_strides,
                                                 const int64_t* k_strides, const int64_t* v_strides, int out_len,
                                                 float softmax_scale, int is_causal, int kernel_size, int stride,
                                                 int padding, int block_size, int local_blocks, int init_blocks) {
    IV2_CHECK(kernel_size == 5 && stride == 4 && padding == 1 && block_size == kBlockN,
              "varlen_fwd_stage1_pooled: only the 5/4/1 window on 64-token blocks is fused (got %d/%d/%d on %d); "
              "use varlen_fwd_stage1 and max_pooling_1d", kernel_size, stride, padding, block_size);
    IV2_CHECK(out_len >= 0 && cache_len >= 0, "varlen_fwd_stage1_pooled: negative out_len or cache_len");
    if (out_len == 0) return 0;
    const Stage1Pool pool{cache_lens, cache_len, out_len, local_blocks, init_blocks};
    return launch_stage1("varlen_fwd_stage1_pooled", stream, q, k, v, pooled, cu_seqlens_q, cu_seqlens_k, cu_seqlens_v,
                         batch, total_q, num_heads, num_heads_k, head_dim, max_seqlen_q, max_seqlen_k, q_strides,
                         k_strides, v_strides, total_q * static_cast<int64_t>(out_len), out_len, softmax_scale,
                         is_causal, &pool);
}

extern "C" int IV2_ENTRY(infllmv2_varlen_fwd_stage1_selected)(void* stream, const void* q, const void* k, const void* v, uint64_t* mask,
                                                   const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                                   const int32_t* cu_seqlens_v, int batch, int64_t total_q, int num_heads,
                                                   int num_heads_k, int head_dim, int max_seqlen_q, int max_seqlen_k,
                                                   const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                                   int out_len, float softmax_scale, int kernel_size, int stride, int padding,
                                                   int block_size, int local_blocks, int init_blocks, int topk, int n_uint64_per_row) {
    IV2_CHECK(kernel_size == 5 && stride == 4 && padding == 1 && block_size == kBlockN,
              "varlen_fwd_stage1_selected: only the 5/4/1 window on 64-token blocks is fused (got %d/%d/%d on %d); "
              "use varlen_fwd_stage1, max_pooling_1d and topk_mask", kernel_size, stride, padding, block_size);
    IV2_CHECK(out_len > 0 && out_len <= INFLLMV2_STAGE1_SELECT_BLOCKS, "varlen_fwd_stage1_selected: 1 to %d blocks (got %d)",
              INFLLMV2_STAGE1_SELECT_BLOCKS, out_len);
    IV2_CHECK(topk >= 0, "topk: negative size");
    IV2_CHECK(topk <= 2048, "topk: k %d exceeds 2048", topk);
    IV2_CHECK(mask != nullptr, "varlen_fwd_stage1_selected: null pointer");
    IV2_CHECK(n_uint64_per_row > 0 && static_cast<int64_t>(n_uint64_per_row) * 64 >= out_len,
              "topk: %d mask words per row cannot hold %d columns", n_uint64_per_row, out_len);
    const Stage1Pool pool{nullptr, 0, out_len, local_blocks, init_blocks, mask, n_uint64_per_row, topk};
    return launch_stage1("varlen_fwd_stage1_selected", stream, q, k, v, nullptr, cu_seqlens_q, cu_seqlens_k, cu_seqlens_v,
                         batch, total_q, num_heads, num_heads_k, head_dim, max_seqlen_q, max_seqlen_k, q_strides,
                         k_strides, v_strides, 0, 0, softmax_scale, 1, &pool);
}
