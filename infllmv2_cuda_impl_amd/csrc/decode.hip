// Stage-2 decode against a KV cache for gfx950: one query token per sequence, attention restricted
// to the 64-key blocks set in the sequence's mask row, optional in-place append of new keys/values.
//
// Semantics follow mha_fwd_kvcache (csrc/flash_attn/flash_api.cpp:1549-1843) on the path the
// Python wrapper takes (infllm_v2/infllmv2_sparse_attention.py:730-757): seqlen_q == 1, so the
// causal flag is dropped (flash_api.cpp:1628); the 16 grouped heads of a KV head form the row tile
// (flash_api.cpp:1633-1639); keys [0, cache_seqlens[b] + seqlen_new) are visible; new k/v are
// written at cache_seqlens[b] first (flash_fwd_kernel.h:792-891); the result must not depend on
// the number of KV splits (combine by LSE, flash_fwd_kernel.h:1866-1946).
//
// Design: decode is HBM-bound (each selected block is 32 KiB of K+V read exactly once, ~2 MiB per
// sequence and KV head), so the kernel reads the cache in the caller's layout, with no repacking
// pass.  A workgroup of one wavefront, or of four where a launch has at most one workgroup per CU, handles one (sequence, KV
// head, split); a split is a contiguous run of the row's selected blocks (by ordinal, so splits are balanced whatever the
// selection looks like).  Whole K and V rows go to an LDS ring by LDS-DMA; K is read from it as the MFMA A operand (contraction
// over d), V, which is contracted over keys, by transposing reads.  Partial results are merged by a small combine kernel.
#include "common.h"
#include "block_walker.h"
#include "decode_step.h"
#include "infllmv2_hip.h"
#include <math.h>
#include <mutex>

namespace IV2_NS {

struct DecodeParams {
    const elem_bits* q;
    elem_bits* kcache;
    elem_bits* vcache;
    const elem_bits* knew;
    const elem_bits* vnew;
    elem_bits* out;
    float* lse;                     // (batch, Hq)
    float* o_part;                  // (batch, Hk, splits, 16, 128) fp32, normalised per split
    float* lse_part;                // (batch, Hk, splits, 16)
    const int* cache_seqlens;       // null: every sequence fills the whole cache
    const uint64_t* mask;           // (batch, Hk, n64) or null
    const int* topk_idx;            // (batch, Hk, k_idx): the selection as an index list instead (-1: unused slot), or null
    int k_idx;
    const elem_bits* scores;         // (batch, Hk, n_scores) block scores: the selection is their k_select largest; or null
    int n_scores, k_select;         // (a whole step: blocks of a row at most)
    int64_t q_batch, q_head;        // element strides of q (batch, head); head dim dense
    int64_t o_batch, o_head;
    int64_t kc_batch, kc_row, kc_head, vc_batch, vc_row, vc_head;
    int64_t kn_batch, kn_row, kn_head, vn_batch, vn_row, vn_head;
    int batch, num_heads_k, capacity, seqlen_new, n64, splits;
    int group;                      // query heads per KV head, 1..16
    float scale_log2;
    // where a sequence's rows lie (flash_api.cpp:1593-1611, 1762-1771, 1800-1808)
    const int* cache_batch_idx;     // sequence b uses cache row cache_batch_idx[b]; null: b
    const int* leftpad;             // the sequence's keys start at cache row leftpad[b]; null: 0
    const int* block_table;         // (batch, pages per sequence): the caches are (pages, page_size, Hk, d)
    int64_t bt_batch;
    int page_size;
    // rotary embedding of the appended keys and of the query (flash_fwd_kernel.h:787-929, rotary.h)
    const elem_bits* rot_cos;       // (seqlen_ro, rotary_dim / 2)
    const elem_bits* rot_sin;
    int rotary_dim, rotary_interleaved;
    int mask_in_place;              // the mask has more words than LDS holds: read where they are
    int far_rows;                   // cache rows lie too far apart (or backwards) for 32-bit offsets inside a block
    int append_here;                // the split kernel itself writes the one new row per sequence (and sees it whatever the cache holds)
};

// element offset of cache row `row` of sequence b (head 0)
__device__ __forceinline__ int64_t cache_row_offset(const DecodeParams& p, int b, int row, int64_t batch_stride,
                                                    int64_t row_stride) {
    if (p.block_table) {
        const int page = p.block_table[b * p.bt_batch + row / p.page_size];
        return page * batch_stride + static_cast<int64_t>(row % p.page_size) * row_stride;
    }
    const int cb = p.cache_batch_idx ? p.cache_batch_idx[b] : b;
    return cb * batch_stride + static_cast<int64_t>(row) * row_stride;
}

// One 16-byte chunk (8 values, d = 8 chunk ...) of a head vector and what turns it at position pos: requested by
// rotary_request, used by rotary_turn, so that a caller with several chunks has all of them in flight (one chunk after the
// other, each waiting for its own, made the set-up of a short split five round trips longer).  Interleaved: pairs (2i, 2i+1)
// lie inside the chunk; contiguous: the partner of d is d +- rotary_dim / 2, in another chunk of the same head vector.
// (a, b) -> (a cos - b sin, a sin + b cos) in fp32, one rounding (rotary.h:57-62, 131-133).
struct RotaryChunk {
    uint4 own, other;
    uint2 c[2], s[2];                                          // table values: four (interleaved) or eight
};
__device__ __forceinline__ RotaryChunk rotary_request(const DecodeParams& p, const elem_bits* head_vec, int chunk, int pos) {
    RotaryChunk r;
    const int half = p.rotary_dim >> 1, d0 = chunk * 8;
    r.own = *reinterpret_cast<const uint4*>(head_vec + d0);
    const int d = d0 < p.rotary_dim ? d0 : 0;                  // beyond the turned part: any valid address
    const int in_half = d < half ? d : d - half;
    r.other = *reinterpret_cast<const uint4*>(head_vec + (p.rotary_interleaved ? d : (d < half ? d + half : d - half)));
    // the tables are only 2-byte aligned, which global loads do not mind; interleaved, the second four may lie beyond the row
    const int64_t at = static_cast<int64_t>(pos) * half + (p.rotary_interleaved ? d >> 1 : in_half);
    const int second = p.rotary_interleaved ? 0 : 4;
    __builtin_memcpy(&r.c[0], p.rot_cos + at, 8);
    __builtin_memcpy(&r.c[1], p.rot_cos + at + second, 8);
    __builtin_memcpy(&r.s[0], p.rot_sin + at, 8);
    __builtin_memcpy(&r.s[1], p.rot_sin + at + second, 8);
    return r;
}
__device__ __forceinline__ uint4 rotary_turn(const DecodeParams& p, const RotaryChunk& r, int chunk) {
    const int d0 = chunk * 8;
    const bool left = d0 < (p.rotary_dim >> 1);
    const uint32_t w[4] = {r.own.x, r.own.y, r.own.z, r.own.w}, ow[4] = {r.other.x, r.other.y, r.other.z, r.other.w};
    const uint32_t cw[4] = {r.c[0].x, r.c[0].y, r.c[1].x, r.c[1].y}, sw[4] = {r.s[0].x, r.s[0].y, r.s[1].x, r.s[1].y};
    uint32_t out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float x0 = elem_lo_to_f32(w[e]), x1 = elem_hi_to_f32(w[e]);
        float y0, y1;
        if (p.rotary_interleaved) {                            // uniform: table value e
            const float c = (e & 1) ? elem_hi_to_f32(cw[e >> 1]) : elem_lo_to_f32(cw[e >> 1]);
            const float sn = (e & 1) ? elem_hi_to_f32(sw[e >> 1]) : elem_lo_to_f32(sw[e >> 1]);
            y0 = x0 * c - x1 * sn;
            y1 = x0 * sn + x1 * c;
        } else {                                               // table values 2 e and 2 e + 1
            const float c0 = elem_lo_to_f32(cw[e]), c1 = elem_hi_to_f32(cw[e]), s0 = elem_lo_to_f32(sw[e]), s1 = elem_hi_to_f32(sw[e]);
            const float o0 = elem_lo_to_f32(ow[e]), o1 = elem_hi_to_f32(ow[e]);
            y0 = left ? x0 * c0 - o0 * s0 : x0 * c0 + o0 * s0;
            y1 = left ? x1 * c1 - o1 * s1 : x1 * c1 + o1 * s1;
        }
        out[e] = d0 < p.rotary_dim ? pack_elem2(y0, y1) : w[e];
    }
    return make_uint4(out[0], out[1], out[2], out[3]);
}
__device__ __forceinline__ uint4 rotary_chunk(const DecodeParams& p, const elem_bits* head_vec, int chunk, int pos) {
    return rotary_turn(p, rotary_request(p, head_vec, chunk, pos), chunk);
}

// Several new rows per sequence (one is written by the split kernel itself): one thread moves 16 bytes of one new row
// of K and of V.
__global__ __launch_bounds__(256)
void decode_append_kernel(const DecodeParams p) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t total = static_cast<int64_t>(p.batch) * p.seqlen_new * p.num_heads_k * 16;
    if (idx >= total) return;
    const int chunk = static_cast<int>(idx & 15);
    int64_t r = idx >> 4;
    const int h = static_cast<int>(r % p.num_heads_k); r /= p.num_heads_k;
    const int t = static_cast<int>(r % p.seqlen_new);
    const int b = static_cast<int>(r / p.seqlen_new);
    const int pos = (p.cache_seqlens ? p.cache_seqlens[b] : 0) + t;             // cache row, left padding included
    if (pos >= p.capacity) return;
    const elem_bits* kvec = p.knew + b * p.kn_batch + t * p.kn_row + h * p.kn_head;
    const uint4 kv = p.rotary_dim > 0 ? rotary_chunk(p, kvec, chunk, pos) : *reinterpret_cast<const uint4*>(kvec + chunk * 8);
    const uint4 vv = *reinterpret_cast<const uint4*>(p.vnew + b * p.vn_batch + t * p.vn_row + h * p.vn_head + chunk * 8);
    *reinterpret_cast<uint4*>(p.kcache + cache_row_offset(p, b, pos, p.kc_batch, p.kc_row) + h * p.kc_head + chunk * 8) = kv;
    *reinterpret_cast<uint4*>(p.vcache + cache_row_offset(p, b, pos, p.vc_batch, p.vc_row) + h * p.vc_head + chunk * 8) = vv;
}

typedef short short4d __attribute__((ext_vector_type(4)));
// 16 lanes x 4 halfwords, transposed (ds_read_b64_tr_b16): lane 16 g + r receives element r % 4 of the four-halfword
// rows offered by lanes 16 g + r / 4 + {0, 4, 8, 12}
__device__ __forceinline__ short4d lds_read_tr(const elem_bits* ptr) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4d*)(ptr));
}

__device__ __forceinline__ uint64_t decode_uniform64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// A block's tile in LDS: 64 rows of 256 bytes (K, then V), filled by LDS-DMA.  A DMA instruction moves four whole rows
// (lane 16 g + n: 16 bytes of row 4 u + g) and lands them in lane order, so the rows are unpadded, and the 16-byte
// pieces of a row are stored XOR-ed with a function of the row instead: both the operand reads of K (16 rows, one piece
// each) and the transposing reads of V (8 rows, two neighbouring pieces each) then touch every bank once.
constexpr int kTileBytes = kBlockN * kHeadDim * 2;             // 16 KiB
constexpr int kSlotBytes = 2 * kTileBytes;
__device__ __forceinline__ int tile_swizzle(int row) { return ((row & 7) << 1) | ((row >> 3) & 1); }
__device__ __forceinline__ uint32_t decode_lds_address(const void* ptr) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)ptr));
}
// 16 bytes per lane from base + lane_off to LDS at lds + 16 lane.  Non-temporal: the rows are read once per step.
// The compiler does not see these loads: whoever reads the tile waits for them by hand.
__device__ __forceinline__ void decode_dma16(const void* base, uint32_t lane_off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(lane_off), "s"(base), "s"(lds) : "memory", "m0");
}
// the same from an address of each lane's own
__device__ __forceinline__ void decode_dma16(const void* lane_src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(lane_src), "s"(lds) : "memory", "m0");
}

// v (wavefront-uniform, more than `rank` bits set) without its `rank` lowest set bits
__device__ __forceinline__ uint64_t drop_set_bits(uint64_t v, int rank) {
    int pos = 0;
#pragma unroll
    for (int width = 32; width > 0; width >>= 1) {
        const int c = __builtin_popcountll((v >> pos) & ((1ull << width) - 1ull));
        if (rank >= c) { rank -= c; pos += width; }
    }
    return v & (~0ull << pos);
}

// A workgroup per (sequence, KV head, split), bound by HBM: 16 KiB of K and of V per block, read once.  The split's run of
// blocks is shared out again among its wavefronts, each with its own tiles, softmax state and output; they meet once, at the
// end.  Whole rows go to LDS by non-temporal DMA (269 MB of selected blocks: 45 us for the loads alone, against 51 us for the
// 16-row pieces of 64 bytes that MFMA operands want straight from memory, and no faster with those marked non-temporal: their
// 128-byte lines are then fetched twice).
//   kWaves == 1: two block tiles per workgroup, two workgroups per CU.  For launches that fill the chip with them.
//   kWaves == 4: one tile per wavefront; K of the next block is requested as soon as S is formed, V after the output.  The
//                same 128 KiB in flight per CU, but four blocks are fetched and used side by side and leave one partial:
//                for the launches whose runs hold a few blocks, where the time is a chain of round trips, not bandwidth
//                (with the merge: 1 sequence x 2 heads x 64 blocks 16 -> 9.1 us, 6 sequences 18.4 -> 10.7, 24 sequences
//                32 -> 23, 64 sequences 51.6 -> 49; 64 x 4 heads, one workgroup each and no merge, 95 -> 89).
//
// The set-up is a chain of round trips in front of the first block, so everything that does not depend on anything is
// requested together: the sequence's length, the mask words (or the index list, OR-ed into words in LDS: no packing
// launch), the query and the new row.  The run's blocks (64 at a time) and their pages are then looked up by the lanes in
// parallel and kept in registers: the walk itself makes no loads but the DMA.
//
// append_here: the sequence's one new row is patched into its block's tile (turned by the rotary embedding where asked
// for), so the row need not be in the cache before the launch: the first workgroup of each (sequence, KV head) writes
// it there on its way out.  What a reader of that row gets from memory does not matter, NaN included: the tile's rows
// behind the end are copies of it, K's are masked by assignment and V's, which are multiplied by P = 0, are patched too.
constexpr int kMergePitch = kHeadDim + 4;                      // floats per head of a wavefront's output in LDS

// The k largest of the first `cols` of a row of block scores (the order of topk.hip: larger first, ties by ascending column), by
// a workgroup of four wavefronts; lane w of each gets mask word w.  Column 256 e + 64 wave + lane is key[e], as signed 16-bit
// integers: scores of Stage 1 are never negative but for -inf, so that is their order, and -32768, the bits of -0, which counts
// as +0, is free for "no column".  Whatever bits the row holds, a round finds its k-th column in the histogram or starts
// the next one 1023 keys further down: with a key on every column there are always k of them to find.
// Bound by the instructions a wavefront issues one after the other (a lone one needs five clocks for each), so it spends few of
// them per column: one histogram of the keys up to 1023 (eight powers of two) below the largest finite score, in LDS, two
// scans over the lanes find the k-th key and how many columns equal it.  Halving the 16 bits by counts took three times as
// long.  Every split of a row repeats this: as a launch of its own the selection took 3.2 us at 12 rows of 313 columns and
// 6.5 at 128 rows of 2048.
struct SelectScratch {
    uint32_t bins[512];                                        // two 16-bit counts each
    int2 tops[2][4];                                           // per wavefront: its largest key up to the limit, its columns above it
    uint32_t equal[32];
    uint64_t words[32];
};
constexpr int kNoColumn = -32768;

template <int kItems>
__device__ __forceinline__ uint64_t select_words(const elem_bits* row, int n, int cols, int k_want, SelectScratch& t, int tid, int wave, int lane) {
    int key[kItems];
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
        const int col = 256 * e + tid;
        key[e] = reinterpret_cast<const int16_t*>(row)[col < n ? col : 0];
    }
    *reinterpret_cast<uint2*>(&t.bins[2 * tid]) = make_uint2(0, 0);
    const int k = k_want < cols ? k_want : cols;
    if (k <= 0) return 0ull;                                   // uniform over the workgroup
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
        key[e] = key[e] == kNoColumn ? 0 : key[e];             // -0
        key[e] = 256 * e + tid < cols ? key[e] : kNoColumn;
    }
    int limit = kElemPosInf - 1, thr, c_above, c_equal;        // the forced blocks (+inf) stay above the histogram
    for (int round = 0;; ++round) {
        int top = kNoColumn, above = 0;
#pragma unroll
        for (int e = 0; e < kItems; ++e) {
            top = max(top, key[e] <= limit ? key[e] : kNoColumn);
            above += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key[e] > limit));
        }
        top = max(top, __builtin_amdgcn_update_dpp(top, top, 0xB1, 0xF, 0xF, false));      // a row's maximum: quad_perm,
        top = max(top, __builtin_amdgcn_update_dpp(top, top, 0x4E, 0xF, 0xF, false));
        top = max(top, __builtin_amdgcn_update_dpp(top, top, 0x124, 0xF, 0xF, false));     // row_ror 4, 8
        top = max(top, __builtin_amdgcn_update_dpp(top, top, 0x128, 0xF, 0xF, false));
        top = max(max(static_cast<int>(__builtin_amdgcn_readlane(top, 0)), static_cast<int>(__builtin_amdgcn_readlane(top, 16))),
                  max(static_cast<int>(__builtin_amdgcn_readlane(top, 32)), static_cast<int>(__builtin_amdgcn_readlane(top, 48))));
        if (lane == 0) t.tops[round & 1][wave] = make_int2(top, above);
        __syncthreads();
        const int2 t0 = t.tops[round & 1][0], t1 = t.tops[round & 1][1], t2 = t.tops[round & 1][2], t3 = t.tops[round & 1][3];
        top = __builtin_amdgcn_readfirstlane(max(max(t0.x, t1.x), max(t2.x, t3.x)));
        above = __builtin_amdgcn_readfirstlane(t0.y + t1.y + t2.y + t3.y);
        if (above >= k) { limit = 32767; continue; }           // only at first: no more than forced blocks are wanted
#pragma unroll
        for (int e = 0; e < kItems; ++e) {
            const int bin = min(top - key[e], 1023);
            if (key[e] <= limit && key[e] != kNoColumn) atomicAdd(&t.bins[bin >> 1], (bin & 1) ? 0x10000u : 1u);
        }
        __syncthreads();
        const uint4 a = *reinterpret_cast<const uint4*>(&t.bins[8 * lane]), b = *reinterpret_cast<const uint4*>(&t.bins[8 * lane + 4]);
        const uint32_t pairs = a.x + a.y + a.z + a.w + b.x + b.y + b.z + b.w;
        const int mine = static_cast<int>((pairs & 0xffffu) + (pairs >> 16));
        const int upto = scan_lanes(mine) + above;
        const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(upto >= k) | 1ull << 63);
        const int fine = lane < 16 ? static_cast<int>(reinterpret_cast<const uint16_t*>(t.bins)[16 * at + lane]) : 0;
        const int fine_upto = scan_lanes(fine) + static_cast<int>(__builtin_amdgcn_readlane(upto - mine, at));
        const int in = __builtin_ctzll(__builtin_amdgcn_ballot_w64(fine_upto >= k) | 1ull << 63) & 15;
        c_equal = __builtin_amdgcn_readlane(fine, in);
        c_above = static_cast<int>(__builtin_amdgcn_readlane(fine_upto, in)) - c_equal;
        thr = top - (16 * at + in);
        if (16 * at + in < 1023) break;
        limit = thr;                                           // the last bin holds everything further down: again from there
        __syncthreads();
        *reinterpret_cast<uint2*>(&t.bins[2 * tid]) = make_uint2(0, 0);
    }
    const int ties = k - c_above;                              // of the columns equal to thr, the first so many
    int equal_before = 0;                                      // lane w: those in the words before w
    if (ties < c_equal) {
#pragma unroll
        for (int e = 0; e < kItems; ++e) {
            const int c = __builtin_popcountll(__builtin_amdgcn_ballot_w64(key[e] == thr));
            if (lane == 0) t.equal[4 * e + wave] = c;
        }
        __syncthreads();
        const int c = lane < 4 * kItems ? static_cast<int>(t.equal[lane]) : 0;
        equal_before = scan_lanes(c) - c;
    }
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
        uint64_t take;
        if (ties < c_equal) {
            const uint64_t eq = __builtin_amdgcn_ballot_w64(key[e] == thr);
            const int rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(eq >> 32),
                                                       __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(eq), __builtin_amdgcn_readlane(equal_before, 4 * e + wave)));
            take = __builtin_amdgcn_ballot_w64(key[e] > thr || (key[e] == thr && rank < ties));
        } else {
            take = __builtin_amdgcn_ballot_w64(key[e] >= thr);
        }
        if (lane == 0) t.words[4 * e + wave] = take;
    }
    __syncthreads();
    return lane < 4 * kItems ? t.words[lane] : 0ull;
}

// kSelect (four wavefronts only): the selection is made here, from block scores
// Keep (four wavefronts only): a whole step that selects every block, so that nothing has to come before the attention.  One workgroup more per (sequence, KV
// head), or the last split's where that would be a second round, keeps the lengths and the compressed keys, which no other looks at; the new row is appended as
// above.  Steps of the layer in us, launches for the front, the scores, the attention and the merge | for the front, the attention and the merge | this and the
// merge, 2 KV heads, 64 blocks selected: one sequence of 4000 tokens 19.0 | 15.2 | 10.6 (all the host's), 16 of up to 4000 23.2 | 15.9 | 13.7, 32 of 2000 26.4 | 18.6 |
// 16.7 (with workgroups for the keepers alone 21.7), 64 of 1500 29.9 | 22.4 | 21.0 (27.4).
struct KeepStep {
    S1DecodeStep step;
    S1DecodeStrides strides;
};
__device__ __forceinline__ const KeepStep& step_of(const KeepStep& keep) { return keep; }
template <bool kDirect, int kWaves, bool kSelect, typename... Keep>
__global__ __launch_bounds__(64 * kWaves)
void decode_split_kernel(const DecodeParams p, const Keep... keep) {
    constexpr bool kKeep = sizeof...(Keep) == 1;
    static_assert(kWaves == 4 || !(kSelect || kKeep), "by four wavefronts");
    constexpr int kSlots = kWaves == 1 ? 2 : 1;                // block tiles per wavefront
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    __shared__ __attribute__((aligned(16))) elem_bits new_row[2 * kHeadDim];        // K, then V
    __shared__ uint4 turned_q[4][64];
    uint64_t* words = reinterpret_cast<uint64_t*>(smem + kWaves * kSlots * kSlotBytes);     // more than 64 mask words: the row's, clipped to the sequence
    warm_kernel_arguments<sizeof(DecodeParams)>();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    auto keep_caches = [&]() {
        if constexpr (kKeep) {
            const KeepStep& with = step_of(keep...);
            const S1DecodeStep& t = with.step;
            const int len = t.lens ? t.lens[b] : t.host_len;
            int add_f, add_c;
            const int rows_f = s1d_step_rows(len, t.capacity, t.kernel_f, t.stride_f, t.fine_capacity, add_f);
            const int rows_c = s1d_step_rows(len, t.capacity, t.kernel_c, t.stride_c, t.coarse_capacity, add_c);
            s1d_keep_caches(with.strides, t, b, h, len, rows_f, rows_c, add_f, add_c, tid, false, true, kHeadDim);
        }
    };
    if (kKeep && split == p.splits) {                          // uniform over the workgroup
        keep_caches();
        return;
    }
    unsigned char* tiles = smem + wave * kSlots * kSlotBytes;
    const int64_t pair = static_cast<int64_t>(b) * p.num_heads_k + h;
    const bool listed = kSelect || p.mask != nullptr || p.topk_idx != nullptr;      // else: every block
    uint64_t bits0 = 0ull;                                     // mask word `lane` of the row
    int first_idx = -1;                                        // or list entry `lane`
    if (!kSelect && p.mask != nullptr && lane < p.n64) bits0 = p.mask[pair * p.n64 + lane];
    if (!kSelect && p.topk_idx != nullptr && lane < p.k_idx) first_idx = p.topk_idx[pair * p.k_idx + lane];
    int without = 0;                                           // the length of a sequence where no lengths are given
    if constexpr (kKeep) without = step_of(keep...).step.host_len;
    else without = p.capacity - p.seqlen_new;
    const int seqlen = p.cache_seqlens ? p.cache_seqlens[b] : without;
    const int lp = p.leftpad ? p.leftpad[b] : 0;              // the sequence's key 0 is cache row lp
    // position of the first appended key; a full cache takes no key, and the tables need not reach beyond it
    const int rot_pos = !p.cache_seqlens ? 0 : (seqlen < p.capacity ? seqlen : p.capacity - 1);
    int L = seqlen + p.seqlen_new;
    if (L > p.capacity) L = p.capacity;
    L -= lp;                                                   // keys of the sequence; mask block j = keys 64 j ..
    const int new_key = (p.append_here && seqlen < p.capacity) ? seqlen - lp : -1;  // its index in the sequence
    const int last_blk = L <= 0 ? -1 : ((L - 1) >> 6);
    int n_words = last_blk < 0 ? 0 : (last_blk >> 6) + 1;
    if (listed && !kSelect && n_words > p.n64) n_words = p.n64;

    auto lds_fence = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    // The query and the new row (lanes 0..15: K, lanes 16..31: V, 16 bytes each).  The query is turned at the position of the
    // first appended key (flash_fwd_kernel.h:899-901), a quarter by each of four wavefronts: every one turning all of it for
    // itself pulled 100 KiB of tables and rows through the CU.
    elem8 qf[4];
    {
        const int qh = p.group * h + (n < p.group ? n : p.group - 1);      // rows beyond the group repeat its last head
        const elem_bits* qp = p.q + b * p.q_batch + qh * p.q_head;
        if (p.rotary_dim > 0) {
            constexpr int kOwn = 4 / kWaves;                   // 16-byte chunks of a lane's four that this wavefront turns
            RotaryChunk r[kOwn];
#pragma unroll
            for (int c = 0; c < kOwn; ++c) r[c] = rotary_request(p, qp, 4 * (wave * kOwn + c) + g, rot_pos);
#pragma unroll
            for (int c = 0; c < kOwn; ++c) turned_q[wave * kOwn + c][lane] = rotary_turn(p, r[c], 4 * (wave * kOwn + c) + g);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const elem8*>(qp + 8 * g + 32 * c);
        }
        if (p.append_here && wave == kWaves - 1 && g < 2) {
            const elem_bits* kvec = p.knew + b * p.kn_batch + h * p.kn_head;
            uint4 kept;
            if (g == 1) kept = *reinterpret_cast<const uint4*>(p.vnew + b * p.vn_batch + h * p.vn_head + n * 8);
            else kept = p.rotary_dim > 0 ? rotary_chunk(p, kvec, n, rot_pos) : *reinterpret_cast<const uint4*>(kvec + n * 8);
            *reinterpret_cast<uint4*>(new_row + g * kHeadDim + n * 8) = kept;
        }
        if (p.append_here || p.rotary_dim > 0) {
            if constexpr (kWaves > 1) __syncthreads();
            else lds_fence();
        }
        if (p.rotary_dim > 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const elem8*>(&turned_q[c][lane]);
        }
    }

    // ---- the selected blocks: words in LDS, how many there are, and which run of them is this wavefront's ----
    // bits of words w0 + lane, and how many bits lie in words up to and including this lane's, from word w0 on
    const uint64_t last_word_bits = (last_blk & 63) == 63 ? ~0ull : ((1ull << ((last_blk & 63) + 1)) - 1ull);
    auto mask_word = [&](int w) -> uint64_t {
        const uint64_t v = p.mask[pair * p.n64 + w];
        return w == (last_blk >> 6) ? v & last_word_bits : v;
    };
    const bool in_place = kWaves == 1 && p.mask_in_place && n_words > 64;           // uniform: more words than LDS holds
    auto scan_words = [&](int w0, uint64_t& bits) -> int {
        if (in_place) bits = w0 + lane < n_words ? mask_word(w0 + lane) : 0ull;
        else bits = w0 + lane < n_words ? words[w0 + lane] : 0ull;
        return scan_lanes(__builtin_popcountll(bits));
    };
    int total = 0, incl0 = 0;                                  // incl0, bits0: the first 64 words
    if constexpr (kSelect) {
        // blocks of the sequence only: the columns beyond them, if any, would lose to every one of them or be dropped
        int cols = last_blk + 1 < p.n_scores ? last_blk + 1 : p.n_scores;
        cols = __builtin_amdgcn_readfirstlane(cols < 0 ? 0 : cols);
        __shared__ __attribute__((aligned(16))) SelectScratch scratch_words;
        const elem_bits* row = p.scores + pair * p.n_scores;
        if (p.n_scores <= 512) bits0 = select_words<2>(row, p.n_scores, cols, p.k_select, scratch_words, tid, wave, lane);
        else bits0 = select_words<8>(row, p.n_scores, cols, p.k_select, scratch_words, tid, wave, lane);
        incl0 = scan_lanes(__builtin_popcountll(bits0));
        total = __builtin_amdgcn_readlane(incl0, 63);
        lds_fence();
    } else if (!listed) {
        total = last_blk + 1;
        if constexpr (kKeep) total = total < p.n_scores ? total : p.n_scores;      // a longer sequence than was announced
        lds_fence();
    } else {
        if (p.mask != nullptr && n_words <= 64) {              // straight into registers
            bits0 = lane < n_words ? (lane == (last_blk >> 6) ? bits0 & last_word_bits : bits0) : 0ull;
            incl0 = scan_lanes(__builtin_popcountll(bits0));
            lds_fence();
        } else {
            // words in LDS: up to 64 in the wavefront's own tile (no barrier), more in an area shared by the workgroup
            const bool shared = kWaves > 1 && n_words > 64;
            if (n_words <= 64) words = reinterpret_cast<uint64_t*>(tiles);
            const int first = shared ? tid : lane, step = shared ? 64 * kWaves : 64;
            auto words_fence = [&]() {
                if (shared) __syncthreads();
                else lds_fence();
            };
            if (p.mask != nullptr) {
                for (int w = in_place ? n_words : first; w < n_words; w += step) words[w] = mask_word(w);
            } else {
                for (int w = first; w < n_words; w += step) words[w] = 0ull;
                words_fence();
                for (int i = first; i < p.k_idx; i += step) {
                    const int j = i == lane ? first_idx : p.topk_idx[pair * p.k_idx + i];
                    if (j >= 0 && j <= last_blk && (j >> 6) < n_words)
                        atomicOr(reinterpret_cast<unsigned long long*>(&words[j >> 6]), 1ull << (j & 63));
                }
            }
            words_fence();
            incl0 = scan_words(0, bits0);
            for (int w0 = 64; w0 < n_words; w0 += 64) {
                uint64_t bits;
                total += __builtin_amdgcn_readlane(scan_words(w0, bits), 63);
            }
            lds_fence();
        }
        total += __builtin_amdgcn_readlane(incl0, 63);
    }
    // equal runs: their lengths differ by one at most
    const int runs = p.splits * kWaves, run = split * kWaves + wave;
    int each = static_cast<int>(static_cast<float>(total) * __builtin_amdgcn_rcpf(static_cast<float>(runs)));       // total / runs, off by one at most
    if (total >= 1 << 20) each = total / runs;                 // where it might be off by more; integer division is a long chain
    each = __builtin_amdgcn_readfirstlane(each);
    each += (each + 1) * runs <= total ? 1 : (each * runs > total ? -1 : 0);
    // So many runs take one block more, dealt out to the splits in turn: a CU's wavefronts share its bandwidth, and all of a split's four runs longer by one
    // were a workgroup that took a quarter longer (24 sequences x 2 heads, 64 blocks over 5 splits: whole paged step 45.0 -> 43.6 us).  Where
    // there are fewer blocks than runs the first runs take them: a row of a few blocks is then the same whatever the number of splits.
    const int longer = total - each * runs;
    const int every = kWaves == 1 ? 0 : (longer >= p.splits ? 1 : 0) + (longer >= 2 * p.splits ? 1 : 0) + (longer >= 3 * p.splits ? 1 : 0);    // of each split's
    const int over = longer - every * p.splits, mine_longer = every + (split < over ? 1 : 0);
    const int begin = each == 0 ? (run < longer ? run : longer) : run * each + split * every + (split < over ? split : over) + (wave < mine_longer ? wave : mine_longer);
    const int count = each + ((each == 0 ? run < longer : wave < mine_longer) ? 1 : 0);

    // Blocks [base, base + 64) of this run, one per lane, and the cache row (page) they lie in.
    const int cache_row = p.block_table ? 0 : (p.cache_batch_idx ? p.cache_batch_idx[b] : b);
    int my_block = 0, my_page = cache_row;
    auto look_up = [&](int base) {
        const int lo = begin + base, hi = begin + (count < base + 64 ? count : base + 64);   // ordinals of the row
        if (!listed) {
            my_block = lo + lane;
        } else {
            // by scalar instructions, a few per block: runs are short, and every lane's block would need as many
            int ord = lo, passed = 0;                          // passed: set bits of the words before w0
            for (int w0 = 0; ord < hi; w0 += 64) {             // hi <= total: some word holds the last one
                uint64_t bits = bits0;
                const int incl = w0 == 0 ? incl0 : scan_words(w0, bits);
                const int upto = passed + __builtin_amdgcn_readlane(incl, 63);
                uint64_t left = __builtin_amdgcn_ballot_w64(passed + incl > ord);  // words that still hold bits of the run
                while (ord < hi && ord < upto) {
                    const int w = __builtin_ctzll(left);
                    left &= left - 1ull;
                    const int w_upto = passed + __builtin_amdgcn_readlane(incl, w);
                    uint64_t v = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(bits >> 32), w))) << 32) |
                                 static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(bits), w));
                    const int skip = ord - (w_upto - static_cast<int>(__builtin_popcountll(v)));
                    if (skip > 0) v = drop_set_bits(v, skip);  // the run starts inside this word
                    for (; v != 0ull && ord < hi; v &= v - 1ull, ++ord)
                        my_block = lane == ord - lo ? (w0 + w) * 64 + __builtin_ctzll(v) : my_block;
                }
                passed = upto;
            }
        }
        if (p.block_table && base + lane < count) my_page = p.block_table[b * p.bt_batch + my_block * kBlockN / p.page_size];
    };
    if (count > 0) look_up(0);

    float m = -INFINITY, l = 0.f;
    floatx4 o[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};

    // ---- block i of the run into slot i % kSlots ----
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(decode_lds_address(tiles));
    const uint32_t k_pitch = static_cast<uint32_t>(p.kc_row) * 2u, v_pitch = static_cast<uint32_t>(p.vc_row) * 2u;   // bytes; not with far_rows
    uint32_t k_off[4], v_off[4];                               // this lane's piece of rows g, 4 + g, 8 + g, 12 + g
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        k_off[u] = (4 * u + g) * k_pitch + (n ^ tile_swizzle(4 * u + g)) * 16;
        v_off[u] = (4 * u + g) * v_pitch + (n ^ tile_swizzle(4 * u + g)) * 16;
    }
    // 16 DMA instructions for K or V of a block, which never straddles two pages (page_size is a multiple of 64 and paged
    // caches have no left padding)
    auto request_tile = [&](int i, const elem_bits* cache, int64_t batch_stride, int64_t row_stride, int64_t head_stride, uint32_t pitch,
                            const uint32_t (&off)[4], uint32_t tile) {
        const int jb = __builtin_amdgcn_readlane(my_block, i & 63), page = __builtin_amdgcn_readlane(my_page, i & 63);
        const int key0 = jb * kBlockN;
        const int64_t in_page = p.block_table ? key0 % p.page_size : lp + key0;
        const elem_bits* base = cache + page * batch_stride + in_page * row_stride + h * head_stride;
        uint32_t slot = lds0 + (kSlots == 2 ? i & 1 : 0) * kSlotBytes + tile;
        // the slot's previous tile has been read; and the sixteen addresses in it are no loop invariants worth a register each
        asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(slot) : : "memory");
        const int last = L - 1 - key0;
        if (p.far_rows) {
#pragma unroll 1
            for (int u = 0; u < 16; ++u) {
                const int row = 4 * u + g;
                decode_dma16(base + (row < last ? row : last) * row_stride + (n ^ tile_swizzle(row)) * 8, slot + u * 1024);
            }
        } else if (last >= kBlockN - 1) {
#pragma unroll
            for (int u = 0; u < 16; ++u) decode_dma16(base + (u >> 2) * 16 * row_stride, off[u & 3], slot + u * 1024);
        } else {
            // rows past the end are read from the last row (K is masked below, P is zero there); where that is the row being
            // appended, memory need not hold it yet and the tile is patched
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                int row = 4 * u + g;
                row = row < last ? row : last;
                decode_dma16(base, row * pitch + (n ^ tile_swizzle(4 * u + g)) * 16, slot + u * 1024);
            }
        }
    };
    auto request_k = [&](int i) { request_tile(i, p.kcache, p.kc_batch, p.kc_row, p.kc_head, k_pitch, k_off, 0); };
    auto request_v = [&](int i) { request_tile(i, p.vcache, p.vc_batch, p.vc_row, p.vc_head, v_pitch, v_off, kTileBytes); };
    // every ordinary load so far has to be back before the waits below count DMA loads only
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[c]));
    asm volatile("" : "+v"(my_page));
    if (count > 0) { request_k(0); request_v(0); }
    if (kSlots == 2 && count > 1) { request_k(1); request_v(1); }
    for (int i = 0; i < count; ++i) {
        // in flight, oldest first: K and V of this block, and with two slots K and V of the next one
        const bool ahead = kSlots == 2 && i + 1 < count && (i & 63) != 63;
        if (ahead) asm volatile("s_waitcnt vmcnt(48)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        const int j = __builtin_amdgcn_readlane(my_block, i & 63), key0 = j * kBlockN;
        unsigned char* ktile = tiles + (kSlots == 2 ? i & 1 : 0) * kSlotBytes;
        const bool patch = new_key >= key0 && new_key < key0 + kBlockN;            // uniform: the block of the row that is being appended
        // the new row, into the rows of K's tile (0) or V's (1) from its own up to `end`
        auto patch_rows = [&](int which, int end) {
            const uint4 kept = *reinterpret_cast<const uint4*>(new_row + which * kHeadDim + 8 * n);
            for (int r = new_key - key0 + g; r < end; r += 4)
                *reinterpret_cast<uint4*>(ktile + which * kTileBytes + r * 256 + (n ^ tile_swizzle(r)) * 16) = kept;
            lds_fence();
        };
        if (patch) patch_rows(0, new_key - key0 + 1);          // the keys behind it are masked
        floatx4 s[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            s[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const elem8 kf = *reinterpret_cast<const elem8*>(ktile + (16 * kt + n) * 256 + ((4 * c + g) ^ tile_swizzle(n)) * 16);
                s[kt] = IV2_MFMA(kf, qf[c], s[kt], 0, 0, 0);
            }
        }
        bool next_k = false;
        if (kSlots == 1 && i + 1 < count) {
            if ((i & 63) == 63) {                              // the looked-up blocks run out
                look_up(i + 1);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                asm volatile("" : "+v"(my_page));
            }
            request_k(i + 1);
            next_k = true;
        }
        const int lim = L - 1 - key0;                           // in-block index of the last valid key
        if (lim < kBlockN - 1) {
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (16 * kt + 4 * g + e > lim) s[kt][e] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[kt][e]);
        mx = wave_max_over_g(mx);
        const float m_new = fmaxf(m, mx * p.scale_log2);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);
        float rs = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float pv = __builtin_amdgcn_exp2f(s[kt][e] * p.scale_log2 - m_use);
                s[kt][e] = pv;
                rs += pv;
            }
        l = l * alpha + rs;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt] *= alpha;
        elem8 pf[2];
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pf[cc][e] = static_cast<elem_t>(s[2 * cc][e]);
                pf[cc][4 + e] = static_cast<elem_t>(s[2 * cc + 1][e]);
            }
        if (ahead) asm volatile("s_waitcnt vmcnt(32)" ::: "memory");
        else if (next_k) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (patch) patch_rows(1, kBlockN);                     // P is zero behind it, and 0 x what unwritten memory holds may be NaN
        // A operand of O^T += V^T P^T: lane (n, g) needs V[32 cc + 4 g + {0..3}, 32 cc + 16 + 4 g + {0..3}][16 dt + n], the
        // keys in the order in which the lane holds P.  One transposing read hands a lane four rows' worth of one
        // column: within 16 lanes, lane i offers the four columns 16 dt + 4 (i % 4) .. of key 4 g + i / 4 (+ 32 cc),
        // and lane n receives column 16 dt + n of the keys 4 g + {0, 1, 2, 3}.
        const int vrow = 4 * g + (n >> 2);                     // + 16, 32, 48: the same swizzle
        const unsigned char* vtile = ktile + kTileBytes + vrow * 256 + (n & 1) * 8;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            const int piece = ((2 * dt + ((n & 3) >> 1)) ^ tile_swizzle(vrow)) * 16;
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                const short4d lo = lds_read_tr(reinterpret_cast<const elem_bits*>(vtile + (32 * cc) * 256 + piece));
                const short4d hi = lds_read_tr(reinterpret_cast<const elem_bits*>(vtile + (32 * cc + 16) * 256 + piece));
                elem8 vf;
                __builtin_memcpy(&vf, &lo, 8);
                __builtin_memcpy(reinterpret_cast<unsigned char*>(&vf) + 8, &hi, 8);
                o[dt] = IV2_MFMA(vf, pf[cc], o[dt], 0, 0, 0);
            }
        }
        if (kSlots == 1) {
            if (next_k) request_v(i + 1);
        } else if ((i & 63) + 2 >= 64 && i + 1 < count) {      // the looked-up blocks run out: drain, look up, start again
            if ((i & 63) == 63) {
                look_up(i + 1);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                asm volatile("" : "+v"(my_page));
                request_k(i + 1); request_v(i + 1);
                if (i + 2 < count) { request_k(i + 2); request_v(i + 2); }
            }
        } else if (i + 2 < count) {                            // into the slot that has just been read
            request_k(i + 2); request_v(i + 2);
        }
    }

    if (p.append_here && split == 0 && wave == 0 && seqlen < p.capacity && g < 2) {
        const int64_t at = g == 0 ? cache_row_offset(p, b, seqlen, p.kc_batch, p.kc_row) + h * p.kc_head
                                  : cache_row_offset(p, b, seqlen, p.vc_batch, p.vc_row) + h * p.vc_head;
        *reinterpret_cast<uint4*>((g == 0 ? p.kcache : p.vcache) + at + 8 * n) = *reinterpret_cast<const uint4*>(new_row + g * kHeadDim + 8 * n);
    }
    const float l_tot = wave_sum_over_g(l);
    const int64_t slot = pair * p.splits + split;
    const float no_keys = kDirect ? INFINITY : -INFINITY;
    if constexpr (kWaves > 1) {
        // merge of the wavefronts' (m, l, O): each leaves its own in its tile, then 16 threads per head, 8 columns each
        __shared__ float merge_m[kWaves][16], merge_l[kWaves][16];
        float* mine = reinterpret_cast<float*>(tiles) + n * kMergePitch + 4 * g;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<floatx4*>(mine + 16 * dt) = o[dt];
        if (g == 0) { merge_m[wave][n] = m; merge_l[wave][n] = l_tot; }
        __syncthreads();
        for (int t = tid; t < 256; t += 64 * kWaves) {
            const int head = t >> 4, col = (t & 15) * 8;
            float top = -INFINITY;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) top = fmaxf(top, merge_m[w][head]);
            const float ref = top == -INFINITY ? 0.f : top;
            float sum = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const float f = __builtin_amdgcn_exp2f(merge_m[w][head] - ref);
                const float* theirs = reinterpret_cast<const float*>(smem + w * kSlots * kSlotBytes) + head * kMergePitch + col;
                sum += f * merge_l[w][head];
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[e] += f * theirs[e];
            }
            const float inv = sum > 0.f ? 1.f / sum : 0.f;
            const float lse = sum > 0.f ? top * 0.69314718055994530942f + logf(sum) : no_keys;
            if (kDirect) {
                if (head >= p.group) continue;
                *reinterpret_cast<uint4*>(p.out + b * p.o_batch + (p.group * h + head) * p.o_head + col) =
                    make_uint4(pack_elem2(acc[0] * inv, acc[1] * inv), pack_elem2(acc[2] * inv, acc[3] * inv),
                               pack_elem2(acc[4] * inv, acc[5] * inv), pack_elem2(acc[6] * inv, acc[7] * inv));
                if (col == 0) p.lse[static_cast<int64_t>(b) * p.num_heads_k * p.group + p.group * h + head] = lse;
            } else {
                if (col == 0) p.lse_part[slot * 16 + head] = lse;
                float* op = p.o_part + (slot * 16 + head) * kHeadDim + col;        // LSE -inf: the combine kernel does not use it
                *reinterpret_cast<float4*>(op) = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
                *reinterpret_cast<float4*>(op + 4) = make_float4(acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv);
            }
        }
        if (kKeep && static_cast<int>(gridDim.x) == p.splits && split == p.splits - 1) keep_caches();      // no workgroup of their own
        return;
    }
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const float lse = l_tot > 0.f ? m * 0.69314718055994530942f + logf(l_tot) : no_keys;
    if (kDirect) {
        if (n >= p.group) return;
        elem_bits* op = p.out + b * p.o_batch + (p.group * h + n) * p.o_head + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            uint2 w;
            w.x = pack_elem2(o[dt][0] * inv, o[dt][1] * inv);
            w.y = pack_elem2(o[dt][2] * inv, o[dt][3] * inv);
            *reinterpret_cast<uint2*>(op + 16 * dt) = w;
        }
        if (g == 0) p.lse[static_cast<int64_t>(b) * p.num_heads_k * p.group + p.group * h + n] = lse;
    } else {
        if (g == 0) p.lse_part[slot * 16 + n] = lse;
        if (count <= 0) return;                                // LSE -inf: the combine kernel does not use the partial
        float* op = p.o_part + (slot * 16 + n) * kHeadDim + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
            *reinterpret_cast<float4*>(op + 16 * dt) = make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    }
}

// Merge of the per-split partials: one wavefront per (sequence, query head), lane l holds columns 2 l and 2 l + 1 and,
// for the weights, split l.  kMax >= splits: the loads are unrolled (beyond the last split the last one is read again),
// so every partial is requested before the first is used.  A wavefront per head keeps the merge of 64 splits at one
// round trip; one workgroup per KV head pulled 16 times as much through one CU.
// What it spends is latency: its arguments in one cache line, reductions over the lanes by DPP (12 exchanges through LDS took 0.55 us of its 2.4).
constexpr int kCombineWaves = 4;
struct CombineParams {
    const float* o_part;
    const float* lse_part;
    elem_bits* out;
    float* lse;
    int64_t o_batch, o_head;
    int num_heads_k, splits, group;
};
template <int kMax>
__global__ __launch_bounds__(64 * kCombineWaves)
void decode_combine_kernel(const CombineParams p) {
    const int lane = threadIdx.x & 63;
    const int head = blockIdx.x * kCombineWaves + (threadIdx.x >> 6);
    const int h = blockIdx.y, b = blockIdx.z;
    if (head >= p.group) return;                               // partial rows that only filled the MFMA tile
    const int64_t slot0 = (static_cast<int64_t>(b) * p.num_heads_k + h) * p.splits;
    float2 part[kMax];
    const float lse = lane < p.splits ? p.lse_part[(slot0 + lane) * 16 + head] : -INFINITY;
#pragma unroll
    for (int s = 0; s < kMax; ++s)
        part[s] = *reinterpret_cast<const float2*>(p.o_part + ((slot0 + (s < p.splits ? s : p.splits - 1)) * 16 + head) * kHeadDim + 2 * lane);
    // exchanges by 1, 2, 4 and 8 lanes (4 and 8 as mirrors: by then every quad, every eight lanes agree), and between rows where splits reach beyond one
    auto over_splits = [&](float x, auto both) {
        x = both(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0xB1, 0xF, 0xF, false)));
        x = both(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x4E, 0xF, 0xF, false)));
        x = both(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x141, 0xF, 0xF, false)));
        x = both(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x140, 0xF, 0xF, false)));
        if constexpr (kMax > 16) {
            float mine, other;
            row_pair_xor16(x, mine, other);
            x = both(mine, other);
            row_pair_xor32(x, mine, other);
            x = both(mine, other);
        } else {
            x = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
        }
        return x;
    };
    const float mx = over_splits(lse, [](float x, float y) { return fmaxf(x, y); });
    const float w = lse == -INFINITY ? 0.f : expf(lse - mx);   // a split without blocks has no partial
    const float wsum = over_splits(w, [](float x, float y) { return x + y; });
    float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
    for (int s = 0; s < kMax; ++s) {
        const float ws = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s));
        acc0 += ws != 0.f ? ws * part[s].x : 0.f;              // what a split without blocks left in memory may be anything
        acc1 += ws != 0.f ? ws * part[s].y : 0.f;
    }
    const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
    reinterpret_cast<uint32_t*>(p.out + b * p.o_batch + (p.group * h + head) * p.o_head)[lane] = pack_elem2(acc0 * inv, acc1 * inv);
    if (lane == 0)
        p.lse[static_cast<int64_t>(b) * p.num_heads_k * p.group + p.group * h + head] = wsum > 0.f ? mx + logf(wsum) : INFINITY;
}

}  // namespace IV2_NS

using namespace IV2_NS;

// Up to so many workgroups a launch takes the four-wavefront form of the split kernel: one on every CU.
constexpr int kGroupedWorkgroups = 256;

#ifndef IV2_F16        // element-type independent: defined once
extern "C" int infllmv2_fwd_kvcache_num_splits(int batch, int num_heads_k, int requested) {
    if (requested > 0) return requested > 64 ? 64 : requested;
    // What fills 256 CUs once, with the four-wavefront workgroups (one per CU) as long as every (sequence, KV head) gets one
    // of them, with the single-wavefront ones (two per CU) beyond; one more and a second, nearly empty round follows.  More
    // than 16 partials cost the merge more than the shorter runs gain.
    const int pairs = batch * num_heads_k > 0 ? batch * num_heads_k : 1;
    const int fit = kGroupedWorkgroups / pairs;
    if (fit >= 1) return fit > 16 ? 16 : fit;
    return 512 / pairs > 1 ? 512 / pairs : 1;
}
#endif

static size_t decode_partials_bytes(int batch, int num_heads_k, int num_splits) {
    if (num_splits <= 1) return 0;
    return static_cast<size_t>(batch) * num_heads_k * num_splits * 16 * (kHeadDim + 1) * sizeof(float);
}

#ifndef IV2_F16        // both element types are 2 bytes wide: defined once
extern "C" size_t infllmv2_fwd_kvcache_workspace_bytes(int batch, int num_heads_k, int num_splits) {
    return decode_partials_bytes(batch, num_heads_k, num_splits);
}
#endif

static int fwd_kvcache_impl(void* stream, const void* q, void* kcache, void* vcache, const void* k_new,
                                    const void* v_new, const int32_t* cache_seqlens, void* out, float* softmax_lse,
                                    const uint64_t* blockmask, const int32_t* topk_idx, int k_idx, const void* scores, int n_scores,
                                    int k_select, void* workspace, size_t workspace_bytes, int batch,
                                    int seqlen_q, int num_heads, int num_heads_k, int head_dim, int cache_capacity,
                                    int seqlen_new, const int64_t* q_strides, const int64_t* kcache_strides,
                                    const int64_t* vcache_strides, const int64_t* knew_strides,
                                    const int64_t* vnew_strides, const int64_t* o_strides, int n_uint64_per_row,
                                    int num_splits, float softmax_scale, const int32_t* cache_batch_idx,
                                    const int32_t* cache_leftpad, const int32_t* block_table,
                                    int64_t block_table_batch_stride, int page_block_size, const void* rotary_cos,
                                    const void* rotary_sin, int rotary_dim, int rotary_interleaved, const KeepStep* keep = nullptr) {
    IV2_CHECK(head_dim == kHeadDim, "fwd_kvcache: this build only supports head_dim 128 (got %d)", head_dim);
    IV2_CHECK(seqlen_q == 1, "fwd_kvcache: this build only supports one query token per sequence (got %d)", seqlen_q);
    IV2_CHECK(valid_group(num_heads, num_heads_k),
              "fwd_kvcache: requires num_heads == g * num_heads_k with g in {1, 2, 4, 8, 16} (got %d and %d)", num_heads, num_heads_k);
    IV2_CHECK(batch > 0 && cache_capacity > 0, "fwd_kvcache: batch size and cache capacity must be positive");
    IV2_CHECK(batch <= 65535 && num_heads_k <= 65535, "fwd_kvcache: batch and num_heads_k must not exceed 65535");
    IV2_CHECK(q && kcache && vcache && out && softmax_lse, "fwd_kvcache: null pointer");
    IV2_CHECK((k_new == nullptr) == (v_new == nullptr), "fwd_kvcache: k and v must be given together");
    IV2_CHECK(k_new == nullptr || seqlen_new > 0, "fwd_kvcache: new keys given with seqlen_new == 0");
    IV2_CHECK(blockmask == nullptr || n_uint64_per_row > 0, "fwd_kvcache: mask given without words per row");
    IV2_CHECK(softmax_scale > 0.f, "fwd_kvcache: softmax_scale must be positive");
    IV2_CHECK(num_splits >= 1 && num_splits <= 64, "fwd_kvcache: num_splits must be in [1, 64]");
    IV2_CHECK(workspace_bytes >= infllmv2_fwd_kvcache_workspace_bytes(batch, num_heads_k, num_splits),
              "fwd_kvcache: workspace too small");
    IV2_CHECK(workspace != nullptr || num_splits == 1, "fwd_kvcache: split decode needs a workspace");
    IV2_CHECK(blockmask == nullptr || topk_idx == nullptr, "fwd_kvcache: give the selection as a mask or as indices, not both");
    IV2_CHECK(topk_idx == nullptr || k_idx >= 0, "fwd_kvcache: negative number of indices");
    IV2_CHECK(block_table == nullptr || cache_batch_idx == nullptr, "Paged KVcache does not support cache_batch_idx");
    IV2_CHECK(block_table == nullptr || cache_leftpad == nullptr,
              "We don't support Paged KV and leftpad_k running at the same time yet");
    IV2_CHECK(block_table == nullptr || (page_block_size > 0 && page_block_size % kBlockN == 0 && block_table_batch_stride > 0),
              "fwd_kvcache: the page size of a paged KV cache must be a positive multiple of 64 (got %d)", page_block_size);
    IV2_CHECK((rotary_cos == nullptr) == (rotary_sin == nullptr), "If rotary cos is provided, rotary sin must also be provided");
    IV2_CHECK(rotary_cos == nullptr || k_new != nullptr,
              "If rotary cos/sin are provided, new key / value to be appended to KV cache must also be provided");
    IV2_CHECK(rotary_cos == nullptr || (rotary_dim > 0 && rotary_dim <= head_dim), "rotary_dim must be <= headdim");
    IV2_CHECK(rotary_cos == nullptr || rotary_dim % 16 == 0, "Only rotary dimensions divisible by 16 are currently supported");
    IV2_CHECK(rotary_cos == nullptr || (reinterpret_cast<uintptr_t>(rotary_cos) % 2 == 0 && reinterpret_cast<uintptr_t>(rotary_sin) % 2 == 0),
              "fwd_kvcache: rotary tables must be 2-byte aligned");
    const void* aligned16[] = {q, kcache, vcache, out};
    for (const void* a : aligned16) IV2_CHECK(reinterpret_cast<uintptr_t>(a) % 16 == 0, "fwd_kvcache: tensors must be 16-byte aligned");
    IV2_CHECK(q_strides[0] % 8 == 0 && q_strides[1] % 8 == 0 && o_strides[0] % 8 == 0 && o_strides[1] % 8 == 0,
              "fwd_kvcache: q/out strides must be multiples of 8 elements");
    for (int s = 0; s < 3; ++s)
        IV2_CHECK(kcache_strides[s] % 8 == 0 && vcache_strides[s] % 8 == 0, "fwd_kvcache: cache strides must be multiples of 8 elements");

    DecodeParams p{};
    // a lane's offset inside a block is a 32-bit operand wherever it fits: up to 62 rows, or 15 and a piece of one
    const auto far = [](int64_t row_stride) { return row_stride < 0 || row_stride >= (1 << 24); };
    p.far_rows = far(kcache_strides[1]) || far(vcache_strides[1]) ? 1 : 0;
    p.q = static_cast<const elem_bits*>(q);
    p.kcache = static_cast<elem_bits*>(kcache);
    p.vcache = static_cast<elem_bits*>(vcache);
    p.knew = static_cast<const elem_bits*>(k_new);
    p.vnew = static_cast<const elem_bits*>(v_new);
    p.out = static_cast<elem_bits*>(out);
    p.lse = softmax_lse;
    p.cache_seqlens = cache_seqlens;
    p.mask = blockmask;
    p.q_batch = q_strides[0]; p.q_head = q_strides[1];
    p.o_batch = o_strides[0]; p.o_head = o_strides[1];
    p.kc_batch = kcache_strides[0]; p.kc_row = kcache_strides[1]; p.kc_head = kcache_strides[2];
    p.vc_batch = vcache_strides[0]; p.vc_row = vcache_strides[1]; p.vc_head = vcache_strides[2];
    p.batch = batch; p.num_heads_k = num_heads_k; p.capacity = cache_capacity;
    p.group = num_heads / num_heads_k;
    p.seqlen_new = k_new ? seqlen_new : 0;
    p.n64 = n_uint64_per_row; p.splits = num_splits;
    p.scale_log2 = softmax_scale * 1.44269504088896340736f;
    p.cache_batch_idx = cache_batch_idx; p.leftpad = cache_leftpad;
    p.block_table = block_table; p.bt_batch = block_table_batch_stride; p.page_size = block_table ? page_block_size : 1;
    p.rot_cos = static_cast<const elem_bits*>(rotary_cos); p.rot_sin = static_cast<const elem_bits*>(rotary_sin);
    p.rotary_dim = rotary_cos ? rotary_dim : 0; p.rotary_interleaved = rotary_interleaved;
    p.topk_idx = topk_idx; p.k_idx = k_idx;
    p.scores = static_cast<const elem_bits*>(scores); p.n_scores = n_scores; p.k_select = k_select;
    if (topk_idx != nullptr) p.n64 = ((cache_capacity + kBlockN - 1) / kBlockN + 63) / 64;
    // mask words of one row, kept in LDS beside the tiles; 8192 words are 33 million tokens, 2048 still fit beside four tiles
    constexpr size_t kMaxWords = 8192;
    size_t words = (blockmask || topk_idx) ? ((static_cast<size_t>(cache_capacity) + kBlockN - 1) / kBlockN + 63) / 64 : 0;
    IV2_CHECK(words <= kMaxWords || topk_idx == nullptr, "fwd_kvcache_topk: a cache of %d rows needs more mask words than the kernel holds", cache_capacity);
    if (words > kMaxWords) {
        p.mask_in_place = 1;
        words = 0;
    }
    const int64_t pairs = static_cast<int64_t>(batch) * num_heads_k;
    const bool grouped = pairs * num_splits <= kGroupedWorkgroups && words <= 2048 && !p.mask_in_place;
    IV2_CHECK(keep == nullptr || grouped, "decode_step_all: at most %d (sequence, KV head, split) triples are served", kGroupedWorkgroups);
    IV2_CHECK(scores == nullptr || (grouped && n_scores > 0 && n_scores <= INFLLMV2_DECODE_MAX_SCORES && k_select > 0),
              "fwd_kvcache_scores: 1 to %d block scores per row, topk >= 1 and at most %d (sequence, KV head, split) triples are served",
              INFLLMV2_DECODE_MAX_SCORES, kGroupedWorkgroups);
    const size_t lds = (grouped ? 4 : 2) * static_cast<size_t>(kSlotBytes) + words * sizeof(uint64_t);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (k_new != nullptr) {
        IV2_CHECK(reinterpret_cast<uintptr_t>(k_new) % 16 == 0 && reinterpret_cast<uintptr_t>(v_new) % 16 == 0,
                  "fwd_kvcache: new k/v must be 16-byte aligned");
        for (int s = 0; s < 3; ++s)
            IV2_CHECK(knew_strides[s] % 8 == 0 && vnew_strides[s] % 8 == 0, "fwd_kvcache: new k/v strides must be multiples of 8 elements");
        p.kn_batch = knew_strides[0]; p.kn_row = knew_strides[1]; p.kn_head = knew_strides[2];
        p.vn_batch = vnew_strides[0]; p.vn_row = vnew_strides[1]; p.vn_head = vnew_strides[2];
        // one new row at a known place: the split kernel takes care of it (one launch less, and no wait for it)
        p.append_here = seqlen_new == 1 && (cache_seqlens != nullptr || keep != nullptr) ? 1 : 0;
        if (!p.append_here) {
            const int64_t total = static_cast<int64_t>(batch) * seqlen_new * num_heads_k * 16;
            hipLaunchKernelGGL(decode_append_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, st, p);
            IV2_LAUNCH_CHECK();
        }
    }
    if (num_splits > 1) {
        float* ws = static_cast<float*>(workspace);
        p.o_part = ws;
        p.lse_part = ws + static_cast<size_t>(batch) * num_heads_k * num_splits * 16 * kHeadDim;
    }
    auto launch = [&](auto kernel, int workgroups, const auto&... with) -> int {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        IV2_CHECK(e == hipSuccess, "fwd_kvcache: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        hipLaunchKernelGGL(kernel, dim3(workgroups, num_heads_k, batch), dim3(grouped ? 256 : 64), lds, st, p, with...);
        IV2_LAUNCH_CHECK();
        return 0;
    };
    int rc;
    if (keep != nullptr) rc = launch(num_splits == 1 ? decode_split_kernel<true, 4, false, KeepStep> : decode_split_kernel<false, 4, false, KeepStep>,
                                     num_splits + (pairs * (num_splits + 1) <= kGroupedWorkgroups ? 1 : 0), *keep);
    else if (scores != nullptr) rc = launch(num_splits == 1 ? decode_split_kernel<true, 4, true> : decode_split_kernel<false, 4, true>, num_splits);
    else if (grouped) rc = launch(num_splits == 1 ? decode_split_kernel<true, 4, false> : decode_split_kernel<false, 4, false>, num_splits);
    else rc = launch(num_splits == 1 ? decode_split_kernel<true, 1, false> : decode_split_kernel<false, 1, false>, num_splits);
    if (rc != 0) return rc;
    if (num_splits > 1) {
        const CombineParams c{p.o_part, p.lse_part, p.out, p.lse, p.o_batch, p.o_head, num_heads_k, num_splits, p.group};
        const dim3 cgrid((p.group + kCombineWaves - 1) / kCombineWaves, num_heads_k, batch), cblock(64 * kCombineWaves);
        if (num_splits <= 4) hipLaunchKernelGGL(decode_combine_kernel<4>, cgrid, cblock, 0, st, c);
        else if (num_splits <= 16) hipLaunchKernelGGL(decode_combine_kernel<16>, cgrid, cblock, 0, st, c);
        else hipLaunchKernelGGL(decode_combine_kernel<64>, cgrid, cblock, 0, st, c);
        IV2_LAUNCH_CHECK();
    }
    return 0;
}

extern "C" int IV2_ENTRY(infllmv2_fwd_kvcache)(void* stream, const void* q, void* kcache, void* vcache, const void* k_new,
                                    const void* v_new, const int32_t* cache_seqlens, void* out, float* softmax_lse,
                                    const uint64_t* blockmask, void* workspace, size_t workspace_bytes, int batch,
                                    int seqlen_q, int num_heads, int num_heads_k, int head_dim, int cache_capacity,
                                    int seqlen_new, const int64_t* q_strides, const int64_t* kcache_strides,
                                    const int64_t* vcache_strides, const int64_t* knew_strides,
                                    const int64_t* vnew_strides, const int64_t* o_strides, int n_uint64_per_row,
                                    int num_splits, float softmax_scale, const int32_t* cache_batch_idx,
                                    const int32_t* cache_leftpad, const int32_t* block_table,
                                    int64_t block_table_batch_stride, int page_block_size, const void* rotary_cos,
                                    const void* rotary_sin, int rotary_dim, int rotary_interleaved) {
    return fwd_kvcache_impl(stream, q, kcache, vcache, k_new, v_new, cache_seqlens, out, softmax_lse, blockmask, nullptr, 0, nullptr, 0, 0,
                            workspace, workspace_bytes, batch, seqlen_q, num_heads, num_heads_k, head_dim, cache_capacity, seqlen_new,
                            q_strides, kcache_strides, vcache_strides, knew_strides, vnew_strides, o_strides,
                            n_uint64_per_row, num_splits, softmax_scale, cache_batch_idx, cache_leftpad, block_table,
                            block_table_batch_stride, page_block_size, rotary_cos, rotary_sin, rotary_dim,
                            rotary_interleaved);
}

extern "C" int IV2_ENTRY(infllmv2_fwd_kvcache_topk)(void* stream, const void* q, void* kcache, void* vcache, const void* k_new,
                                         const void* v_new, const int32_t* cache_seqlens, void* out, float* softmax_lse,
                                         const int32_t* topk_idx, int k_idx, void* workspace, size_t workspace_bytes, int batch,
                                         int seqlen_q, int num_heads, int num_heads_k, int head_dim, int cache_capacity,
                                         int seqlen_new, const int64_t* q_strides, const int64_t* kcache_strides,
                                         const int64_t* vcache_strides, const int64_t* knew_strides,
                                         const int64_t* vnew_strides, const int64_t* o_strides,
                                         int num_splits, float softmax_scale, const int32_t* cache_batch_idx,
                                         const int32_t* cache_leftpad, const int32_t* block_table,
                                         int64_t block_table_batch_stride, int page_block_size, const void* rotary_cos,
                                         const void* rotary_sin, int rotary_dim, int rotary_interleaved) {
    IV2_CHECK(topk_idx != nullptr, "fwd_kvcache_topk: null pointer");
    return fwd_kvcache_impl(stream, q, kcache, vcache, k_new, v_new, cache_seqlens, out, softmax_lse, nullptr, topk_idx, k_idx, nullptr, 0, 0,
                            workspace, workspace_bytes, batch, seqlen_q, num_heads, num_heads_k, head_dim, cache_capacity,
                            seqlen_new, q_strides, kcache_strides, vcache_strides, knew_strides, vnew_strides, o_strides, 0,
                            num_splits, softmax_scale, cache_batch_idx, cache_leftpad, block_table, block_table_batch_stride,
                            page_block_size, rotary_cos, rotary_sin, rotary_dim, rotary_interleaved);
}

extern "C" int IV2_ENTRY(infllmv2_fwd_kvcache_scores)(void* stream, const void* q, void* kcache, void* vcache, const int32_t* cache_seqlens,
                                         void* out, float* softmax_lse, const void* scores, int n_scores, int topk, void* workspace,
                                         size_t workspace_bytes, int batch, int num_heads, int num_heads_k, int head_dim,
                                         int cache_capacity, const int64_t* q_strides, const int64_t* kcache_strides,
                                         const int64_t* vcache_strides, const int64_t* o_strides, int num_splits, float softmax_scale) {
    IV2_CHECK(scores != nullptr, "fwd_kvcache_scores: null pointer");
    const int64_t none[3] = {0, 0, 0};
    return fwd_kvcache_impl(stream, q, kcache, vcache, nullptr, nullptr, cache_seqlens, out, softmax_lse, nullptr, nullptr, 0, scores,
                            n_scores, topk, workspace, workspace_bytes, batch, 1, num_heads, num_heads_k, head_dim, cache_capacity, 0,
                            q_strides, kcache_strides, vcache_strides, none, none, o_strides, 0, num_splits, softmax_scale, nullptr,
                            nullptr, nullptr, 0, 0, nullptr, nullptr, 0, 0);
}

extern "C" int IV2_ENTRY(infllmv2_decode_step_all)(void* stream, const void* q, const void* k_new, const void* v_new, void* kcache, void* vcache,
                                      void* fine_cache, void* coarse_cache, const int32_t* lens, int host_len, int32_t* new_lens,
                                      int32_t* fine_lens, int32_t* coarse_lens, void* out, float* softmax_lse, void* workspace, size_t workspace_bytes,
                                      int batch, int num_heads, int num_heads_k, int head_dim, int capacity, int fine_rows, int coarse_rows, int max_len,
                                      const int64_t* q_strides, const int64_t* knew_strides, const int64_t* vnew_strides, const int64_t* kcache_strides,
                                      const int64_t* vcache_strides, const int64_t* fine_strides, const int64_t* coarse_strides, const int64_t* o_strides,
                                      int kernel_size_f, int stride_f, int kernel_size_c, int stride_c, int num_splits, float softmax_scale) {
    const char* who = "decode_step_all";
    IV2_CHECK(k_new && v_new && fine_cache && coarse_cache && fine_lens && coarse_lens, "%s: null pointer", who);
    IV2_CHECK(fine_rows > 0 && coarse_rows > 0 && max_len > 0 && host_len >= 0, "%s: bad sizes", who);
    IV2_CHECK(kernel_size_f > 0 && stride_f > 0 && kernel_size_c > 0 && stride_c > 0, "%s: kernel_size and stride must be positive", who);
    IV2_CHECK(reinterpret_cast<uintptr_t>(fine_cache) % 16 == 0 && reinterpret_cast<uintptr_t>(coarse_cache) % 16 == 0, "%s: tensors must be 16-byte aligned", who);
    for (int s = 0; s < 3; ++s)
        IV2_CHECK(fine_strides[s] % 8 == 0 && coarse_strides[s] % 8 == 0, "%s: strides must be multiples of 8 elements", who);
    KeepStep keep{};
    S1DecodeStep& t = keep.step;
    t.knew = static_cast<const elem_bits*>(k_new);
    t.vnew = static_cast<const elem_bits*>(v_new);
    t.kcache = static_cast<elem_bits*>(kcache);
    t.vcache = static_cast<elem_bits*>(vcache);
    t.fine = static_cast<elem_bits*>(fine_cache);
    t.coarse = static_cast<elem_bits*>(coarse_cache);
    t.kn_batch = knew_strides[0]; t.kn_head = knew_strides[1]; t.vn_batch = vnew_strides[0]; t.vn_head = vnew_strides[1];
    t.kc_batch = kcache_strides[0]; t.kc_row = kcache_strides[1]; t.kc_head = kcache_strides[2];
    t.vc_batch = vcache_strides[0]; t.vc_row = vcache_strides[1]; t.vc_head = vcache_strides[2];
    t.lens = lens; t.host_len = host_len;
    t.new_lens = new_lens; t.fine_lens = fine_lens; t.coarse_lens = coarse_lens;
    t.capacity = capacity; t.fine_capacity = fine_rows; t.coarse_capacity = coarse_rows;
    t.kernel_f = kernel_size_f; t.stride_f = stride_f; t.kernel_c = kernel_size_c; t.stride_c = stride_c;
    keep.strides = {fine_strides[0], fine_strides[1], fine_strides[2], coarse_strides[0], coarse_strides[1], coarse_strides[2]};
    const int64_t kn[3] = {knew_strides[0], 0, knew_strides[1]}, vn[3] = {vnew_strides[0], 0, vnew_strides[1]};     // of the one row
    return fwd_kvcache_impl(stream, q, kcache, vcache, k_new, v_new, lens, out, softmax_lse, nullptr, nullptr, 0, nullptr,
                            (max_len + kBlockN - 1) / kBlockN, 0, workspace, workspace_bytes, batch, 1, num_heads, num_heads_k, head_dim, capacity, 1, q_strides,
                            kcache_strides, vcache_strides, kn, vn, o_strides, 0, num_splits, softmax_scale, nullptr, nullptr, nullptr, 0, 0, nullptr, nullptr,
                            0, 0, &keep);
}

#ifndef IV2_F16        // one such entry point in the library: bfloat16 only
// ---- decode for callers that cannot allocate ---------------------------------------------------------------------
//
// The split partials live in a device array that belongs to the library's code object: every GPU
// the library runs on holds one copy of it, at its own address, from module load to process end.  `scratch` below is
// only the host-side handle of that array; the device address is looked up once per device with
// hipGetSymbolAddress and is what the kernels get.  Nothing in the array has to start at zero: every (sequence, KV
// head, split) workgroup writes its log-sum-exp record, and its partial unless it has no block, which the record then says, before
// the combine kernel reads them.  All calls on one GPU share the array, so calls that overlap on one GPU (two streams, two
// threads) race; calls on one stream are ordered by the stream.
static __device__ __align__(256) unsigned char scratch[INFLLMV2_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

extern "C" int infllmv2_fwd_kvcache_static(void* stream, const void* q, void* kcache, void* vcache, const void* k_new,
                                           const void* v_new, const int32_t* cache_seqlens, void* out,
                                           float* softmax_lse, const uint64_t* blockmask, int batch, int seqlen_q,
                                           int num_heads, int num_heads_k, int head_dim, int cache_capacity,
                                           int seqlen_new, const int64_t* q_strides, const int64_t* kcache_strides,
                                           const int64_t* vcache_strides, const int64_t* knew_strides,
                                           const int64_t* vnew_strides, const int64_t* o_strides, int n_uint64_per_row,
                                           int num_splits, float softmax_scale, const int32_t* cache_batch_idx,
                                           const int32_t* cache_leftpad, const int32_t* block_table,
                                           int64_t block_table_batch_stride, int page_block_size,
                                           const void* rotary_cos, const void* rotary_sin, int rotary_dim,
                                           int rotary_interleaved) {
    IV2_CHECK(batch > 0 && num_heads_k > 0 && num_splits >= 1 && num_splits <= 64,
              "fwd_kvcache_static: batch, num_heads_k must be positive and num_splits in [1, 64]");
    const size_t need = infllmv2_fwd_kvcache_workspace_bytes(batch, num_heads_k, num_splits);
    IV2_CHECK(need <= static_cast<size_t>(INFLLMV2_STATIC_SCRATCH_BYTES),
              "fwd_kvcache_static: batch %d x %d KV heads x %d splits needs %zu bytes of scratch, the built-in buffer holds %zu; "
              "use fewer splits or infllmv2_fwd_kvcache with a workspace", batch, num_heads_k, num_splits, need,
              static_cast<size_t>(INFLLMV2_STATIC_SCRATCH_BYTES));
    // the copy of the array that belongs to the GPU the stream runs on (the null stream: the current device); the
    // symbol lookup below answers for the current device, so the two must be the same
    int dev = -1, stream_dev = -1;
    hipError_t e = hipGetDevice(&dev);
    IV2_CHECK(e == hipSuccess && dev >= 0 && dev < kMaxDevices, "fwd_kvcache_static: hipGetDevice failed or device index %d out of range", dev);
    if (stream != nullptr) {
        e = hipStreamGetDevice(static_cast<hipStream_t>(stream), &stream_dev);
        IV2_CHECK(e == hipSuccess, "fwd_kvcache_static: hipStreamGetDevice failed: %s", hipGetErrorString(e));
        IV2_CHECK(stream_dev == dev, "fwd_kvcache_static: the stream belongs to device %d but the current device is %d; "
                  "make the stream's device current before the call", stream_dev, dev);
    }
    void* ws = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        if (g_scratch_ptr[dev] == nullptr) {
            void* sym = nullptr;
            e = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));           // this device's copy of the array
            IV2_CHECK(e == hipSuccess && sym != nullptr, "fwd_kvcache_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            g_scratch_ptr[dev] = sym;
        }
        ws = g_scratch_ptr[dev];
    }
    return fwd_kvcache_impl(stream, q, kcache, vcache, k_new, v_new, cache_seqlens, out, softmax_lse, blockmask, nullptr, 0, nullptr, 0, 0, ws,
                            static_cast<size_t>(INFLLMV2_STATIC_SCRATCH_BYTES), batch, seqlen_q, num_heads, num_heads_k,
                            head_dim, cache_capacity, seqlen_new, q_strides, kcache_strides, vcache_strides, knew_strides,
                            vnew_strides, o_strides, n_uint64_per_row, num_splits, softmax_scale, cache_batch_idx,
                            cache_leftpad, block_table, block_table_batch_stride, page_block_size, rotary_cos, rotary_sin,
                            rotary_dim, rotary_interleaved);
}
#endif
