// Stage-1 scoring for decode on gfx950: ONE query token per sequence, a batch of sequences, each scored against
// its own compressed keys.
//
// Same arithmetic and rules as stage1.hip (compute_attn_1rowblock_splitkv_stage1,
// csrc/flash_attn/src/flash_fwd_kernel.h:1203-1744; Mask::apply_mask_stage1, mask.h:225-319; hdim16_reduce,
// flash_fwd_kernel.h:53-112) for a sequence with q_len == 1:
//   vis_s = L for a non-causal launch, clamp(L - 1, 0, L) for a causal one (mask.h:273-281 with i = 0, q_len = 1)
//   lse_g = log sum_{c < vis_c} exp(scale * q_g . kc_c)
//   score[h, b, j] = bf16( sum_g exp(scale * q_g . kf_j - lse_g) )  for j < vis_f, else 0; all 0 when vis_c == 0
// and, with pooling, the max-pooling rule of csrc/max_pooling_1d.cuh:12-160 applied to that row.
//
// Shape of the work: per sequence and KV head the whole compressed-key set is read once (256 bytes per key) for 16
// query rows, so the launch is bound by memory bandwidth and the stage1.hip kernel (one workgroup per 16 tokens,
// keys staged for reuse by 16 tokens) is the wrong shape: it would stream every sequence through one workgroup.
// Here the keys of one (sequence, KV head) are cut into runs of 64-key tiles, the same run length (one or two tiles unless
// the longest sequence would then need more than 64 runs) for every sequence of the batch, and every run goes to a
// wavefront of its own that loads its tiles straight into MFMA operand registers: long sequences get many
// workgroups, short ones few, and every workgroup carries the same load.
// The log-sum-exp needs all coarse keys before any score can be normalised, so there are two launches:
//   1. stage1_decode_lse_kernel: per run of coarse tiles the running (max, sum) of the 16 heads -> workspace;
//   2. stage1_decode_score_kernel: merges the partials of its (sequence, head) (16 lanes in parallel), then scores its run of
//      fine tiles and writes either the score row or its pooling onto key blocks.  A pooled block needs the last
//      key of the tile before the run: that one 16-key group is scored again by the run that needs it (same MFMA,
//      same operands, same bits).
// Few and short sequences take one launch instead, in which every workgroup forms the log-sum-exp for itself (stage1_decode_whole_kernel): the same bits.
// Keys can be packed (cu_seqlens) or lie in per-sequence caches (batch stride + lengths).
#include "common.h"
#include "decode_step.h"
#include "infllmv2_hip.h"
#include <math.h>
#include <type_traits>

namespace IV2_NS {

struct S1DecodeParams {
    const elem_bits* q;
    const elem_bits* k;              // fine compressed keys
    const elem_bits* c;              // coarse compressed keys (the key set of the log-sum-exp)
    elem_bits* out;
    float* partial;                  // (batch, Hk, splits_c, 32): log2-domain max of the 16 heads, then their sums
    const int* cu_seqlens_q;         // null: sequence b's query is row b
    const int* cu_seqlens_k;         // packed keys: rows [cu[b], cu[b+1]); null: cache layout, k_lens[b] rows at b * k_batch
    const int* k_lens;
    const int* cu_seqlens_c;
    const int* c_lens;
    int64_t q_tok_stride, q_grp_stride, q_kvh_stride;
    int64_t k_batch_stride, k_row_stride, k_head_stride;
    int64_t c_batch_stride, c_row_stride, c_head_stride;
    int64_t out_head_stride, out_row_stride;
    int cols;                        // score columns to define per row (max_seqlen_k)
    float scale_log2;
    int causal;
    int group;                       // query heads per KV head, 1..16: MFMA rows >= group repeat head group - 1 and add nothing
    int splits_c, splits_f;          // runs the longest sequence is cut into (grid size; record slots per pair)
    int run_c, run_f;                // tiles per run
    // pooled output
    const int* cache_lens;           // per sequence, or null: cache_len for all
    int cache_len;
    int pool_len, local_blocks, init_blocks;
};

__device__ __forceinline__ int s1d_visible(int s, int L, bool causal) {
    if (!causal) return L;
    // mask.h:273-281 for token 0 of a 1-token query: (0+1)/s - 1 + L - (1 - s + 1)/s, C++ truncating divisions
    int v = 1 / s - 1 + L - (2 - s) / s;
    v = v < 0 ? 0 : v;
    return v < L ? v : L;
}

struct S1DecodeSeq {
    int q_row, Sq, Lk, Lc;
    const elem_bits* kbase;
    const elem_bits* cbase;
};

__device__ __forceinline__ S1DecodeSeq s1d_sequence(const S1DecodeParams& p, int b, int h) {
    S1DecodeSeq s;
    if (p.cu_seqlens_q) { s.q_row = p.cu_seqlens_q[b]; s.Sq = p.cu_seqlens_q[b + 1] - s.q_row; }
    else { s.q_row = b; s.Sq = 1; }
    int64_t koff, coff;
    if (p.cu_seqlens_k) { const int k0 = p.cu_seqlens_k[b]; s.Lk = p.cu_seqlens_k[b + 1] - k0; koff = k0 * p.k_row_stride; }
    else { s.Lk = p.k_lens[b]; koff = b * p.k_batch_stride; }
    if (p.cu_seqlens_c) { const int c0 = p.cu_seqlens_c[b]; s.Lc = p.cu_seqlens_c[b + 1] - c0; coff = c0 * p.c_row_stride; }
    else { s.Lc = p.c_lens[b]; coff = b * p.c_batch_stride; }
    s.kbase = p.k + koff + h * p.k_head_stride;
    s.cbase = p.c + coff + h * p.c_head_stride;
    return s;
}

// 64 keys x 128 d as MFMA B operands: register kt*4 + c of lane (n, g) = K[key0 + 16 kt + n][32 c + 8 g ..].
// Rows past the last key read the last key (finite values that every consumer masks).
__device__ __forceinline__ void s1d_load_tile(elem8 (&t)[16], const elem_bits* base, int64_t row_stride, int key0,
                                              int L, int n, int g) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        int row = key0 + 16 * kt + n;
        row = row < L ? row : L - 1;
        const elem_bits* src = base + row * row_stride + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[kt * 4 + c] = *reinterpret_cast<const elem8*>(src + 32 * c);
    }
}

__device__ __forceinline__ void s1d_load_q(elem8 (&qf)[4], const S1DecodeParams& p, const S1DecodeSeq& s, int h, int n, int g) {
    const elem_bits* qp = p.q + static_cast<int64_t>(s.q_row) * p.q_tok_stride + h * p.q_kvh_stride + (n < p.group ? n : p.group - 1) * p.q_grp_stride + 8 * g;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const elem8*>(qp + 32 * c);
}

// run [t0, t1) of `tiles` tiles that split `split` works on: runs of `per` tiles, the same length for every sequence
// of the batch (a long sequence has many runs, a short one few: every wavefront gets the same amount of work)
__device__ __forceinline__ void s1d_run_fixed(int tiles, int per, int split, int& t0, int& t1) {
    t0 = split * per;
    t0 = t0 < tiles ? t0 : tiles;
    t1 = t0 + per;
    t1 = t1 < tiles ? t1 : tiles;
}
__device__ __forceinline__ float s1d_quad_xor1(float x) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ float s1d_quad_xor2(float x) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x4E, 0xF, 0xF, false));
}
// maximum and sum over the 16 lanes of a row, by DPP operands of the operations themselves (quad_perm, row_ror)
__device__ __forceinline__ float s1d_row_max(float x) {
    x = fmaxf(x, s1d_quad_xor1(x));
    x = fmaxf(x, s1d_quad_xor2(x));
    x = fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x124, 0xF, 0xF, false)));
    return fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x128, 0xF, 0xF, false)));
}
__device__ __forceinline__ float s1d_row_sum(float x) {
    x += s1d_quad_xor1(x);
    x += s1d_quad_xor2(x);
    x += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x124, 0xF, 0xF, false));
    return x + __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x128, 0xF, 0xF, false));
}
// Running (max, sum) in log2 units of head 4g + e over the keys == n (mod 16) of the coarse tiles seen so far: tile ti's are added.
__device__ __forceinline__ void s1d_lse_tile(const S1DecodeParams& p, const elem8 (&qf)[4], const elem8 (&t)[16], int ti, int vis_c, int n,
                                             float (&m)[4], float (&l)[4]) {
    floatx4 s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        s[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) s[kt] = IV2_MFMA(qf[c], t[kt * 4 + c], s[kt], 0, 0, 0);
    }
    const bool cut = (ti + 1) * 64 > vis_c;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) v[kt] = s[kt][e] * p.scale_log2;
        if (cut) {
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) v[kt] = (ti * 64 + kt * 16 + n < vis_c) ? v[kt] : -INFINITY;
        }
        const float mx = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
        const float m_new = fmaxf(m[e], mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        float acc = l[e] * __builtin_amdgcn_exp2f(m[e] - m_use);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) acc += __builtin_amdgcn_exp2f(v[kt] - m_use);
        l[e] = acc;
        m[e] = m_new;
    }
}
// ... merged over the 16 key-column lanes: every lane of row g gets the values of its four heads
__device__ __forceinline__ void s1d_lse_close(const float (&m)[4], const float (&l)[4], float (&m_out)[4], float (&l_out)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        m_out[e] = s1d_row_max(m[e]);
        l_out[e] = s1d_row_sum(l[e] * __builtin_amdgcn_exp2f(m[e] - (m_out[e] == -INFINITY ? 0.f : m_out[e])));
    }
}
// Both over the coarse tiles [t0, t1) of one sequence and KV head.  patch(tile registers, tile) runs after a tile is requested.
template <typename Patch>
__device__ __forceinline__ void s1d_lse_run(const S1DecodeParams& p, const S1DecodeSeq& sq, const elem8 (&qf)[4], int vis_c,
                                            int t0, int t1, int n, int g, float (&m_out)[4], float (&l_out)[4], Patch patch) {
    float m[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) { m[e] = -INFINITY; l[e] = 0.f; }
    elem8 ta[16], tb[16];
    auto load = [&](elem8 (&t)[16], int ti) {
        s1d_load_tile(t, sq.cbase, p.c_row_stride, ti * 64, sq.Lc, n, g);
        patch(t, ti);
    };
    if (t0 < t1) load(ta, t0);
    if (t0 + 1 < t1) load(tb, t0 + 1);
    for (int ti = t0; ti < t1; ti += 2) {
        s1d_lse_tile(p, qf, ta, ti, vis_c, n, m, l);
        if (ti + 2 < t1) load(ta, ti + 2);
        if (ti + 1 < t1) {
            s1d_lse_tile(p, qf, tb, ti + 1, vis_c, n, m, l);
            if (ti + 3 < t1) load(tb, ti + 3);
        }
    }
    s1d_lse_close(m, l, m_out, l_out);
}

// The partial records {max x 16, sum x 16} of one (sequence, head) as a lane needs them: lane (n, g) takes the records
// n, n + 16, n + 32, n + 48 (at most 64 runs) for its four heads, two 16-byte loads per record.  The number of loads
// does not depend on the data (an index beyond the last record reads the last one again and is ignored later), so that
// the loads requested after these can stay in flight while these are waited for.
struct S1DRecords {
    floatx4 m[4], l[4];
};
__device__ __forceinline__ void s1d_load_records(S1DRecords& r, const float* part, int count, int n, int g) {
    auto fetch = [&](int k) {
        int s = n + 16 * k;
        s = s < count ? s : count - 1;
        r.m[k] = *reinterpret_cast<const floatx4*>(part + s * 32 + 4 * g);
        r.l[k] = *reinterpret_cast<const floatx4*>(part + s * 32 + 16 + 4 * g);
    };
    fetch(0);
    if (count > 16) {                                          // uniform
#pragma unroll
        for (int k = 1; k < 4; ++k) fetch(k);
    }
}
// log-sum-exp (log2 units) of head 4g + e from those records: the row's maximum, then the sum of everything relative to it
// (every lane of a row ends with the same bits).
__device__ __forceinline__ void s1d_merge_records(const S1DRecords& r, int count, int n, int g, int group, float (&lse2)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float mm = n < count ? r.m[0][e] : -INFINITY;          // a record that is not there is the neutral element
        if (count > 16) {                                      // uniform
#pragma unroll
            for (int k = 1; k < 4; ++k) mm = n + 16 * k < count ? fmaxf(mm, r.m[k][e]) : mm;
        }
        mm = s1d_row_max(mm);
        const float mu = mm == -INFINITY ? 0.f : mm;
        float ll = n < count ? r.l[0][e] * __builtin_amdgcn_exp2f(r.m[0][e] - mu) : 0.f;
        if (count > 16) {
#pragma unroll
            for (int k = 1; k < 4; ++k) ll += n + 16 * k < count ? r.l[k][e] * __builtin_amdgcn_exp2f(r.m[k][e] - mu) : 0.f;
        }
        lse2[e] = mm + __builtin_amdgcn_logf(s1d_row_sum(ll));   // v_log_f32 is log2
        if (4 * g + e >= group) lse2[e] = INFINITY;              // a row that only fills the tile adds exp2(x - inf) = 0
    }
}

__device__ __forceinline__ void s1d_store_record(const S1DecodeParams& p, int b, int h, int split, const float (&m)[4], const float (&l)[4],
                                                 int n, int g) {
    float* slot = p.partial + ((static_cast<int64_t>(b) * gridDim.y + h) * p.splits_c + split) * 32;
    if (n != 0) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) { slot[4 * g + e] = m[e]; slot[16 + 4 * g + e] = l[e]; }
}

// Two wavefronts per workgroup, a run each: see the front kernel below.
constexpr int kLseWaves = 2;
__global__ __launch_bounds__(64 * kLseWaves)
void stage1_decode_lse_kernel(const S1DecodeParams p) {
    warm_kernel_arguments<sizeof(S1DecodeParams)>();
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int split = blockIdx.x * kLseWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = blockIdx.y, b = blockIdx.z;
    const S1DecodeSeq sq = s1d_sequence(p, b, h);
    if (sq.Sq <= 0) return;
    const int s1 = (sq.Lk == sq.Lc) ? 16 : 64;                 // flash_fwd_kernel.h:1236-1240
    const int vis_c = s1d_visible(s1, sq.Lc, p.causal != 0);
    int t0, t1;
    s1d_run_fixed((vis_c + 63) >> 6, p.run_c, split, t0, t1);
    if (t0 >= t1 && split > 0) return;                         // beyond this sequence's runs; run 0 always leaves a record
    elem8 qf[4];
    s1d_load_q(qf, p, sq, h, n, g);
    float mm[4], ll[4];
    s1d_lse_run(p, sq, qf, vis_c, t0, t1, n, g, mm, ll, [](elem8 (&)[16], int) {});
    s1d_store_record(p, b, h, split, mm, ll, n, g);
}

// ---- the front of a decode step -------------------------------------------------------------------------------------
// One launch appends the new token to the K/V caches, extends the two compressed-key caches where the token completes a
// window, and leaves the log-sum-exp records of the coarse keys (the launch above).  Per (sequence, KV head): one
// workgroup per coarse run, and one that keeps the caches.  Nothing waits for another workgroup: the run that holds a
// coarse key completed by this very token computes it itself (128 rows of K, of which the newest comes from the
// caller), writes it to its cache and uses it from LDS; the fine key is used by the next launch only.  As launches of their own
// the lengths, the append, the compressed keys and the records were six.
__device__ __forceinline__ S1DecodeStrides s1d_strides(const S1DecodeParams& p) {
    return {p.k_batch_stride, p.k_row_stride, p.k_head_stride, p.c_batch_stride, p.c_row_stride, p.c_head_stride};
}

__global__ __launch_bounds__(64 * kLseWaves)
void stage1_decode_front_kernel(const S1DecodeParams p, const S1DecodeStep t) {
    __shared__ __attribute__((aligned(16))) elem_bits newest_key[kHeadDim];         // the coarse key this token completes
    warm_kernel_arguments<sizeof(S1DecodeParams) + sizeof(S1DecodeStep)>();
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int first = (static_cast<int>(blockIdx.x) - 1) * kLseWaves, h = blockIdx.y, b = blockIdx.z;
    const int len = t.lens ? t.lens[b] : t.host_len;
    int add_f, add_c;
    const int rows_f = s1d_step_rows(len, t.capacity, t.kernel_f, t.stride_f, t.fine_capacity, add_f);
    const int rows_c = s1d_step_rows(len, t.capacity, t.kernel_c, t.stride_c, t.coarse_capacity, add_c);
    if (first < 0) {                                           // the caches' keepers
        s1d_keep_caches(s1d_strides(p), t, b, h, len, rows_f, rows_c, add_f, add_c, tid, true, !t.with_scores, 0);
        return;
    }
    const int tiles = (rows_c + 63) >> 6, split = first + wave;
    if (first * p.run_c >= tiles && first > 0) return;         // beyond this sequence's runs; run 0 always leaves a record
    int t0, t1;
    s1d_run_fixed(tiles, p.run_c, split, t0, t1);
    S1DecodeSeq sq;
    sq.q_row = b; sq.Sq = 1; sq.Lk = rows_f; sq.Lc = rows_c;
    sq.kbase = nullptr;
    sq.cbase = p.c + b * p.c_batch_stride + h * p.c_head_stride;
    elem8 qf[4];
    s1d_load_q(qf, p, sq, h, n, g);
    // uniform over the workgroup; add_c is the last key
    const bool adds = add_c >= 0 && (add_c >> 6) >= first * p.run_c && (add_c >> 6) < (first + kLseWaves) * p.run_c;
    if (adds) {
        const elem_bits mean = s1d_window_mean(t, b, h, add_c, t.kernel_c, t.stride_c, tid);
        t.coarse[b * p.c_batch_stride + add_c * p.c_row_stride + h * p.c_head_stride + tid] = mean;
        newest_key[tid] = mean;
        __syncthreads();
    }
    if (t0 >= t1 && split > 0) return;
    float mm[4], ll[4];
    s1d_lse_run(p, sq, qf, rows_c, t0, t1, n, g, mm, ll, [&](elem8 (&tile)[16], int ti) {
        if (!adds || ti != add_c >> 6) return;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
            if (ti * 64 + 16 * kt + n >= add_c) {              // the last key, and the lanes beyond it that repeat it
#pragma unroll
                for (int c = 0; c < 4; ++c) tile[kt * 4 + c] = *reinterpret_cast<const elem8*>(newest_key + 32 * c + 8 * g);
            }
    });
    s1d_store_record(p, b, h, split, mm, ll, n, g);
}

__device__ __forceinline__ float s1d_fold_rows16(float x, float y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float s1d_fold_rows32(float x, float y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The 16 keys before tile t0 (the last group of tile t0 - 1), whose last key opens the first pooling window of a run
// that does not start the row; with t0 == 0 the request goes to the row's first keys and is ignored.
__device__ __forceinline__ void s1d_load_group_before(elem8 (&t4)[4], const S1DecodeSeq& sq, int64_t row_stride, int t0, int n, int g) {
    int row = (t0 > 0 ? t0 * 64 - 16 : 0) + n;
    row = row < sq.Lk ? row : sq.Lk - 1;
    const elem_bits* src = sq.kbase + row * row_stride + 8 * g;
#pragma unroll
    for (int c = 0; c < 4; ++c) t4[c] = *reinterpret_cast<const elem8*>(src + 32 * c);
}

// Scores (or pooled block scores) of the fine tiles [t0, t1) of one sequence and KV head, by one wavefront; ta / tb
// hold tiles t0 and t0 + 1 already and before4 the 16 keys before tile t0 (all requested by the caller before it
// waited for the log-sum-exp).
template <bool kPool>
__device__ __forceinline__ void s1d_score_run(const S1DecodeParams& p, const S1DecodeSeq& sq, const elem8 (&qf)[4],
                                              const float (&lse2)[4], const elem8 (&before4)[4], elem8 (&ta)[16], elem8 (&tb)[16], int vis_f,
                                              int tiles, int t0, int t1, bool owns_tail, int b, int h, int lane) {
    const int n = lane & 15, g = lane >> 4;
    const int64_t out_row = static_cast<int64_t>(h) * p.out_head_stride + static_cast<int64_t>(sq.q_row) * p.out_row_stride;
    elem_bits* out = p.out + out_row;
    const int bq = kPool ? ((p.cache_lens ? p.cache_lens[b] : p.cache_len) / kBlockN) : 0;   // the query's own key block
    const int Lk_cols = sq.Lk < p.cols ? sq.Lk : p.cols;
    auto pool_rest = [&](int kb, float reached) -> elem_bits {
        const bool forced = (kb < p.init_blocks) || (bq >= kb && bq <= kb + p.local_blocks);
        const int first = kb * 4 - 1;
        const bool empty = (first < 0 ? 0 : first) >= Lk_cols;
        return forced ? kElemPosInf : (empty ? kElemNegInf : f32_to_elem_hw(reached));
    };
    // one 16-key group: this lane's four heads summed for key 16 kt + n of the tile
    auto group_part = [&](const elem8* t4) -> float {
        floatx4 s = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) s = IV2_MFMA(qf[c], t4[c], s, 0, 0, 0);
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += __builtin_amdgcn_exp2f(s[e] * p.scale_log2 - lse2[e]);
        return sum;
    };

    float carry = 0.f;                                         // score of the last key before the current tile
    if (kPool && t0 > 0 && t0 < t1) {
        const float part3 = group_part(before4);               // keys of the last group of tile t0 - 1: all exist
        float prev = s1d_fold_rows32(s1d_fold_rows16(0.f, 0.f), s1d_fold_rows16(0.f, part3));
        prev = (t0 * 64 - 64 + lane < vis_f) ? prev : 0.f;
        carry = __shfl(prev, 63);
    }

    auto consume = [&](const elem8 (&t)[16], int ti) {
        float part[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) part[kt] = group_part(&t[kt * 4]);
        const int col = ti * 64 + lane;                        // lane 16 g + n <-> key 16 g + n of the tile
        float mine = s1d_fold_rows32(s1d_fold_rows16(part[0], part[1]), s1d_fold_rows16(part[2], part[3]));
        mine = (col < vis_f) ? mine : 0.f;
        if (!kPool) {
            if (col < p.cols) out[col] = f32_to_elem_hw(mine);
        } else {
            float left = __shfl_up(mine, 1);
            if (lane == 0) left = carry;
            carry = __shfl(mine, 63);
            float best = fmaxf(mine, s1d_quad_xor1(mine));
            best = fmaxf(best, s1d_quad_xor2(best));
            best = fmaxf(best, left);
            const int kb = col >> 2;
            if ((lane & 3) == 0 && kb < p.pool_len) out[kb] = pool_rest(kb, best);
        }
    };

    for (int ti = t0; ti < t1; ti += 2) {
        consume(ta, ti);
        if (ti + 2 < t1) s1d_load_tile(ta, sq.kbase, p.k_row_stride, (ti + 2) * 64, sq.Lk, n, g);
        if (ti + 1 < t1) {
            consume(tb, ti + 1);
            if (ti + 3 < t1) s1d_load_tile(tb, sq.kbase, p.k_row_stride, (ti + 3) * 64, sq.Lk, n, g);
        }
    }
    if (owns_tail) {                                           // columns no tile covers
        if (!kPool) {
            for (int col = tiles * 64 + lane; col < p.cols; col += 64) out[col] = 0;
        } else {
            // the first of them still sees the last key of the last tile
            for (int kb = tiles * 16 + lane; kb < p.pool_len; kb += 64) out[kb] = pool_rest(kb, kb == tiles * 16 ? carry : 0.f);
        }
    }
}

// visible fine keys and tiles of a sequence (0 when no coarse key is visible: early exit of flash_fwd_kernel.h:1271-1276)
template <bool kPool>
__device__ __forceinline__ void s1d_fine_extent(const S1DecodeParams& p, const S1DecodeSeq& sq, int& vis_c, int& vis_f, int& tiles) {
    const int s1 = (sq.Lk == sq.Lc) ? 16 : 64;                 // flash_fwd_kernel.h:1236-1240
    vis_c = s1d_visible(s1, sq.Lc, p.causal != 0);
    vis_f = vis_c == 0 ? 0 : s1d_visible(16, sq.Lk, p.causal != 0);
    if (kPool && vis_f > p.cols) vis_f = p.cols;               // the score row the pooling would have read ends there
    tiles = (vis_f + 63) >> 6;
}

template <bool kPool>
__global__ __launch_bounds__(64)
void stage1_decode_score_kernel(const S1DecodeParams p) {
    warm_kernel_arguments<sizeof(S1DecodeParams)>();
    const int lane = threadIdx.x, n = lane & 15, g = lane >> 4;
    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const S1DecodeSeq sq = s1d_sequence(p, b, h);
    if (sq.Sq <= 0) return;
    int vis_c, vis_f, tiles;
    s1d_fine_extent<kPool>(p, sq, vis_c, vis_f, tiles);
    int t0, t1;
    s1d_run_fixed(tiles, p.run_f, split, t0, t1);
    const bool owns_tail = tiles == 0 ? split == 0 : (t0 < t1 && t1 == tiles);
    if (t0 >= t1 && !owns_tail) return;

    // Everything this run reads is requested before anything waits on memory, in the order in which it is needed:
    // the partial records of the log-sum-exp (merged while the keys are still on their way), the query, two tiles.
    // A run has one or two tiles (more only when a sequence has over 128 of them); a second one is requested wherever runs
    // may have two (the first again where this run has one), so that the number of requests in flight is known.
    int records = (((vis_c + 63) >> 6) + p.run_c - 1) / p.run_c;                    // the coarse runs of this sequence
    records = records < 1 ? 1 : records;
    S1DRecords rec;
    elem8 qf[4], before4[4], ta[16], tb[16];
    float lse2[4] = {0.f, 0.f, 0.f, 0.f};
    if (t0 < t1) {                                             // uniform; otherwise this run only fills the row's tail
        s1d_load_records(rec, p.partial + (static_cast<int64_t>(b) * gridDim.y + h) * p.splits_c * 32, records, n, g);
        s1d_load_q(qf, p, sq, h, n, g);
        if (kPool) s1d_load_group_before(before4, sq, p.k_row_stride, t0, n, g);
        s1d_load_tile(ta, sq.kbase, p.k_row_stride, t0 * 64, sq.Lk, n, g);
        if (p.run_f > 1) s1d_load_tile(tb, sq.kbase, p.k_row_stride, (t0 + 1 < t1 ? t0 + 1 : t0) * 64, sq.Lk, n, g);
        s1d_merge_records(rec, records, n, g, p.group, lse2);
    }
    s1d_score_run<kPool>(p, sq, qf, lse2, before4, ta, tb, vis_f, tiles, t0, t1, owns_tail, b, h, lane);
}


// One tile's results: lane l brings the score of key l (pooled: and the last key before the tile), the row's last tile also fills the columns behind it.
template <bool kPool>
__device__ __forceinline__ void s1d_store_tile(const S1DecodeParams& p, const S1DecodeSeq& sq, float mine, float carry, int vis_f, int tiles, int ti, bool live,
                                               bool owns_tail, int b, int h, int lane) {
    elem_bits* out = p.out + static_cast<int64_t>(h) * p.out_head_stride + static_cast<int64_t>(sq.q_row) * p.out_row_stride;
    if constexpr (!kPool) {
        if (owns_tail)
            for (int col = tiles * 64 + lane; col < p.cols; col += 64) out[col] = 0;
    } else {
        const int bq = (p.cache_lens ? p.cache_lens[b] : p.cache_len) / kBlockN;
        const int Lk_cols = sq.Lk < p.cols ? sq.Lk : p.cols;
        auto pool_rest = [&](int kb, float reached) -> elem_bits {
            const bool forced = (kb < p.init_blocks) || (bq >= kb && bq <= kb + p.local_blocks);
            const int first = kb * 4 - 1;
            const bool empty = (first < 0 ? 0 : first) >= Lk_cols;
            return forced ? kElemPosInf : (empty ? kElemNegInf : f32_to_elem_hw(reached));
        };
        float left = __shfl_up(mine, 1);
        if (lane == 0) left = carry;
        float best = fmaxf(mine, s1d_quad_xor1(mine));
        best = fmaxf(best, s1d_quad_xor2(best));
        best = fmaxf(best, left);
        const int kb = ti * 16 + (lane >> 2);
        if (live && (lane & 3) == 0 && kb < p.pool_len) out[kb] = pool_rest(kb, best);
        if (owns_tail) {
            const float last = live ? __shfl(mine, 63) : 0.f;
            for (int k = tiles * 16 + lane; k < p.pool_len; k += 64) out[k] = pool_rest(k, k == tiles * 16 ? last : 0.f);
        }
    }
}

// Both halves in one launch, for few and short sequences: a workgroup per fine tile, of four wavefronts, forms the log-sum-exp of its sequence and KV head for
// itself.  The coarse tiles go round the wavefronts, their records through LDS; then a wavefront scores 16 keys of the fine tile, and the last one
// also the key before it that opens the tile's first pooling window.  The time is a chain of round trips: arguments and lengths 0.8 us, the keys 1.4 to 2.7
// (112 KiB through one CU with four coarse tiles), records, merge and scores 1.5; which launches: s1d_whole.
// kStep: and the rest of the front of a decode step (above).  The keys this very token completes are not read from the caches, which a workgroup of this launch
// is writing: a workgroup that needs one forms it itself.
constexpr int kWholeWaves = 4;
constexpr int kWholeWindow = 128;                              // rows of a coarse window at most
constexpr int kWholeRecords = 8;                               // coarse tiles at most (s1d_whole takes fewer)
struct S1DecodeNoStep {};

template <bool kPool, typename Step>
__global__ __launch_bounds__(64 * kWholeWaves)
void stage1_decode_whole_kernel(const S1DecodeParams p, const Step t) {
    constexpr bool kStep = !std::is_same<Step, S1DecodeNoStep>::value;
    __shared__ __attribute__((aligned(16))) float records[kWholeRecords * 32];
    __shared__ float score[64];                                // of the tile's keys
    __shared__ __attribute__((aligned(16))) elem_bits window[kStep ? kWholeWindow * kHeadDim : 8];
    __shared__ __attribute__((aligned(16))) elem_bits newest[kStep ? 2 * kHeadDim : 8];                 // the coarse key this token completes, and the fine one
    warm_kernel_arguments<sizeof(S1DecodeParams) + (kStep ? sizeof(Step) : 0)>();
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ti = static_cast<int>(blockIdx.x) - (kStep ? 1 : 0), h = blockIdx.y, b = blockIdx.z;
    int add_f = -1, add_c = -1;
    S1DecodeSeq sq;
    if constexpr (kStep) {
        const int len = t.lens ? t.lens[b] : t.host_len;
        sq.q_row = b; sq.Sq = 1;
        sq.Lk = s1d_step_rows(len, t.capacity, t.kernel_f, t.stride_f, t.fine_capacity, add_f);
        sq.Lc = s1d_step_rows(len, t.capacity, t.kernel_c, t.stride_c, t.coarse_capacity, add_c);
        sq.kbase = p.k + b * p.k_batch_stride + h * p.k_head_stride;
        sq.cbase = p.c + b * p.c_batch_stride + h * p.c_head_stride;
        if (ti < 0) {                                          // the caches' keepers
            s1d_keep_caches(s1d_strides(p), t, b, h, len, sq.Lk, sq.Lc, add_f, add_c, tid, true, !t.with_scores, 0);
            return;
        }
    } else {
        sq = s1d_sequence(p, b, h);
        if (sq.Sq <= 0) return;
    }
    int vis_c, vis_f, tiles;
    s1d_fine_extent<kPool>(p, sq, vis_c, vis_f, tiles);
    if (ti >= tiles && ti > 0) return;                         // uniform over the workgroup
    const bool live = ti < tiles, owns_tail = ti + 1 >= tiles; // not live: the row's first workgroup, which fills a row without scores
    const int tiles_c = vis_c > 64 * kWholeRecords ? kWholeRecords : (vis_c + 63) >> 6;     // lengths beyond what the launch was announced stay inside

    // what is read, requested in the order in which it is needed
    elem8 qf[4], ca[16], cb[16], mine[4], before[4];
    s1d_load_q(qf, p, sq, h, n, g);
    if (wave < tiles_c) s1d_load_tile(ca, sq.cbase, p.c_row_stride, wave * 64, sq.Lc, n, g);
    if (wave + kWholeWaves < tiles_c) s1d_load_tile(cb, sq.cbase, p.c_row_stride, (wave + kWholeWaves) * 64, sq.Lc, n, g);
    if (live) {
        int row = ti * 64 + 16 * wave + n;
        row = row < sq.Lk ? row : sq.Lk - 1;
        const elem_bits* src = sq.kbase + row * p.k_row_stride + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; ++c) mine[c] = *reinterpret_cast<const elem8*>(src + 32 * c);
        if (kPool) s1d_load_group_before(before, sq, p.k_row_stride, ti, n, g);     // every wavefront: a condition on it costs a wait for the loads
    }
    if constexpr (kStep) {
        const bool adds_f = live && add_f >> 6 == ti;          // uniform over the workgroup
        if (add_c >= 0) {
            // the window's rows to LDS, all of them requested at once; its last row is the new token's
            const elem_bits* rows = t.kcache + b * t.kc_batch + static_cast<int64_t>(add_c) * t.stride_c * t.kc_row + h * t.kc_head + (tid & 15) * 8;
            const elem_bits* last = t.knew + b * t.kn_batch + h * t.kn_head + (tid & 15) * 8;
            uint4 w[kWholeWindow / (4 * kWholeWaves)];
#pragma unroll
            for (int i = 0; i < kWholeWindow / (4 * kWholeWaves); ++i) {
                const int row = 4 * kWholeWaves * i + (tid >> 4);
                w[i] = *reinterpret_cast<const uint4*>(row < t.kernel_c - 1 ? rows + row * t.kc_row : last);
            }
#pragma unroll
            for (int i = 0; i < kWholeWindow / (4 * kWholeWaves); ++i)
                *reinterpret_cast<uint4*>(&window[(4 * kWholeWaves * i + (tid >> 4)) * kHeadDim + (tid & 15) * 8]) = w[i];
        }
        if (adds_f && wave >= 2) newest[kHeadDim + (tid & 127)] = s1d_window_mean(t, b, h, add_f, t.kernel_f, t.stride_f, tid & 127);
        if (add_c >= 0) {
            __syncthreads();
            if (wave < 2) {
                // in window order; the next rows are on their way while these are added up
                constexpr int kRows = 32;
                float sum = 0.f;
                elem_bits even[kRows], odd[kRows];
                auto fetch = [&](elem_bits (&rows)[kRows], int from) {
#pragma unroll
                    for (int r = 0; r < kRows; ++r) rows[r] = window[(from + r) * kHeadDim + tid];
                };
                auto add = [&](const elem_bits (&rows)[kRows], int from) {
                    if (from + kRows <= t.kernel_c) {
#pragma unroll
                        for (int r = 0; r < kRows; ++r) sum += elem_to_f32(rows[r]);
                    } else {
#pragma unroll
                        for (int r = 0; r < kRows; ++r) sum += from + r < t.kernel_c ? elem_to_f32(rows[r]) : 0.f;
                    }
                };
                fetch(even, 0);
#pragma unroll
                for (int from = 0; from < kWholeWindow; from += 2 * kRows) {
                    fetch(odd, from + kRows);
                    add(even, from);
                    if (from + 2 * kRows < kWholeWindow) fetch(even, from + 2 * kRows);
                    add(odd, from + kRows);
                }
                const elem_bits mean = f32_to_elem_hw(sum / static_cast<float>(t.kernel_c));
                newest[tid] = mean;
                if (ti == 0) t.coarse[b * p.c_batch_stride + add_c * p.c_row_stride + h * p.c_head_stride + tid] = mean;
            }
        }
        if (adds_f || add_c >= 0) __syncthreads();
        if (adds_f && ti * 64 + 16 * wave + n >= add_f) {      // the newest key, and the lanes beyond it that repeat it
#pragma unroll
            for (int c = 0; c < 4; ++c) mine[c] = *reinterpret_cast<const elem8*>(newest + kHeadDim + 32 * c + 8 * g);
        }
    }
    auto patch = [&](elem8 (&tile)[16], int r) {
        if (!kStep || add_c < 0 || r != add_c >> 6) return;    // uniform
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
            if (r * 64 + 16 * kt + n >= add_c) {
#pragma unroll
                for (int c = 0; c < 4; ++c) tile[kt * 4 + c] = *reinterpret_cast<const elem8*>(newest + 32 * c + 8 * g);
            }
    };
    auto record = [&](elem8 (&tile)[16], int r) {
        patch(tile, r);
        float m[4], l[4], mm[4], ll[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { m[e] = -INFINITY; l[e] = 0.f; }
        s1d_lse_tile(p, qf, tile, r, vis_c, n, m, l);
        s1d_lse_close(m, l, mm, ll);
        if (n == 0) {
            *reinterpret_cast<floatx4*>(records + r * 32 + 4 * g) = floatx4{mm[0], mm[1], mm[2], mm[3]};
            *reinterpret_cast<floatx4*>(records + r * 32 + 16 + 4 * g) = floatx4{ll[0], ll[1], ll[2], ll[3]};
        }
    };
    static_assert(kWholeRecords <= 2 * kWholeWaves, "two coarse tiles to a wavefront");
    if (wave < tiles_c) record(ca, wave);
    if (wave + kWholeWaves < tiles_c) record(cb, wave + kWholeWaves);
    // S of the 16 keys, before the wait for the other records
    auto products = [&](const elem8 (&t4)[4]) {
        floatx4 s = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) s = IV2_MFMA(qf[c], t4[c], s, 0, 0, 0);
        return s;
    };
    floatx4 s_mine = {0.f, 0.f, 0.f, 0.f}, s_before = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        s_mine = products(mine);
        if (kPool && wave == kWholeWaves - 1 && ti > 0) s_before = products(before);
    }
    __syncthreads();
    float carry = 0.f;                                         // score of the last key before the tile (the last wavefront's)
    if (live) {
        S1DRecords rec;
        float lse2[4];
        s1d_load_records(rec, records, tiles_c, n, g);
        s1d_merge_records(rec, tiles_c, n, g, p.group, lse2);
        auto score_of = [&](const floatx4& s) {                // of key n of the 16, in every row
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) sum += __builtin_amdgcn_exp2f(s[e] * p.scale_log2 - lse2[e]);
            const float rows = s1d_fold_rows16(sum, sum);
            return s1d_fold_rows32(rows, rows);
        };
        const float got = score_of(s_mine);
        const int key = ti * 64 + 16 * wave + n;
        if (!kPool) {
            if (g == 0 && key < p.cols) p.out[static_cast<int64_t>(h) * p.out_head_stride + static_cast<int64_t>(sq.q_row) * p.out_row_stride + key] =
                f32_to_elem_hw(key < vis_f ? got : 0.f);
        } else {
            if (g == 0) score[16 * wave + n] = key < vis_f ? got : 0.f;
            if (wave == kWholeWaves - 1 && ti > 0) {
                const float prev = ti * 64 - 16 + n < vis_f ? score_of(s_before) : 0.f;
                carry = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(prev), 15));
            }
        }
    }
    if constexpr (kPool) __syncthreads();
    if (wave != kWholeWaves - 1) return;
    s1d_store_tile<kPool>(p, sq, live ? score[lane] : 0.f, carry, vis_f, tiles, ti, live, owns_tail, b, h, lane);
}

}  // namespace IV2_NS

using namespace IV2_NS;

namespace {

// Every run is `run` tiles long whatever its sequence's length, so the wavefronts all carry the same load; the longest
// sequence is cut into at most 64 runs.  One tile per run while that makes no more than two wavefronts per SIMD (the time is
// one wavefront's chain of round trips then), two beyond, both requested before the first is used.
void s1d_splits(int batch, int num_heads_k, int max_keys, int max_coarse, int& splits_f, int& splits_c, int& run_f, int& run_c) {
    auto plan = [&](int tiles, int& splits, int& run) {
        run = static_cast<int64_t>(batch) * num_heads_k * tiles <= 2048 ? 1 : 2;
        if ((tiles + run - 1) / run > 64) run = (tiles + 63) / 64;
        splits = (tiles + run - 1) / run;
        if (splits < 1) splits = 1;
    };
    plan((max_keys + 63) / 64, splits_f, run_f);
    plan((max_coarse + 63) / 64, splits_c, run_c);
}
// One launch (stage1_decode_whole_kernel) instead of two: up to five coarse tiles, i.e. 20 607 tokens, and a workgroup per CU.  Every workgroup loads all coarse
// tiles, 16 KiB each, through its CU's vector memory path and forms their records; that costs 0.4 us a tile, and the launch it saves is worth 1.5 us of the device
// and 2.5 us of the host that issues it.  A decode step in us, two launches | one: one sequence of 1000 tokens 17.5 | 14.8, 4000 17.6 | 15.1, 8000 17.9 | 15.9, 16 000
// 18.0 | 16.9, 20 000 18.0 | 18.1, 24 000 18.1 | 18.6, 32 000 18.0 | 19.4; two of up to 8000 17.5 | 15.6, six of up to 20 000 19.2 | 18.1, eight of up to 8000 19.7 | 17.9,
// 16 of them (256 workgroups) 24.2 | 23.0; 32 (512) 34.4 | 37.4, 24 of up to 16 000 34.0 | 41.8; eight paged ones of up to 8000, called operator by operator, 25.5 | 22.8.
constexpr int kWholeCoarseTiles = 5;
static_assert(kWholeCoarseTiles <= kWholeRecords, "a record per coarse tile");
constexpr int kWholeWorkgroups = 256;
bool s1d_whole(const S1DecodeParams& p, int batch, int num_heads_k) {
    return p.run_c == 1 && p.run_f == 1 && p.splits_c <= kWholeCoarseTiles &&
           static_cast<int64_t>(batch) * num_heads_k * p.splits_f <= kWholeWorkgroups;
}
unsigned s1d_lse_workgroups(int splits_c) { return static_cast<unsigned>((splits_c + kLseWaves - 1) / kLseWaves); }

}  // namespace

#ifndef IV2_F16        // element-type independent: defined once
extern "C" size_t infllmv2_stage1_decode_workspace_bytes(int batch, int num_heads_k, int max_seqlen_k, int max_seqlen_v) {
    int sf, sc, rf, rc;
    s1d_splits(batch, num_heads_k, max_seqlen_k, max_seqlen_v, sf, sc, rf, rc);
    return static_cast<size_t>(batch > 0 ? batch : 0) * (num_heads_k > 0 ? num_heads_k : 0) * sc * 32 * sizeof(float);
}
#endif

extern "C" int IV2_ENTRY(infllmv2_stage1_decode)(void* stream, const void* q, const void* k, const void* v, void* out,
                                      const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, const int32_t* k_lens,
                                      const int32_t* cu_seqlens_v, const int32_t* v_lens, void* workspace,
                                      size_t workspace_bytes, int batch, int num_heads, int num_heads_k, int head_dim,
                                      int max_seqlen_k, int max_seqlen_v, const int64_t* q_strides,
                                      const int64_t* k_strides, const int64_t* v_strides, int64_t out_head_stride,
                                      int64_t out_row_stride, float softmax_scale, int is_causal, int pooled,
                                      const int32_t* cache_lens, int cache_len, int out_len, int kernel_size, int stride,
                                      int padding, int block_size, int local_blocks, int init_blocks) {
    const char* who = "stage1_decode";
    IV2_CHECK(head_dim == kHeadDim, "%s: this build only supports head_dim 128 (got %d)", who, head_dim);
    IV2_CHECK(valid_group(num_heads, num_heads_k),
              "%s: requires num_heads == g * num_heads_k with g in {1, 2, 4, 8, 16} (got %d and %d)", who, num_heads, num_heads_k);
    IV2_CHECK(batch > 0 && max_seqlen_k >= 0 && max_seqlen_v >= 0, "%s: bad sizes", who);
    IV2_CHECK(num_heads_k <= 65535 && batch <= 65535, "%s: batch and num_heads_k must not exceed 65535", who);
    IV2_CHECK(q && k && v && out, "%s: null pointer", who);
    IV2_CHECK((cu_seqlens_k != nullptr) != (k_lens != nullptr) && (cu_seqlens_v != nullptr) != (v_lens != nullptr),
              "%s: give either cumulative lengths (packed keys) or per-sequence lengths (key caches), for k and for v", who);
    IV2_CHECK(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(v) % 16 == 0, "%s: q, k, v must be 16-byte aligned", who);
    for (int s = 0; s < 3; ++s)
        IV2_CHECK(q_strides[s] % 8 == 0 && k_strides[s] % 8 == 0 && v_strides[s] % 8 == 0,
                  "%s: strides must be multiples of 8 elements", who);
    if (pooled) {
        IV2_CHECK(kernel_size == 5 && stride == 4 && padding == 1 && block_size == kBlockN,
                  "%s: only the 5/4/1 pooling window on 64-token blocks is fused (got %d/%d/%d on %d)", who, kernel_size,
                  stride, padding, block_size);
        IV2_CHECK(out_len >= 0 && cache_len >= 0 && out_row_stride >= out_len, "%s: bad out_len, cache_len or output row stride", who);
        if (out_len == 0) return 0;
    } else {
        IV2_CHECK(out_row_stride >= max_seqlen_k, "%s: score row stride shorter than max_seqlen_k", who);
    }
    S1DecodeParams p{};
    s1d_splits(batch, num_heads_k, max_seqlen_k, max_seqlen_v, p.splits_f, p.splits_c, p.run_f, p.run_c);
    IV2_CHECK(workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
              workspace_bytes >= infllmv2_stage1_decode_workspace_bytes(batch, num_heads_k, max_seqlen_k, max_seqlen_v),
              "%s: workspace missing, misaligned or too small", who);
    p.q = static_cast<const elem_bits*>(q);
    p.k = static_cast<const elem_bits*>(k);
    p.c = static_cast<const elem_bits*>(v);
    p.out = static_cast<elem_bits*>(out);
    p.partial = static_cast<float*>(workspace);
    p.cu_seqlens_q = cu_seqlens_q;
    p.cu_seqlens_k = cu_seqlens_k; p.k_lens = k_lens;
    p.cu_seqlens_c = cu_seqlens_v; p.c_lens = v_lens;
    p.q_tok_stride = q_strides[0]; p.q_grp_stride = q_strides[1]; p.q_kvh_stride = q_strides[2];
    p.k_batch_stride = k_strides[0]; p.k_row_stride = k_strides[1]; p.k_head_stride = k_strides[2];
    p.c_batch_stride = v_strides[0]; p.c_row_stride = v_strides[1]; p.c_head_stride = v_strides[2];
    p.out_head_stride = out_head_stride; p.out_row_stride = out_row_stride;
    p.cols = max_seqlen_k;
    p.group = num_heads / num_heads_k;
    p.scale_log2 = softmax_scale * 1.44269504088896340736f;
    p.causal = is_causal;
    p.cache_lens = cache_lens; p.cache_len = cache_len; p.pool_len = out_len;
    p.local_blocks = local_blocks; p.init_blocks = init_blocks;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (s1d_whole(p, batch, num_heads_k)) {
        auto kernel = pooled ? stage1_decode_whole_kernel<true, S1DecodeNoStep> : stage1_decode_whole_kernel<false, S1DecodeNoStep>;
        hipLaunchKernelGGL(kernel, dim3(p.splits_f, num_heads_k, batch), dim3(64 * kWholeWaves), 0, st, p, S1DecodeNoStep{});
        IV2_LAUNCH_CHECK();
        return 0;
    }
    hipLaunchKernelGGL(stage1_decode_lse_kernel, dim3(s1d_lse_workgroups(p.splits_c), num_heads_k, batch), dim3(64 * kLseWaves), 0, st, p);
    IV2_LAUNCH_CHECK();
    const dim3 grid(p.splits_f, num_heads_k, batch);
    if (pooled) hipLaunchKernelGGL(stage1_decode_score_kernel<true>, grid, dim3(64), 0, st, p);
    else hipLaunchKernelGGL(stage1_decode_score_kernel<false>, grid, dim3(64), 0, st, p);
    IV2_LAUNCH_CHECK();
    return 0;
}

extern "C" int IV2_ENTRY(infllmv2_decode_step_scores)(void* stream, const void* q, const void* k_new, const void* v_new, void* kcache,
                                           void* vcache, void* fine_cache, void* coarse_cache, const int32_t* lens, int host_len,
                                           int32_t* new_lens, int32_t* fine_lens, int32_t* coarse_lens, void* pooled,
                                           void* workspace, size_t workspace_bytes, int batch, int num_heads, int num_heads_k,
                                           int head_dim, int capacity, int fine_rows, int coarse_rows, int max_len,
                                           const int64_t* q_strides, const int64_t* knew_strides, const int64_t* vnew_strides,
                                           const int64_t* kcache_strides, const int64_t* vcache_strides,
                                           const int64_t* fine_strides, const int64_t* coarse_strides, int kernel_size_f,
                                           int stride_f, int kernel_size_c, int stride_c, float softmax_scale, int out_len,
                                           int local_blocks, int init_blocks) {
    const char* who = "decode_step_scores";
    IV2_CHECK(head_dim == kHeadDim, "%s: this build only supports head_dim 128 (got %d)", who, head_dim);
    IV2_CHECK(valid_group(num_heads, num_heads_k),
              "%s: requires num_heads == g * num_heads_k with g in {1, 2, 4, 8, 16} (got %d and %d)", who, num_heads, num_heads_k);
    IV2_CHECK(batch > 0 && batch <= 65535 && num_heads_k <= 65535, "%s: batch and num_heads_k must be in [1, 65535]", who);
    IV2_CHECK(capacity > 0 && fine_rows > 0 && coarse_rows > 0 && max_len > 0 && host_len >= 0 && out_len >= 0, "%s: bad sizes", who);
    IV2_CHECK(kernel_size_f > 0 && stride_f > 0 && kernel_size_c > 0 && stride_c > 0, "%s: kernel_size and stride must be positive", who);
    IV2_CHECK(k_new && v_new && kcache && vcache && fine_cache && coarse_cache && fine_lens && coarse_lens, "%s: null pointer", who);
    IV2_CHECK(pooled == nullptr || (q != nullptr && workspace != nullptr), "%s: null pointer", who);
    const void* aligned16[] = {q, k_new, v_new, kcache, vcache, fine_cache, coarse_cache, workspace};
    for (const void* a : aligned16) IV2_CHECK(reinterpret_cast<uintptr_t>(a) % 16 == 0, "%s: tensors must be 16-byte aligned", who);
    for (int s = 0; s < 3; ++s)
        IV2_CHECK(kcache_strides[s] % 8 == 0 && vcache_strides[s] % 8 == 0 && fine_strides[s] % 8 == 0 && coarse_strides[s] % 8 == 0 &&
                  (pooled == nullptr || q_strides[s] % 8 == 0), "%s: strides must be multiples of 8 elements", who);
    IV2_CHECK(knew_strides[0] % 8 == 0 && knew_strides[1] % 8 == 0 && vnew_strides[0] % 8 == 0 && vnew_strides[1] % 8 == 0,
              "%s: strides must be multiples of 8 elements", who);
    S1DecodeParams p{};
    S1DecodeStep t{};
    // the compressed keys the longest sequence can hold after the step
    auto windows = [&](int len, int ks, int st) { return len >= ks ? (len - ks) / st + 1 : 0; };
    int max_f = windows(max_len, kernel_size_f, stride_f), max_c = windows(max_len, kernel_size_c, stride_c);
    max_f = max_f < fine_rows ? max_f : fine_rows;
    max_c = max_c < coarse_rows ? max_c : coarse_rows;
    if (pooled) {
        s1d_splits(batch, num_heads_k, max_f, max_c, p.splits_f, p.splits_c, p.run_f, p.run_c);
        IV2_CHECK(workspace_bytes >= infllmv2_stage1_decode_workspace_bytes(batch, num_heads_k, max_f, max_c), "%s: workspace too small", who);
    }
    p.q = static_cast<const elem_bits*>(q);
    p.k = static_cast<const elem_bits*>(fine_cache);
    p.c = static_cast<const elem_bits*>(coarse_cache);
    p.out = static_cast<elem_bits*>(pooled);
    p.partial = static_cast<float*>(workspace);
    p.k_lens = fine_lens; p.c_lens = coarse_lens;
    if (pooled) { p.q_tok_stride = q_strides[0]; p.q_grp_stride = q_strides[1]; p.q_kvh_stride = q_strides[2]; }
    p.k_batch_stride = fine_strides[0]; p.k_row_stride = fine_strides[1]; p.k_head_stride = fine_strides[2];
    p.c_batch_stride = coarse_strides[0]; p.c_row_stride = coarse_strides[1]; p.c_head_stride = coarse_strides[2];
    p.out_head_stride = out_len; p.out_row_stride = static_cast<int64_t>(num_heads_k) * out_len;
    p.cols = fine_rows;
    p.group = num_heads / num_heads_k;
    p.scale_log2 = softmax_scale * 1.44269504088896340736f;
    // the query sits at the position of the new token: its own block is lens[b] / 64
    p.cache_lens = lens; p.cache_len = host_len; p.pool_len = out_len;
    p.local_blocks = local_blocks; p.init_blocks = init_blocks;
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
    t.with_scores = pooled != nullptr ? 1 : 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (pooled != nullptr && out_len > 0 && kernel_size_c <= kWholeWindow && s1d_whole(p, batch, num_heads_k)) {
        hipLaunchKernelGGL((stage1_decode_whole_kernel<true, S1DecodeStep>), dim3(1 + p.splits_f, num_heads_k, batch),
                           dim3(64 * kWholeWaves), 0, st, p, t);
        IV2_LAUNCH_CHECK();
        return 0;
    }
    hipLaunchKernelGGL(stage1_decode_front_kernel, dim3(1 + s1d_lse_workgroups(p.splits_c), num_heads_k, batch), dim3(64 * kLseWaves), 0, st, p, t);
    IV2_LAUNCH_CHECK();
    if (pooled == nullptr || out_len == 0) return 0;
    hipLaunchKernelGGL(stage1_decode_score_kernel<true>, dim3(p.splits_f, num_heads_k, batch), dim3(64), 0, st, p);
    IV2_LAUNCH_CHECK();
    return 0;
}
