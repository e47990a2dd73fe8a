// Stage-2 block-sparse flash-attention forward for gfx950 (head_dim 128, up to 16 query heads per KV head): the
// K/V image pre-pass and the C entry point; the attention kernel itself is in stage2_fwd_hybrid.hip.
//
// Semantics follow compute_attn_1rowblock (csrc/flash_attn/src/flash_fwd_kernel.h:137-602) with
// the bitmask walk of flash_blockmask.h:5-100: token i of a sequence attends key t iff
// t <= i + Sk - Sq (causal, bottom-right aligned), t < Sk, and bit t/64 of its mask row is set;
// O = softmax(scale * q.K^T) V with fp32 softmax and P rounded to bf16 before P.V; rows with no
// allowed key give O = 0 and LSE = +inf (softmax.h:240-256).
//
// Design (not the reference's): the 16 grouped heads of one token form the 16-column N side of
// v_mfma_f32_16x16x32_bf16.  S^T = K.Q^T puts keys on the M side, so one lane owns one head's
// scores for 16 keys and the same registers, converted to bf16, are the B operand of
// O^T = V^T.P^T.  K and V come from fragment-major block images (kv_image.h) built by
// pack_kv_kernel, so every operand fetch is one contiguous 1 KiB wavefront load.  Q, O and the
// LSE are addressed through strides: the caller's (T, Hq, d) tensors are used in place.
#include "common.h"
#include "kv_image.h"
#include "block_walker.h"
#include "stage2_fwd.h"
#include "in_step.h"
#include "mask_tile.h"
#include "infllmv2_hip.h"
#include <math.h>

namespace IV2_NS {

// ---------------------------------------------------------------------------------------------
// K/V -> block images
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void pack_kv_kernel(const PackParams p) {
    __shared__ __attribute__((aligned(16))) elem_bits rows[kPackElems];
    pack_block(p, blockIdx.x, blockIdx.y, blockIdx.z, rows);
}

#ifndef IV2_F16
// The images, and the mask words of an index list, in one launch: for each sequence and KV head the first `blocks` workgroups pack, the others take four
// rows of the list each.  Both are bound by latency.
constexpr int kMaskRowsPerWg = 4;

__global__ __launch_bounds__(256)
void pack_kv_and_topk_kernel(const PackParams p, int blocks, const int32_t* __restrict__ idx, uint64_t* __restrict__ mask, int64_t rows, int k, int n64) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    if (static_cast<int>(blockIdx.x) < blocks) {
        pack_block(p, blockIdx.x, blockIdx.y, blockIdx.z, reinterpret_cast<elem_bits*>(lds));
        return;
    }
    const int64_t wg = (static_cast<int64_t>(blockIdx.z) * gridDim.y + blockIdx.y) * (gridDim.x - blocks) + (blockIdx.x - blocks);
    const int wave = threadIdx.x >> 6;
    topk_row_words(idx, mask, wg * kMaskRowsPerWg + wave, rows, k, n64, reinterpret_cast<unsigned long long*>(lds) + wave * n64, threadIdx.x & 63);
}

// The images, and mask words of rows that all have their first `set` blocks, kWordsPerWg to a workgroup: the front of a prefill whose sequences hold no more blocks than are
// selected, in place of compressed keys, scores and selection.  Whole prefill in us, 2 KV heads,
// 64 blocks: 500 tokens 23.8 -> 16.8, 1000 31.2 -> 26.6, 2048 61.1 -> 57.0, 4096 175 -> 169, four of 2000 194 -> 186; 30 of 300, 16 blocks, 98 -> 89.
constexpr int kWordsPerWg = 2048;

__global__ __launch_bounds__(256)
void pack_kv_and_first_kernel(const PackParams p, int blocks, uint64_t* __restrict__ mask, int64_t words, int set, int n64) {
    __shared__ __attribute__((aligned(16))) elem_bits rows[kPackElems];
    if (static_cast<int>(blockIdx.x) < blocks) {
        pack_block(p, blockIdx.x, blockIdx.y, blockIdx.z, rows);
        return;
    }
    const int64_t wg = (static_cast<int64_t>(blockIdx.z) * gridDim.y + blockIdx.y) * (gridDim.x - blocks) + (blockIdx.x - blocks);
    for (int i = threadIdx.x; i < kWordsPerWg; i += 256) {
        const int64_t at = wg * kWordsPerWg + i;
        if (at >= words) return;
        const int from = n64 == 1 ? 0 : 64 * static_cast<int>(at % n64);
        mask[at] = from + 64 <= set ? ~0ull : from < set ? (1ull << (set - from)) - 1ull : 0ull;
    }
}
#endif

}  // namespace IV2_NS

using namespace IV2_NS;

#ifndef IV2_F16        // both element types are 2 bytes wide: defined once
extern "C" size_t infllmv2_kv_image_bytes(int64_t total_k, int batch, int num_heads_k) {
    return image_bytes(total_k, batch, num_heads_k) + kInStepBytes;           // behind the images: counters of the launch that walks them
}
#endif

namespace IV2_NS {
int check_pack(const void* k, const void* v, const int32_t* cu_seqlens_k, const void* workspace, size_t workspace_bytes, int batch,
               int64_t total_k, int num_heads_k, int max_seqlen_k, const int64_t* k_strides, const int64_t* v_strides) {
    IV2_CHECK(k && v && cu_seqlens_k && workspace, "pack_kv: null pointer");
    IV2_CHECK(batch > 0 && num_heads_k > 0 && total_k >= 0 && max_seqlen_k >= 0, "pack_kv: bad sizes");
    IV2_CHECK(num_heads_k <= 65535 && batch <= 65535, "pack_kv: batch and num_heads_k must not exceed 65535");
    IV2_CHECK(workspace_bytes >= image_bytes(total_k, batch, num_heads_k), "pack_kv: workspace too small");
    IV2_CHECK(reinterpret_cast<uintptr_t>(k) % 16 == 0 && reinterpret_cast<uintptr_t>(v) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "pack_kv: k, v and workspace must be 16-byte aligned");
    IV2_CHECK(k_strides[0] % 8 == 0 && k_strides[1] % 8 == 0 && v_strides[0] % 8 == 0 && v_strides[1] % 8 == 0,
              "pack_kv: k/v row and head strides must be multiples of 8 elements");
    return 0;
}
int launch_pack(hipStream_t st, const void* k, const void* v, const int32_t* cu_seqlens_k, void* workspace,
                size_t workspace_bytes, int batch, int64_t total_k, int num_heads_k, int max_seqlen_k,
                const int64_t* k_strides, const int64_t* v_strides, unsigned* in_step) {
    const int rc = check_pack(k, v, cu_seqlens_k, workspace, workspace_bytes, batch, total_k, num_heads_k, max_seqlen_k, k_strides, v_strides);
    if (rc != 0) return rc;
    const int max_blocks = (max_seqlen_k + kBlockN - 1) / kBlockN;
    if (max_blocks == 0 || total_k == 0) return 0;
    const PackParams pp = pack_params(k, v, cu_seqlens_k, workspace, batch, total_k, num_heads_k, k_strides, v_strides, in_step);
    hipLaunchKernelGGL(pack_kv_kernel, dim3(max_blocks, batch, num_heads_k), dim3(256), 0, st, pp);
    IV2_LAUNCH_CHECK();
    return 0;
}
}  // namespace IV2_NS

#ifndef IV2_F16        // the images are a permutation of 2-byte elements: one entry point serves both element types
extern "C" int infllmv2_pack_kv(void* stream, const void* k, const void* v, const int32_t* cu_seqlens_k,
                                void* workspace, size_t workspace_bytes, int batch, int64_t total_k,
                                int num_heads_k, int head_dim, int max_seqlen_k, const int64_t* k_strides,
                                const int64_t* v_strides) {
    IV2_CHECK(head_dim == kHeadDim, "pack_kv: this build only supports head_dim 128 (got %d)", head_dim);
    return launch_pack(static_cast<hipStream_t>(stream), k, v, cu_seqlens_k, workspace, workspace_bytes, batch,
                       total_k, num_heads_k, max_seqlen_k, k_strides, v_strides);
}

extern "C" int infllmv2_pack_kv_and_topk(void* stream, const void* k, const void* v, const int32_t* cu_seqlens_k, void* workspace, size_t workspace_bytes,
                                         int batch, int64_t total_k, int num_heads_k, int head_dim, int max_seqlen_k, const int64_t* k_strides,
                                         const int64_t* v_strides, const int32_t* topk_idx, uint64_t* mask, int64_t rows, int topk, int n_uint64_per_row) {
    IV2_CHECK(head_dim == kHeadDim, "pack_kv: this build only supports head_dim 128 (got %d)", head_dim);
    IV2_CHECK(rows >= 0 && topk >= 0 && n_uint64_per_row >= 0 && n_uint64_per_row <= 1024, "pack_kv_and_topk: bad sizes");
    IV2_CHECK(rows == 0 || n_uint64_per_row == 0 || (mask && (topk_idx || topk == 0)), "pack_kv_and_topk: null pointer");
    if (int rc = check_pack(k, v, cu_seqlens_k, workspace, workspace_bytes, batch, total_k, num_heads_k, max_seqlen_k, k_strides, v_strides)) return rc;
    const int blocks = total_k == 0 ? 0 : (max_seqlen_k + kBlockN - 1) / kBlockN;
    const int64_t pairs = static_cast<int64_t>(batch) * num_heads_k;
    const int64_t mask_wgs = n_uint64_per_row == 0 ? 0 : ((rows + kMaskRowsPerWg - 1) / kMaskRowsPerWg + pairs - 1) / pairs;
    if (blocks + mask_wgs == 0) return 0;
    IV2_CHECK(blocks + mask_wgs <= max_workgroups(256), "pack_kv_and_topk: too many rows");
    const PackParams pp = pack_params(k, v, cu_seqlens_k, workspace, batch, total_k, num_heads_k, k_strides, v_strides, nullptr);
    size_t lds = sizeof(uint64_t) * kMaskRowsPerWg * n_uint64_per_row;
    if (lds < kPackElems * sizeof(elem_bits)) lds = kPackElems * sizeof(elem_bits);
    hipLaunchKernelGGL(pack_kv_and_topk_kernel, dim3(static_cast<unsigned>(blocks + mask_wgs), batch, num_heads_k), dim3(256), lds,
                       static_cast<hipStream_t>(stream), pp, blocks, topk_idx, mask, rows, topk, n_uint64_per_row);
    IV2_LAUNCH_CHECK();
    return 0;
}

extern "C" int infllmv2_pack_kv_and_first(void* stream, const void* k, const void* v, const int32_t* cu_seqlens_k, void* workspace, size_t workspace_bytes,
                                          int batch, int64_t total_k, int num_heads_k, int head_dim, int max_seqlen_k, const int64_t* k_strides,
                                          const int64_t* v_strides, uint64_t* mask, int64_t rows, int blocks_set, int n_uint64_per_row) {
    IV2_CHECK(head_dim == kHeadDim, "pack_kv: this build only supports head_dim 128 (got %d)", head_dim);
    IV2_CHECK(rows >= 0 && blocks_set >= 0 && n_uint64_per_row >= 0, "pack_kv_and_first: bad sizes");
    IV2_CHECK(rows == 0 || n_uint64_per_row == 0 || mask, "pack_kv_and_first: null pointer");
    if (int rc = check_pack(k, v, cu_seqlens_k, workspace, workspace_bytes, batch, total_k, num_heads_k, max_seqlen_k, k_strides, v_strides)) return rc;
    const int blocks = total_k == 0 ? 0 : (max_seqlen_k + kBlockN - 1) / kBlockN;
    const int64_t pairs = static_cast<int64_t>(batch) * num_heads_k, words = rows * n_uint64_per_row;
    const int64_t mask_wgs = ((words + kWordsPerWg - 1) / kWordsPerWg + pairs - 1) / pairs;
    if (blocks + mask_wgs == 0) return 0;
    IV2_CHECK(blocks + mask_wgs <= max_workgroups(256), "pack_kv_and_first: too many rows");
    const PackParams pp = pack_params(k, v, cu_seqlens_k, workspace, batch, total_k, num_heads_k, k_strides, v_strides, nullptr);
    hipLaunchKernelGGL(pack_kv_and_first_kernel, dim3(static_cast<unsigned>(blocks + mask_wgs), batch, num_heads_k), dim3(256), 0,
                       static_cast<hipStream_t>(stream), pp, blocks, mask, words, blocks_set, n_uint64_per_row);
    IV2_LAUNCH_CHECK();
    return 0;
}
#endif

extern "C" int IV2_ENTRY(infllmv2_varlen_fwd_selected)(void* stream, const void* q, const void* k, const void* v, void* out,
                                   float* softmax_lse, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                   const uint64_t* blockmask, void* workspace, size_t workspace_bytes,
                                   int kv_prepacked, int batch, int64_t total_q, int64_t total_k, int num_heads,
                                   int num_heads_k, int head_dim, int max_seqlen_q, int max_seqlen_k,
                                   const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                   const int64_t* o_strides, const int64_t* lse_strides,
                                   int n_uint64_per_row, float softmax_scale, int is_causal, int most_selected) {
    IV2_CHECK(head_dim == kHeadDim, "varlen_fwd: this build only supports head_dim 128 (got %d)", head_dim);
    IV2_CHECK(valid_group(num_heads, num_heads_k),
              "varlen_fwd: requires num_heads == g * num_heads_k with g in {1, 2, 4, 8, 16} (got %d and %d)", num_heads, num_heads_k);
    IV2_CHECK(batch > 0 && total_q >= 0 && total_k >= 0 && max_seqlen_q >= 0 && max_seqlen_k >= 0, "varlen_fwd: bad sizes");
    IV2_CHECK(q && out && softmax_lse && cu_seqlens_q && cu_seqlens_k && workspace, "varlen_fwd: null pointer");
    IV2_CHECK(num_heads_k <= 65535 && batch <= 65535, "varlen_fwd: batch and num_heads_k must not exceed 65535");
    IV2_CHECK(workspace_bytes >= image_bytes(total_k, batch, num_heads_k), "varlen_fwd: workspace too small");
    IV2_CHECK(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "varlen_fwd: q and workspace must be 16-byte aligned, out 8-byte");
    for (int s = 0; s < 3; ++s) {
        IV2_CHECK(q_strides[s] % 8 == 0 && o_strides[s] % 4 == 0, "varlen_fwd: q strides must be multiples of 8 and out strides of 4 elements");
    }
    IV2_CHECK(blockmask == nullptr || n_uint64_per_row > 0, "varlen_fwd: mask given without words per row");
    IV2_CHECK(softmax_scale > 0.f, "varlen_fwd: softmax_scale must be positive");
    if (total_q == 0 || max_seqlen_q == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Images packed by an earlier call may be read by several launches at once: those leave the workspace as it is.
    const size_t images = image_bytes(total_k, batch, num_heads_k);
    unsigned* in_step = kv_prepacked || workspace_bytes < images + kInStepBytes || max_seqlen_k <= kInStepKeys || total_k == 0 || blockmask == nullptr
                            ? nullptr : reinterpret_cast<unsigned*>(static_cast<unsigned char*>(workspace) + images);
    if (!kv_prepacked) {
        int rc = launch_pack(st, k, v, cu_seqlens_k, workspace, workspace_bytes, batch, total_k, num_heads_k,
                             max_seqlen_k, k_strides, v_strides, in_step);
        if (rc != 0) return rc;
    }
    const int64_t n_slots = image_slots(total_k, batch);
    FwdParams fp{};
    fp.q = static_cast<const elem_bits*>(q);
    fp.out = static_cast<elem_bits*>(out);
    fp.lse = softmax_lse;
    fp.kimg = static_cast<const elem_bits*>(workspace);
    fp.vimg = fp.kimg + n_slots * num_heads_k * kImageElems;
    fp.cu_seqlens_q = cu_seqlens_q; fp.cu_seqlens_k = cu_seqlens_k;
    fp.mask = blockmask;
    fp.q_tok_stride = q_strides[0]; fp.q_grp_stride = q_strides[1]; fp.q_kvh_stride = q_strides[2];
    fp.o_tok_stride = o_strides[0]; fp.o_grp_stride = o_strides[1]; fp.o_kvh_stride = o_strides[2];
    fp.lse_tok_stride = lse_strides[0]; fp.lse_grp_stride = lse_strides[1]; fp.lse_kvh_stride = lse_strides[2];
    fp.n_slots = n_slots;
    fp.total_q = total_q; fp.total_k = total_k;
    fp.group = num_heads / num_heads_k;
    fp.n64 = n_uint64_per_row;
    fp.scale_log2 = softmax_scale * 1.44269504088896340736f;
    return launch_stage2_fwd_hybrid(st, fp, batch, num_heads_k, max_seqlen_q, max_seqlen_k, is_causal != 0, most_selected, in_step);
}

extern "C" int IV2_ENTRY(infllmv2_varlen_fwd)(void* stream, const void* q, const void* k, const void* v, void* out,
                                   float* softmax_lse, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                   const uint64_t* blockmask, void* workspace, size_t workspace_bytes,
                                   int kv_prepacked, int batch, int64_t total_q, int64_t total_k, int num_heads,
                                   int num_heads_k, int head_dim, int max_seqlen_q, int max_seqlen_k,
                                   const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                   const int64_t* o_strides, const int64_t* lse_strides,
                                   int n_uint64_per_row, float softmax_scale, int is_causal) {
    return IV2_ENTRY(infllmv2_varlen_fwd_selected)(stream, q, k, v, out, softmax_lse, cu_seqlens_q, cu_seqlens_k, blockmask, workspace,
                                                   workspace_bytes, kv_prepacked, batch, total_q, total_k, num_heads, num_heads_k, head_dim,
                                                   max_seqlen_q, max_seqlen_k, q_strides, k_strides, v_strides, o_strides, lse_strides,
                                                   n_uint64_per_row, softmax_scale, is_causal, 0);
}
