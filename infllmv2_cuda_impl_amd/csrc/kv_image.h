// Fragment-major K/V block images.
//
// Stage-2 kernels never read K or V in the caller's (token, head, d) layout.  A pre-pass
// rewrites every 64-key block of one KV head into two 16 KiB "images" whose 16-byte units are
// already the per-lane operands of v_mfma_f32_16x16x32_bf16, so a wavefront fetches one MFMA
// operand with a single fully-coalesced 1 KiB load (global) or a conflict-free ds_read_b128
// (LDS copy of the image).  With lane = 16*g + r (r = lane % 16, g = lane / 16):
//
//   K image  unit (kt, c, lane), kt,c in [0,4):   8 x bf16  K[key = 16*kt + r][d = 32*c + 8*g + j]
//            = A operand of  S^T(16 keys x 16 heads) += K(16 x 32) * Q^T(32 x 16)
//   V image  unit (dt, cc, lane), dt in [0,8), cc in [0,2):
//            8 x bf16  V[key = 32*cc + (j < 4 ? 4*g + j : 16 + 4*g + j - 4)][d = 16*dt + r]
//            = A operand of  O^T(16 d x 16 heads) += V^T(16 x 32) * P^T(32 x 16)
//            where the key order inside a 32-key chunk is exactly the order in which one lane
//            holds two S^T accumulator tiles, so P needs no data movement between the GEMMs.
//
// Keys past the end of a sequence are stored as zeros.  Block `j` of packed sequence `b` lives in
// slot  cu_seqlens_k[b] / 64 + b + j  (a bound that never overlaps and needs no host sync).
#pragma once
#include "common.h"
#include "in_step.h"

namespace IV2_NS {

constexpr int kImageElems = kBlockN * kHeadDim;            // 8192 bf16 = 16 KiB per image

__host__ __device__ inline int64_t image_slots(int64_t total_k, int batch) {
    return total_k / kBlockN + batch + 1;
}

// bytes of both images of every block
inline size_t image_bytes(int64_t total_k, int batch, int num_heads_k) {
    return static_cast<size_t>(image_slots(total_k, batch)) * num_heads_k * kImageElems * sizeof(elem_bits) * 2;
}

__device__ __forceinline__ int64_t image_slot0(const int* cu_seqlens_k, int b) {
    return cu_seqlens_k[b] / kBlockN + b;
}

// One block's K image, by a workgroup of 256: rows is the block's first row, `valid` of its keys are inside the sequence.
__device__ __forceinline__ void write_k_image(const elem_bits* rows, int64_t row_stride, int valid, elem_bits* image, int tid) {
    uint4 val[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int u = tid + 256 * i, c = (u >> 6) & 3, lane = u & 63;
        const int key = 16 * (u >> 8) + (lane & 15);
        val[i] = make_uint4(0, 0, 0, 0);
        if (key < valid) val[i] = *reinterpret_cast<const uint4*>(rows + key * row_stride + 32 * c + 8 * (lane >> 4));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(image + (tid + 256 * i) * 8) = val[i];
}
// Both images of a block.
struct PackParams {
    const elem_bits* k;
    const elem_bits* v;
    elem_bits* kimg;                // K in K-image order (operand of a GEMM contracting over d)
    elem_bits* vimg;                // V in V-image order (A operand of a GEMM contracting over keys)
    const int* cu_seqlens_k;
    int64_t k_row_stride, k_head_stride;
    int64_t v_row_stride, v_head_stride;
    int64_t n_slots;
    unsigned* in_step;              // counters of in_step.h to clear for the launch that walks the images, or null (a launch of its own took 10 us)
};
static_assert(8 * kInStepPitch == 256, "one counter word per thread of a packing workgroup");

constexpr int kVPitch = kHeadDim + 8;                      // LDS row (elements) of the V transposition, padded
constexpr int kPackElems = kBlockN * kVPitch;

// Block j of sequence b and KV head h, by a workgroup of 256; vt: kPackElems elements of LDS.
__device__ __forceinline__ void pack_block(const PackParams& p, int j, int b, int h, elem_bits* vt) {
    if (p.in_step != nullptr && j + b + h == 0) p.in_step[threadIdx.x] = 0u;
    const int k0 = p.cu_seqlens_k[b];
    const int Sk = p.cu_seqlens_k[b + 1] - k0;
    if (static_cast<int64_t>(j) * kBlockN >= Sk) return;
    const int64_t slot = image_slot0(p.cu_seqlens_k, b) + j;
    const int tid = threadIdx.x;
    const elem_bits* kb = p.k + (k0 + static_cast<int64_t>(j) * kBlockN) * p.k_row_stride + h * p.k_head_stride;
    const elem_bits* vb = p.v + (k0 + static_cast<int64_t>(j) * kBlockN) * p.v_row_stride + h * p.v_head_stride;
    const int64_t img_off = (static_cast<int64_t>(h) * p.n_slots + slot) * kImageElems;
    const int valid = Sk - j * kBlockN;                    // keys of this block inside the sequence
    uint4 val[4];                                          // requested together with K's rows
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int u = tid + 256 * i, key = u >> 4, d0 = (u & 15) * 8;
        val[i] = make_uint4(0, 0, 0, 0);
        if (key < valid) val[i] = *reinterpret_cast<const uint4*>(vb + key * p.v_row_stride + d0);
    }
    write_k_image(kb, p.k_row_stride, valid, p.kimg + img_off, tid);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int u = tid + 256 * i;
        *reinterpret_cast<uint4*>(vt + (u >> 4) * kVPitch + (u & 15) * 8) = val[i];
    }
    __syncthreads();
    for (int u = tid; u < 1024; u += 256) {
        const int dt = u >> 7, cc = (u >> 6) & 1, lane = u & 63;
        const int r = lane & 15, g = lane >> 4;
        const elem_bits* column = vt + 16 * dt + r;
        uint32_t w[4];
#pragma unroll
        for (int jj = 0; jj < 8; jj += 2) {
            const int key_a = 32 * cc + (jj < 4 ? 4 * g + jj : 16 + 4 * g + jj - 4);
            w[jj >> 1] = static_cast<uint32_t>(column[key_a * kVPitch]) | (static_cast<uint32_t>(column[(key_a + 1) * kVPitch]) << 16);
        }
        *reinterpret_cast<uint4*>(p.vimg + img_off + u * 8) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}
inline PackParams pack_params(const void* k, const void* v, const int32_t* cu_seqlens_k, void* workspace, int batch, int64_t total_k,
                              int num_heads_k, const int64_t* k_strides, const int64_t* v_strides, unsigned* in_step) {
    PackParams p{};
    p.n_slots = image_slots(total_k, batch);
    p.k = static_cast<const elem_bits*>(k);
    p.v = static_cast<const elem_bits*>(v);
    p.kimg = static_cast<elem_bits*>(workspace);
    p.vimg = p.kimg + p.n_slots * num_heads_k * kImageElems;
    p.cu_seqlens_k = cu_seqlens_k;
    p.k_row_stride = k_strides[0]; p.k_head_stride = k_strides[1];
    p.v_row_stride = v_strides[0]; p.v_head_stride = v_strides[1];
    p.in_step = in_step;
    return p;
}
// What the images ask of k and v.
int check_pack(const void* k, const void* v, const int32_t* cu_seqlens_k, const void* workspace, size_t workspace_bytes, int batch,
               int64_t total_k, int num_heads_k, int max_seqlen_k, const int64_t* k_strides, const int64_t* v_strides);
// Launches the packing pre-pass.  workspace receives [K image | V image].  in_step: counters of in_step.h to clear, or null.
int launch_pack(hipStream_t st, const void* k, const void* v, const int32_t* cu_seqlens_k, void* workspace,
                size_t workspace_bytes, int batch, int64_t total_k, int num_heads_k, int max_seqlen_k,
                const int64_t* k_strides, const int64_t* v_strides, unsigned* in_step = nullptr);

}  // namespace IV2_NS
