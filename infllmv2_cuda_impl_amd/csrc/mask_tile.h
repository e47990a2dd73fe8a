// Block masks: their words from an index list, and their transposition, a 64 x 64 bit tile at a time.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// Row `row` of topk_idx (rows, k) int32 as words (rows, n64) uint64, by one wavefront of a workgroup whose wavefronts all come here.  Each lane ORs
// its indices into an LDS copy of the row's words (ds_or_b64), then the first n64 lanes store the row: every input index is read exactly once
// and every output word is written exactly once.
static __device__ __forceinline__ void topk_row_words(const int32_t* __restrict__ idx, uint64_t* __restrict__ out, int64_t row, int64_t rows, int k, int n64,
                                                      unsigned long long* words, int lane) {
    for (int w = lane; w < n64; w += 64) words[w] = 0ull;
    __syncthreads();
    if (row < rows) {
        const int32_t* src = idx + row * k;
        const int limit = n64 * 64;
        for (int i = lane; i < k; i += 64) {
            const int v = src[i];
            if (v >= 0 && v < limit) atomicOr(&words[v >> 6], 1ull << (v & 63));
        }
    }
    __syncthreads();
    if (row < rows) {
        for (int w = lane; w < n64; w += 64) out[row * n64 + w] = words[w];
    }
}

// bwd[h, kb, w] bit u = fwd[h, 64 w + u, kb / 64] bit (kb % 64).  One wavefront takes one tile: lane u holds the forward word of token
// 64 w + u, 64 ballots produce the 64 backward words of the tile, lane b stores word b.
static __device__ __forceinline__ void transpose_mask_tile(const uint64_t* __restrict__ fwd, uint64_t* __restrict__ bwd, int64_t tile, int lane, int heads,
                                                           int64_t total_q, int n64_fwd, int k_blocks, int n64_bwd) {
    const int64_t tiles_per_head = static_cast<int64_t>(n64_bwd) * n64_fwd;
    if (tile >= tiles_per_head * heads) return;              // uniform per wavefront
    const int h = static_cast<int>(tile / tiles_per_head);
    const int64_t rem = tile - h * tiles_per_head;
    const int w = static_cast<int>(rem / n64_fwd);           // 64-token group
    const int c = static_cast<int>(rem - static_cast<int64_t>(w) * n64_fwd);   // forward word column
    const int64_t tok = static_cast<int64_t>(w) * 64 + lane;
    uint64_t mine = 0;
    if (tok < total_q) mine = fwd[(static_cast<int64_t>(h) * total_q + tok) * n64_fwd + c];
    uint64_t result = 0;
#pragma unroll
    for (int b = 0; b < 64; ++b) {
        const uint64_t col = __builtin_amdgcn_ballot_w64(((mine >> b) & 1ull) != 0);
        if (lane == b) result = col;
    }
    const int kb = c * 64 + lane;
    if (kb < k_blocks) bwd[(static_cast<int64_t>(h) * k_blocks + kb) * n64_bwd + w] = result;
}
