// What a decode step of a layer leaves behind besides its output: the new token's rows in the K/V caches, the lengths, and the compressed keys that the
// token completes.  Kept by a workgroup of the step's first launch per (sequence, KV head): Stage 1's (stage1_decode.hip), or the attention's where a
// step selects every block (decode.hip).
#pragma once
#include "common.h"
#include <type_traits>

namespace IV2_NS {

struct S1DecodeStep {
    const elem_bits* knew;           // (batch, Hk, 128) with strides
    const elem_bits* vnew;
    elem_bits* kcache;
    elem_bits* vcache;
    elem_bits* fine;                 // the compressed caches (S1DecodeParams' k and c), to be written
    elem_bits* coarse;
    int64_t kn_batch, kn_head, vn_batch, vn_head;
    int64_t kc_batch, kc_row, kc_head, vc_batch, vc_row, vc_head;
    const int* lens;                 // tokens held before the step; null: host_len for every sequence
    int host_len;
    int* new_lens;                   // (batch) each: tokens and compressed keys held afterwards
    int* fine_lens;
    int* coarse_lens;
    int capacity, fine_capacity, coarse_capacity;
    int kernel_f, stride_f, kernel_c, stride_c;
    int with_scores;                 // 0: no query, no records (a step that does not score)
};

__device__ __forceinline__ int s1d_windows(int len, int kernel_size, int stride) {
    return len >= kernel_size ? (len - kernel_size) / stride + 1 : 0;
}
// rows a compressed cache holds after the step and the row this token completes (-1: none); the rules of
// infllmv2_compress_keys_cache with max_new_rows = 1
__device__ __forceinline__ int s1d_step_rows(int len, int capacity, int kernel_size, int stride, int out_capacity, int& added) {
    const int first = s1d_windows(len, kernel_size, stride);
    int rows = s1d_windows(len + 1 < capacity ? len + 1 : capacity, kernel_size, stride);
    rows = rows < out_capacity ? rows : out_capacity;
    rows = rows < first + 1 ? rows : first + 1;
    added = rows > first ? first : -1;
    return rows;
}
// One column of the mean of K rows [j stride, j stride + kernel_size) of one head: an fp32 sum in window order divided by
// kernel_size, rounded once, as compress.hip computes it.  The window's last row is the new token (that is why it is complete
// now) and comes from the caller.  Rows are requested 64 (32) at a time before they are added up.  A column per lane, over two
// wavefronts, because a lone wavefront is bound by the instructions it issues: two columns per lane, unpacked, took 640 of them.
__device__ __forceinline__ elem_bits s1d_window_mean(const S1DecodeStep& t, int b, int h, int j, int kernel_size, int stride, int col) {
    const elem_bits* row = t.kcache + b * t.kc_batch + static_cast<int64_t>(j) * stride * t.kc_row + h * t.kc_head + col;
    const elem_bits newest = t.knew[b * t.kn_batch + h * t.kn_head + col];
    float sum = 0.f;
    int left = kernel_size;
    auto chunk = [&](auto size) {
        constexpr int kRows = decltype(size)::value;
        for (; left >= kRows; left -= kRows) {
            elem_bits w[kRows];
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                w[i] = *row;
                row += t.kc_row;
                asm volatile("" : "+v"(row));                  // one running address, not one scalar pair per row
            }
            if (left == kRows) w[kRows - 1] = newest;
#pragma unroll
            for (int i = 0; i < kRows; ++i) sum += elem_to_f32(w[i]);
        }
    };
    chunk(std::integral_constant<int, 64>{});
    chunk(std::integral_constant<int, 32>{});
    chunk(std::integral_constant<int, 1>{});
    return f32_to_elem_hw(sum / static_cast<float>(kernel_size));
}

// What a step leaves behind for one sequence and KV head, by a workgroup of its own: the new token's rows (rows), the lengths, the compressed keys it completes
// (the coarse one only where nobody else forms it: coarse_too).  Of its threads the first 128 have a column of the fine key each, and those from
// coarse_from on, which may be the same, one of the coarse key.
struct S1DecodeStrides {                                        // of the compressed caches
    int64_t fine_batch, fine_row, fine_head, coarse_batch, coarse_row, coarse_head;
};
__device__ __forceinline__ void s1d_keep_caches(const S1DecodeStrides& p, const S1DecodeStep& t, int b, int h, int len, int rows_f, int rows_c, int add_f,
                                                int add_c, int tid, bool rows, bool coarse_too, int coarse_from) {
    const int g = tid >> 4, n = tid & 15;
    if (rows && tid < 32 && len < t.capacity) {
        const elem_bits* src = g == 0 ? t.knew + b * t.kn_batch + h * t.kn_head : t.vnew + b * t.vn_batch + h * t.vn_head;
        elem_bits* dst = g == 0 ? t.kcache + b * t.kc_batch + len * t.kc_row + h * t.kc_head
                                : t.vcache + b * t.vc_batch + len * t.vc_row + h * t.vc_head;
        *reinterpret_cast<uint4*>(dst + 8 * n) = *reinterpret_cast<const uint4*>(src + 8 * n);
    }
    if (h == 0 && tid == 0) {
        if (t.new_lens) t.new_lens[b] = len + 1;
        t.fine_lens[b] = rows_f;
        t.coarse_lens[b] = rows_c;
    }
    if (add_f >= 0 && tid < kHeadDim)
        t.fine[b * p.fine_batch + add_f * p.fine_row + h * p.fine_head + tid] = s1d_window_mean(t, b, h, add_f, t.kernel_f, t.stride_f, tid);
    const int col = tid - coarse_from;
    if (add_c >= 0 && coarse_too && col >= 0 && col < kHeadDim)
        t.coarse[b * p.coarse_batch + add_c * p.coarse_row + h * p.coarse_head + col] = s1d_window_mean(t, b, h, add_c, t.kernel_c, t.stride_c, col);
}

}  // namespace IV2_NS
