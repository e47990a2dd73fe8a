// Compressed keys for Stage 1 (gfx950): row j of a sequence is the mean of its K rows
// [stride*j, stride*j + kernel_size), full windows only.
//
// The reference leaves this step to its callers; the rule is the one its tests use to build the
// Stage-1 inputs (compress_tensor / calc_chunks_with_stride, tests/test_stage1_compressed_lse.py:16-99:
// windows that fit entirely inside a sequence, mean over the window, result in the input dtype).
// The mean is an fp32 sum taken in window order divided by kernel_size, rounded once to bf16.
//
// Small: K is read once from memory (the overlap of the windows hits in cache) and the output is 1/stride of its size, so
// for prompts of a few thousand tokens what counts is latency: how many round trips to memory a workgroup makes, and
// how many launches there are.
#include "common.h"
#include "kv_image.h"
#include "infllmv2_hip.h"

namespace IV2_NS {

__device__ __forceinline__ int compressed_rows(int len, int kernel_size, int stride) {
    return len >= kernel_size ? (len - kernel_size) / stride + 1 : 0;
}

// One set of compressed keys of packed sequences.  (The host passes two where a caller wants two sets of one K.)
struct CompressParams {
    const elem_bits* k;
    elem_bits* out;
    const int* cu_k;
    int* cu_out;
    int64_t k_row_stride, k_head_stride;
    int num_heads, units_per_head;   // 16-byte units of one head (head_dim / 8)
    int kernel_size, stride;
    int first_row;                   // rows before this one are left alone (appending to a buffer of compressed keys)
    int rows_per_wg;                 // output rows of one workgroup
};

constexpr int kCompressRowsPerWg = 8;
constexpr int kCompressThreads = 256;
constexpr int kCompressUnits = 16;           // units of one output row a workgroup works on: 128 elements
constexpr int kCompressMaxLds = 49152;       // the K rows a workgroup stages: 192 rows of 256 bytes
constexpr int kCompressPieces = kCompressMaxLds / 16 / kCompressThreads;      // of 16 bytes, per thread

// A workgroup takes rows_per_wg consecutive output rows of one KV head (128 elements of it).  Their windows are one
// stretch of (rows - 1) * stride + kernel_size K rows: it goes into LDS with every load in flight at once, and then
// one thread per two output elements adds its columns in window order.  Summing straight from memory, a window walked
// row by row is a chain of kernel_size round trips: 26 us for the two sets of 2048 tokens where this takes 4.3.
// Windows longer than the LDS holds are added up in several such steps.
// kColumns (two rows and fewer, the wide windows): a thread adds one element's column instead, so that all four wavefronts add and the chain
// has half the instructions: 128 keys every 64, two rows to a workgroup, of 2048 tokens 5.04 -> 4.53 us, of 131 072 19.5 -> 18.8.
template <bool kColumns>
__device__ __forceinline__ void compress_rows_of_head(const CompressParams& p, int wg, uint4* stage) {
    const int b = blockIdx.y, head = blockIdx.z / ((p.units_per_head + kCompressUnits - 1) / kCompressUnits);
    const int u0 = (blockIdx.z % ((p.units_per_head + kCompressUnits - 1) / kCompressUnits)) * kCompressUnits;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int k0 = p.cu_k[b];
    const int rows = compressed_rows(p.cu_k[b + 1] - k0, p.kernel_size, p.stride);
    // rows of the sequences before this one, added up by every wavefront for itself
    int before = 0;
    for (int i = lane; i < b; i += 64) before += compressed_rows(p.cu_k[i + 1] - p.cu_k[i], p.kernel_size, p.stride);
    if (b > 0) {
#pragma unroll
        for (int off = 32; off; off >>= 1) before += __shfl_xor(before, off);
    }
    if (wg == 0 && blockIdx.z == 0 && tid == 0) {
        p.cu_out[b + 1] = before + rows;
        if (b == 0) p.cu_out[0] = 0;
    }
    const int j0 = p.first_row + wg * p.rows_per_wg;
    if (j0 >= rows) return;                                    // uniform per workgroup
    const int nrows = rows - j0 < p.rows_per_wg ? rows - j0 : p.rows_per_wg;
    const int nu = p.units_per_head - u0 < kCompressUnits ? p.units_per_head - u0 : kCompressUnits;
    const elem_bits* src = p.k + (static_cast<int64_t>(k0) + static_cast<int64_t>(j0) * p.stride) * p.k_row_stride +
                           head * p.k_head_stride + u0 * 8;
    const int span = (nrows - 1) * p.stride + p.kernel_size;   // K rows the windows cover
    const int step = kCompressMaxLds / (kCompressUnits * 16);  // K rows staged at a time
    float acc[kCompressRowsPerWg / 4][2];                      // rows wave, wave + 4; elements 2 lane, 2 lane + 1
#pragma unroll
    for (int r = 0; r < kCompressRowsPerWg / 4; ++r) acc[r][0] = acc[r][1] = 0.f;
    for (int base = 0; base < span; base += step) {
        const int staged = span - base < step ? span - base : step;
        if (base > 0) __syncthreads();
        // All of them are requested before the first is waited for.  A set on its own, us, four at a time before: 32 keys every 16 of 2048 tokens 4.11 -> 4.03, of 131 072
        // 15.8 -> 15.2; 128 every 64 4.80 -> 4.88, 21.3 -> 19.7; both in one launch, 2048 tokens, 0.35 less.
        uint4 piece[kCompressPieces];
#pragma unroll
        for (int t = 0; t < kCompressPieces; ++t) {
            const int it = tid + t * kCompressThreads, i = it / kCompressUnits, u = it % kCompressUnits;
            piece[t] = make_uint4(0, 0, 0, 0);
            if (i < staged && u < nu) piece[t] = *reinterpret_cast<const uint4*>(src + (base + i) * p.k_row_stride + u * 8);
        }
#pragma unroll
        for (int t = 0; t < kCompressPieces; ++t)
            if ((tid + t * kCompressThreads) / kCompressUnits < staged) stage[tid + t * kCompressThreads] = piece[t];
        __syncthreads();
        if constexpr (kColumns) {
            const int row = tid >> 7;
            if (row < nrows) {
                int lo = row * p.stride - base, hi = lo + p.kernel_size;
                lo = lo < 0 ? 0 : lo;
                hi = hi < staged ? hi : staged;
                const elem_bits* column = reinterpret_cast<const elem_bits*>(stage) + (tid & 127);
#pragma unroll 16
                for (int i = lo; i < hi; ++i) acc[0][0] += elem_to_f32(column[i * kCompressUnits * 8]);
            }
            continue;
        }
        const uint32_t* words = reinterpret_cast<const uint32_t*>(stage) + lane;
#pragma unroll
        for (int r = 0; r < kCompressRowsPerWg / 4; ++r) {
            const int row = wave + 4 * r;
            if (row < nrows) {                                 // uniform per wavefront
                int lo = row * p.stride - base, hi = lo + p.kernel_size;
                lo = lo < 0 ? 0 : lo;
                hi = hi < staged ? hi : staged;
#pragma unroll 8
                for (int i = lo; i < hi; ++i) {
                    const uint32_t w = words[i * kCompressUnits * 4];
                    acc[r][0] += elem_lo_to_f32(w);
                    acc[r][1] += elem_hi_to_f32(w);
                }
            }
        }
    }
    const float n = static_cast<float>(p.kernel_size);
    if constexpr (kColumns) {
        const int row = tid >> 7, col = tid & 127;
        if (row < nrows && col < nu * 8)
            p.out[((static_cast<int64_t>(before) + j0 + row) * p.num_heads + head) * p.units_per_head * 8 + u0 * 8 + col] = f32_to_elem_hw(acc[0][0] / n);
        return;
    }
    if (lane >= nu * 4) return;
#pragma unroll
    for (int r = 0; r < kCompressRowsPerWg / 4; ++r) {
        const int row = wave + 4 * r;
        if (row < nrows) {
            elem_bits* dst = p.out + ((static_cast<int64_t>(before) + j0 + row) * p.num_heads + head) * p.units_per_head * 8 + u0 * 8;
            reinterpret_cast<uint32_t*>(dst)[lane] = pack_elem2(acc[r][0] / n, acc[r][1] / n);
        }
    }
}

template <bool kColumns>
__global__ __launch_bounds__(kCompressThreads)
void compress_keys_kernel(const CompressParams p) {
    extern __shared__ uint4 stage[];
    compress_rows_of_head<kColumns>(p, blockIdx.x, stage);
}
// two sets of the same K in one launch: the first wgs_a workgroups of a sequence and head belong to set a
template <bool kColumnsA, bool kColumnsB>
__global__ __launch_bounds__(kCompressThreads)
void compress_keys_pair_kernel(const CompressParams pa, const CompressParams pb, int wgs_a) {
    extern __shared__ uint4 stage[];
    if (static_cast<int>(blockIdx.x) < wgs_a) compress_rows_of_head<kColumnsA>(pa, blockIdx.x, stage);
    else compress_rows_of_head<kColumnsB>(pb, blockIdx.x - wgs_a, stage);
}

// ... and the block images of the Stage-2 forward behind them: what prefill needs of K and V before its first scores, in one launch.  Bound by
// latency like the two it replaces: a whole prefill of 512 tokens 34.9 -> 32.5 us, of 2048 (64 blocks selected) 83.9 -> 80.7, of 16 384 1363 -> 1356.
template <bool kColumnsA, bool kColumnsB>
__global__ __launch_bounds__(kCompressThreads)
void compress_keys_and_pack_kernel(const CompressParams pa, const CompressParams pb, const PackParams pk, int wgs_a, int wgs_ab) {
    extern __shared__ uint4 stage[];
    const int wg = blockIdx.x;
    if (wg < wgs_a) compress_rows_of_head<kColumnsA>(pa, wg, stage);
    else if (wg < wgs_ab) compress_rows_of_head<kColumnsB>(pb, wg - wgs_a, stage);
    else pack_block(pk, wg - wgs_ab, blockIdx.y, blockIdx.z, reinterpret_cast<elem_bits*>(stage));
}
static_assert(kCompressThreads == 256, "the packing part is written for workgroups of 256");

// The same means for per-sequence key caches (decode): sequence b's keys are rows [0, new_lens[b]) of kcache[b]; the
// rows of its compressed-key cache that windows completed since old_lens[b] tokens are written, the others are left
// alone.  A decode step (one more token) completes at most one window per set.
struct CompressCacheParams {
    const elem_bits* k;
    elem_bits* out;
    const int* old_lens;             // null: 0 for every sequence (build everything)
    const int* new_lens;
    int* out_lens;                   // null, or (batch): rows the compressed cache holds afterwards
    int64_t k_batch, k_row, k_head, o_batch, o_row, o_head;
    int units_per_row, units_per_head;
    int kernel_size, stride;
    int k_capacity;                  // rows of one sequence's key cache: a length beyond it is read as the capacity
    int out_capacity;                // rows of one sequence's compressed cache: nothing is written beyond it
    int max_new_rows;                // rows this call may add per sequence (what the launch covers)
};

// Rows sequence b's compressed cache holds after the call, and the first of them this call writes: the windows
// completed by new_lens[b] tokens, never more than the output has rows, the key cache has windows, or the launch
// covers (so that the reported length never includes a row that was not written).
__device__ __forceinline__ void cache_row_range(const CompressCacheParams& p, int b, int& first, int& rows) {
    int new_len = p.new_lens[b];
    if (new_len > p.k_capacity) new_len = p.k_capacity;
    rows = compressed_rows(new_len, p.kernel_size, p.stride);
    first = p.old_lens ? compressed_rows(p.old_lens[b], p.kernel_size, p.stride) : 0;
    if (first < 0) first = 0;
    if (rows > p.out_capacity) rows = p.out_capacity;
    if (rows > first + p.max_new_rows) rows = first + p.max_new_rows;
}

__global__ __launch_bounds__(256)
void compress_keys_cache_kernel(const CompressCacheParams p) {
    const int b = blockIdx.y;
    int first, rows;
    cache_row_range(p, b, first, rows);
    if (blockIdx.x == 0 && threadIdx.x == 0 && p.out_lens) p.out_lens[b] = rows;
    const int j0 = first + blockIdx.x * kCompressRowsPerWg;
    for (int item = threadIdx.x; item < kCompressRowsPerWg * p.units_per_row; item += 256) {
        const int j = j0 + item / p.units_per_row;
        if (j >= rows) break;
        const int u = item % p.units_per_row;
        const int head = u / p.units_per_head, piece = u % p.units_per_head;
        const elem_bits* src = p.k + b * p.k_batch + static_cast<int64_t>(j) * p.stride * p.k_row + head * p.k_head + piece * 8;
        float acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = 0.f;
        for (int i = 0; i < p.kernel_size; ++i) {
            const uint4 raw = *reinterpret_cast<const uint4*>(src + i * p.k_row);
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[2 * e] += elem_lo_to_f32(w[e]);
                acc[2 * e + 1] += elem_hi_to_f32(w[e]);
            }
        }
        const float n = static_cast<float>(p.kernel_size);
        uint4 o;
        o.x = pack_elem2(acc[0] / n, acc[1] / n);
        o.y = pack_elem2(acc[2] / n, acc[3] / n);
        o.z = pack_elem2(acc[4] / n, acc[5] / n);
        o.w = pack_elem2(acc[6] / n, acc[7] / n);
        *reinterpret_cast<uint4*>(p.out + b * p.o_batch + static_cast<int64_t>(j) * p.o_row + head * p.o_head + piece * 8) = o;
    }
}

// The append of a decode step: few new rows per sequence, so one workgroup takes ONE output row (32 of its 16-byte
// units).  Walking the window row by row in one thread, as the kernel above does, is a chain of kernel_size dependent
// round trips to memory when only a handful of threads are busy; here the whole window goes into LDS with every
// load in flight at once, and then one thread per output element adds its column in window order (the same fp32
// additions in the same order as above: the results are the same bits).
constexpr int kAppendUnits = 32;
constexpr int kAppendMaxLds = 65536;

// new_row: which of the sequence's new rows this workgroup takes
__device__ __forceinline__ void append_one_row(const CompressCacheParams& p, int new_row, uint4* window) {
    const int b = blockIdx.y;
    int first, rows;
    cache_row_range(p, b, first, rows);
    if (new_row == 0 && blockIdx.z == 0 && threadIdx.x == 0 && p.out_lens) p.out_lens[b] = rows;
    const int j = first + new_row;
    if (j >= rows) return;                                     // uniform per workgroup
    const int u0 = blockIdx.z * kAppendUnits;
    const int nu = p.units_per_row - u0 < kAppendUnits ? p.units_per_row - u0 : kAppendUnits;
    const elem_bits* src = p.k + b * p.k_batch + static_cast<int64_t>(j) * p.stride * p.k_row;
    const int items = p.kernel_size * kAppendUnits;
#pragma unroll 8
    for (int it = threadIdx.x; it < items; it += 256) {
        const int i = it / kAppendUnits, uu = it % kAppendUnits;
        if (uu < nu) {
            const int u = u0 + uu;
            window[it] = *reinterpret_cast<const uint4*>(src + i * p.k_row + (u / p.units_per_head) * p.k_head + (u % p.units_per_head) * 8);
        }
    }
    __syncthreads();
    const int uu = threadIdx.x >> 3, e = threadIdx.x & 7;      // one thread per (unit, element)
    if (uu >= nu) return;
    const elem_bits* col = reinterpret_cast<const elem_bits*>(window) + uu * 8 + e;
    float acc = 0.f;
    for (int i = 0; i < p.kernel_size; ++i) acc += elem_to_f32(col[i * kAppendUnits * 8]);
    const float n = static_cast<float>(p.kernel_size);
    const int u = u0 + uu;
    p.out[b * p.o_batch + static_cast<int64_t>(j) * p.o_row + (u / p.units_per_head) * p.o_head + (u % p.units_per_head) * 8 + e] =
        f32_to_elem(acc / n);
}

__global__ __launch_bounds__(256)
void compress_keys_cache_append_kernel(const CompressCacheParams p) {
    extern __shared__ uint4 window[];                          // [kernel_size][kAppendUnits]
    append_one_row(p, blockIdx.x, window);
}
// the appends to two compressed caches of the same key cache (the fine and the coarse keys of a decode step) in one
// launch: the first rows_a workgroups of a sequence belong to cache a
__global__ __launch_bounds__(256)
void compress_keys_cache_append_pair_kernel(const CompressCacheParams pa, const CompressCacheParams pb, int rows_a) {
    extern __shared__ uint4 window[];                          // [the larger kernel_size][kAppendUnits]
    if (static_cast<int>(blockIdx.x) < rows_a) append_one_row(pa, blockIdx.x, window);
    else append_one_row(pb, blockIdx.x - rows_a, window);
}

}  // namespace IV2_NS

using namespace IV2_NS;

namespace {

// workgroups per sequence and head; one writes cu_out in any case
int row_workgroups(const CompressParams& p, int max_seqlen_k) {
    const int max_rows = max_seqlen_k >= p.kernel_size ? (max_seqlen_k - p.kernel_size) / p.stride + 1 : 0;
    return max_rows > p.first_row ? (max_rows - p.first_row + p.rows_per_wg - 1) / p.rows_per_wg : 1;
}
// checks and parameters of one set of compressed keys of packed sequences; wgs: workgroups per sequence and head
int packed_params(const char* who, CompressParams& p, int& wgs, const void* k, void* out, const int32_t* cu_seqlens_k,
                  int32_t* cu_seqlens_out, int batch, int max_seqlen_k, int num_heads_k, int head_dim,
                  int64_t k_row_stride, int64_t k_head_stride, int kernel_size, int stride, int first_row) {
    IV2_CHECK(batch > 0 && batch <= 65535 && max_seqlen_k >= 0, "%s: bad batch or max_seqlen_k", who);
    IV2_CHECK(kernel_size > 0 && stride > 0 && first_row >= 0, "%s: kernel_size and stride must be positive", who);
    IV2_CHECK(k && out && cu_seqlens_k && cu_seqlens_out, "%s: null pointer", who);
    IV2_CHECK(head_dim > 0 && head_dim % 8 == 0 && num_heads_k > 0, "%s: head_dim must be a multiple of 8", who);
    IV2_CHECK(static_cast<int64_t>(num_heads_k) * ((head_dim + 127) / 128) <= 65535, "%s: too many heads", who);
    IV2_CHECK(reinterpret_cast<uintptr_t>(k) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
              k_row_stride % 8 == 0 && k_head_stride % 8 == 0, "%s: k and out must be 16-byte aligned, strides multiples of 8", who);
    p = CompressParams{};
    p.k = static_cast<const elem_bits*>(k);
    p.out = static_cast<elem_bits*>(out);
    p.cu_k = cu_seqlens_k; p.cu_out = cu_seqlens_out;
    p.k_row_stride = k_row_stride; p.k_head_stride = k_head_stride;
    p.num_heads = num_heads_k; p.units_per_head = head_dim / 8;
    p.kernel_size = kernel_size; p.stride = stride; p.first_row = first_row;
    // as many rows as fit the staging buffer together (8 at 32/16, 2 at 128/64), at least one
    const int lds_rows = kCompressMaxLds / (kCompressUnits * 16);
    const int rows_per_wg = lds_rows > kernel_size ? (lds_rows - kernel_size) / stride + 1 : 1;
    p.rows_per_wg = rows_per_wg < kCompressRowsPerWg ? rows_per_wg : kCompressRowsPerWg;
    wgs = row_workgroups(p, max_seqlen_k);
    return 0;
}
// Half the rows to a workgroup where the launch leaves compute units idle: its windows then arrive with fewer loads to a thread, and the K rows
// that two workgroups both read come from the L2.  A set on its own gains as long as all of
// its workgroups run at once (kCompressAlone), us: 32 keys every 16 of 2048 tokens and two KV heads 4.18 -> 3.45, of 32 768 5.77 -> 4.36 (1024
// workgroups), of 131 072 15.1 -> 16.4 (4096, not taken); 128 every 64 4.53 -> 4.15, 6.93 -> 5.50, 18.8 -> 23.5 (not taken).  Two sets share
// the LDS of the larger (kCompressTogether): 2048 tokens 4.67 -> 4.29, 9000 tokens (560 workgroups) 5.06 -> 4.91, 20 011 (1250) 6.4 -> 6.8
// (not taken).
constexpr int64_t kCompressAlone = 1024, kCompressTogether = 640;
void halve_rows(CompressParams& p, int& wgs, int max_seqlen_k) {
    if (p.rows_per_wg > 1) p.rows_per_wg /= 2;
    wgs = row_workgroups(p, max_seqlen_k);
}
size_t staging_bytes(const CompressParams& p) {
    const int64_t rows = static_cast<int64_t>(p.rows_per_wg - 1) * p.stride + p.kernel_size;
    const int64_t bytes = rows * kCompressUnits * 16;
    return static_cast<size_t>(bytes < kCompressMaxLds ? bytes : kCompressMaxLds);
}
// A column to a thread instead of two to a lane (compress_rows_of_head): with two rows and fewer half of the wavefronts would have no row
bool by_columns(const CompressParams& p) { return p.rows_per_wg <= 2; }
unsigned head_parts(const CompressParams& p) {
    return static_cast<unsigned>(p.num_heads * ((p.units_per_head + kCompressUnits - 1) / kCompressUnits));
}

}  // namespace

extern "C" int IV2_ENTRY(infllmv2_compress_keys)(void* stream, const void* k, void* out, const int32_t* cu_seqlens_k,
                                      int32_t* cu_seqlens_out, int batch, int max_seqlen_k, int num_heads_k,
                                      int head_dim, int64_t k_row_stride, int64_t k_head_stride, int kernel_size,
                                      int stride, int first_row) {
    CompressParams p;
    int wgs;
    if (int rc = packed_params("compress_keys", p, wgs, k, out, cu_seqlens_k, cu_seqlens_out, batch, max_seqlen_k, num_heads_k,
                               head_dim, k_row_stride, k_head_stride, kernel_size, stride, first_row))
        return rc;
    if (2 * static_cast<int64_t>(wgs) * batch * head_parts(p) <= kCompressAlone) halve_rows(p, wgs, max_seqlen_k);
    auto kernel = by_columns(p) ? compress_keys_kernel<true> : compress_keys_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(wgs, batch, head_parts(p)), dim3(kCompressThreads), staging_bytes(p), static_cast<hipStream_t>(stream), p);
    IV2_LAUNCH_CHECK();
    return 0;
}

extern "C" int IV2_ENTRY(infllmv2_compress_keys_pair)(void* stream, const void* k, void* out_a, void* out_b, const int32_t* cu_seqlens_k,
                                           int32_t* cu_seqlens_out_a, int32_t* cu_seqlens_out_b, int batch, int max_seqlen_k,
                                           int num_heads_k, int head_dim, int64_t k_row_stride, int64_t k_head_stride,
                                           int kernel_size_a, int stride_a, int kernel_size_b, int stride_b) {
    CompressParams pa, pb;
    int wgs_a, wgs_b;
    if (int rc = packed_params("compress_keys_pair", pa, wgs_a, k, out_a, cu_seqlens_k, cu_seqlens_out_a, batch, max_seqlen_k,
                               num_heads_k, head_dim, k_row_stride, k_head_stride, kernel_size_a, stride_a, 0))
        return rc;
    if (int rc = packed_params("compress_keys_pair", pb, wgs_b, k, out_b, cu_seqlens_k, cu_seqlens_out_b, batch, max_seqlen_k,
                               num_heads_k, head_dim, k_row_stride, k_head_stride, kernel_size_b, stride_b, 0))
        return rc;
    if (2 * (static_cast<int64_t>(wgs_a) + wgs_b) * batch * head_parts(pa) <= kCompressTogether) {
        halve_rows(pa, wgs_a, max_seqlen_k);
        halve_rows(pb, wgs_b, max_seqlen_k);
    }
    const size_t lds = staging_bytes(pa) > staging_bytes(pb) ? staging_bytes(pa) : staging_bytes(pb);
    auto kernel = by_columns(pa) ? (by_columns(pb) ? compress_keys_pair_kernel<true, true> : compress_keys_pair_kernel<true, false>)
                                 : (by_columns(pb) ? compress_keys_pair_kernel<false, true> : compress_keys_pair_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(wgs_a + wgs_b, batch, head_parts(pa)), dim3(kCompressThreads), lds,
                       static_cast<hipStream_t>(stream), pa, pb, wgs_a);
    IV2_LAUNCH_CHECK();
    return 0;
}

extern "C" int IV2_ENTRY(infllmv2_compress_keys_and_pack)(void* stream, const void* k, const void* v, void* out_a, void* out_b,
                                               const int32_t* cu_seqlens_k, int32_t* cu_seqlens_out_a, int32_t* cu_seqlens_out_b,
                                               void* workspace, size_t workspace_bytes, int batch, int64_t total_k, int max_seqlen_k,
                                               int num_heads_k, int head_dim, const int64_t* k_strides, const int64_t* v_strides,
                                               int kernel_size_a, int stride_a, int kernel_size_b, int stride_b) {
    CompressParams pa, pb;
    int wgs_a, wgs_b;
    IV2_CHECK(head_dim == kHeadDim, "compress_keys_and_pack: this build only supports head_dim 128 (got %d)", head_dim);
    if (int rc = packed_params("compress_keys_and_pack", pa, wgs_a, k, out_a, cu_seqlens_k, cu_seqlens_out_a, batch, max_seqlen_k,
                               num_heads_k, head_dim, k_strides[0], k_strides[1], kernel_size_a, stride_a, 0))
        return rc;
    if (int rc = packed_params("compress_keys_and_pack", pb, wgs_b, k, out_b, cu_seqlens_k, cu_seqlens_out_b, batch, max_seqlen_k,
                               num_heads_k, head_dim, k_strides[0], k_strides[1], kernel_size_b, stride_b, 0))
        return rc;
    if (int rc = check_pack(k, v, cu_seqlens_k, workspace, workspace_bytes, batch, total_k, num_heads_k, max_seqlen_k, k_strides, v_strides))
        return rc;
    const PackParams pk = pack_params(k, v, cu_seqlens_k, workspace, batch, total_k, num_heads_k, k_strides, v_strides, nullptr);
    const int blocks = total_k == 0 ? 0 : (max_seqlen_k + kBlockN - 1) / kBlockN;
    if ((2 * (static_cast<int64_t>(wgs_a) + wgs_b) + blocks) * batch * num_heads_k <= kCompressTogether) {
        halve_rows(pa, wgs_a, max_seqlen_k);
        halve_rows(pb, wgs_b, max_seqlen_k);
    }
    size_t lds = staging_bytes(pa) > staging_bytes(pb) ? staging_bytes(pa) : staging_bytes(pb);
    if (lds < kPackElems * sizeof(elem_bits)) lds = kPackElems * sizeof(elem_bits);
    auto kernel = by_columns(pa) ? (by_columns(pb) ? compress_keys_and_pack_kernel<true, true> : compress_keys_and_pack_kernel<true, false>)
                                 : (by_columns(pb) ? compress_keys_and_pack_kernel<false, true> : compress_keys_and_pack_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(wgs_a + wgs_b + blocks, batch, num_heads_k), dim3(kCompressThreads), lds,
                       static_cast<hipStream_t>(stream), pa, pb, pk, wgs_a, wgs_a + wgs_b);
    IV2_LAUNCH_CHECK();
    return 0;
}

namespace {

// checks and parameters of one compressed cache; 0 or an error code
int cache_params(const char* who, CompressCacheParams& p, const void* kcache, void* out_cache, const int32_t* old_lens,
                 const int32_t* new_lens, int32_t* out_lens, int batch, int max_new_rows, int num_heads_k, int head_dim,
                 const int64_t* kcache_strides, const int64_t* out_strides, int kernel_size, int stride, int kcache_rows,
                 int out_rows) {
    IV2_CHECK(batch > 0 && batch <= 65535 && max_new_rows >= 0, "%s: bad batch or max_new_rows", who);
    IV2_CHECK(kcache_rows >= 0 && out_rows >= 0, "%s: negative cache capacity", who);
    IV2_CHECK(kernel_size > 0 && stride > 0, "%s: kernel_size and stride must be positive", who);
    IV2_CHECK(kcache && out_cache && new_lens, "%s: null pointer", who);
    IV2_CHECK(head_dim > 0 && head_dim % 8 == 0 && num_heads_k > 0, "%s: head_dim must be a multiple of 8", who);
    IV2_CHECK(reinterpret_cast<uintptr_t>(kcache) % 16 == 0 && reinterpret_cast<uintptr_t>(out_cache) % 16 == 0,
              "%s: caches must be 16-byte aligned", who);
    for (int s = 0; s < 3; ++s)
        IV2_CHECK(kcache_strides[s] % 8 == 0 && out_strides[s] % 8 == 0, "%s: strides must be multiples of 8 elements", who);
    p = CompressCacheParams{};
    p.k = static_cast<const elem_bits*>(kcache);
    p.out = static_cast<elem_bits*>(out_cache);
    p.old_lens = old_lens; p.new_lens = new_lens; p.out_lens = out_lens;
    p.k_batch = kcache_strides[0]; p.k_row = kcache_strides[1]; p.k_head = kcache_strides[2];
    p.o_batch = out_strides[0]; p.o_row = out_strides[1]; p.o_head = out_strides[2];
    p.units_per_row = num_heads_k * head_dim / 8; p.units_per_head = head_dim / 8;
    p.kernel_size = kernel_size; p.stride = stride;
    p.k_capacity = kcache_rows; p.out_capacity = out_rows; p.max_new_rows = max_new_rows;
    return 0;
}
size_t append_window_bytes(const CompressCacheParams& p) { return static_cast<size_t>(p.kernel_size) * kAppendUnits * 16; }
// a decode step's append: one workgroup per new row and 32 units
bool append_shaped(const CompressCacheParams& p) {
    return p.max_new_rows >= 1 && p.max_new_rows <= 8 && append_window_bytes(p) <= kAppendMaxLds;
}
int launch_cache(hipStream_t st, const CompressCacheParams& p, int batch) {
    if (append_shaped(p)) {
        const dim3 grid(p.max_new_rows, batch, (p.units_per_row + kAppendUnits - 1) / kAppendUnits);
        hipLaunchKernelGGL(compress_keys_cache_append_kernel, grid, dim3(256), append_window_bytes(p), st, p);
        IV2_LAUNCH_CHECK();
        return 0;
    }
    // at least one workgroup per sequence so that out_lens is always written
    const int groups = p.max_new_rows > 0 ? (p.max_new_rows + kCompressRowsPerWg - 1) / kCompressRowsPerWg : 1;
    hipLaunchKernelGGL(compress_keys_cache_kernel, dim3(groups, batch), dim3(256), 0, st, p);
    IV2_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int IV2_ENTRY(infllmv2_compress_keys_cache)(void* stream, const void* kcache, void* out_cache, const int32_t* old_lens,
                                            const int32_t* new_lens, int32_t* out_lens, int batch, int max_new_rows,
                                            int num_heads_k, int head_dim, const int64_t* kcache_strides,
                                            const int64_t* out_strides, int kernel_size, int stride,
                                            int kcache_rows, int out_rows) {
    CompressCacheParams p;
    if (int rc = cache_params("compress_keys_cache", p, kcache, out_cache, old_lens, new_lens, out_lens, batch, max_new_rows,
                              num_heads_k, head_dim, kcache_strides, out_strides, kernel_size, stride, kcache_rows, out_rows))
        return rc;
    return launch_cache(static_cast<hipStream_t>(stream), p, batch);
}

extern "C" int IV2_ENTRY(infllmv2_compress_keys_cache_pair)(void* stream, const void* kcache, void* out_cache_a, void* out_cache_b,
                                                 const int32_t* old_lens, const int32_t* new_lens, int32_t* out_lens_a,
                                                 int32_t* out_lens_b, int batch, int max_new_rows_a, int max_new_rows_b,
                                                 int num_heads_k, int head_dim, const int64_t* kcache_strides,
                                                 const int64_t* out_strides_a, const int64_t* out_strides_b,
                                                 int kernel_size_a, int stride_a, int kernel_size_b, int stride_b,
                                                 int kcache_rows, int out_rows_a, int out_rows_b) {
    CompressCacheParams pa, pb;
    if (int rc = cache_params("compress_keys_cache_pair", pa, kcache, out_cache_a, old_lens, new_lens, out_lens_a, batch,
                              max_new_rows_a, num_heads_k, head_dim, kcache_strides, out_strides_a, kernel_size_a, stride_a,
                              kcache_rows, out_rows_a))
        return rc;
    if (int rc = cache_params("compress_keys_cache_pair", pb, kcache, out_cache_b, old_lens, new_lens, out_lens_b, batch,
                              max_new_rows_b, num_heads_k, head_dim, kcache_strides, out_strides_b, kernel_size_b, stride_b,
                              kcache_rows, out_rows_b))
        return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (append_shaped(pa) && append_shaped(pb)) {
        const size_t lds = append_window_bytes(pa) > append_window_bytes(pb) ? append_window_bytes(pa) : append_window_bytes(pb);
        const dim3 grid(pa.max_new_rows + pb.max_new_rows, batch, (pa.units_per_row + kAppendUnits - 1) / kAppendUnits);
        hipLaunchKernelGGL(compress_keys_cache_append_pair_kernel, grid, dim3(256), lds, st, pa, pb, pa.max_new_rows);
        IV2_LAUNCH_CHECK();
        return 0;
    }
    if (int rc = launch_cache(st, pa, batch)) return rc;
    return launch_cache(st, pb, batch);
}
