// The host side of the package's operators, `infllmv2_cuda_impl_amd._host`: argument checks, output and scratch
// allocation, and the calls into the C ABI, in native code.  The Python modules keep the public signatures and
// documentation and call in here once per operator.
//
// Why native: a decode step of a few sequences is 20 to 40 us of kernels, and the same work done in Python (some sixty
// attribute look-ups for the checks, ctypes arrays for the strides, a device context) took 25 to 30 us per operator, so
// the device waited for the host.  Here an operator costs its launches and its allocations.
//
// Checks and messages follow the reference's (csrc/flash_attn/flash_api.cpp); each function names the lines it follows.
// Nothing is kept between calls except which devices have been checked.
#include <torch/extension.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <algorithm>
#include <atomic>
#include <optional>
#include <string>
#include <tuple>

#include "infllmv2_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
constexpr int64_t kHeadDim = 128;
constexpr int64_t kBlock = 64;

void check_rc(int rc, const char* what) {
    if (rc != 0) {
        const char* msg = infllmv2_last_error();
        TORCH_CHECK(false, (msg && msg[0]) ? std::string(msg) : std::string(what) + " failed with code " + std::to_string(rc));
    }
}

using DeviceGuard = c10::hip::HIPGuardMasqueradingAsCUDA;
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream(); }

// Devices found to be gfx950 so far: asking the runtime for a device's properties takes longer than a launch.
constexpr int kMaxDevices = 64;
std::atomic<bool> g_device_ok[kMaxDevices];

void require_gpu(const Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda(), name, " must be on a GPU device (got ", t.device(), "); this library has no CPU path");
    const int dev = t.get_device();
    if (dev >= 0 && dev < kMaxDevices && g_device_ok[dev].load(std::memory_order_relaxed)) return;
    check_rc(infllmv2_check_device(dev), "infllmv2_check_device");
    if (dev >= 0 && dev < kMaxDevices) g_device_ok[dev].store(true, std::memory_order_relaxed);
}

bool is_half(const Tensor& t) { return t.scalar_type() == at::kHalf; }
void require_16bit(const Tensor& t) {
    TORCH_CHECK(t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16, "FlashAttention only support fp16 and bf16 data type");
}
void* ptr(const Tensor& t) { return t.data_ptr(); }
const void* ptr(const OptTensor& t) { return t.has_value() ? t->data_ptr() : nullptr; }
const int32_t* iptr(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }
const int32_t* iptr(const OptTensor& t) { return t.has_value() ? static_cast<const int32_t*>(t->data_ptr()) : nullptr; }
int as_int(int64_t v) { return static_cast<int>(v); }

Tensor bytes_on(const Tensor& like, size_t n) { return at::empty({static_cast<int64_t>(std::max<size_t>(n, 256))}, like.options().dtype(at::kByte)); }

struct S2 { int64_t v[2]; };
struct S3 { int64_t v[3]; };
S2 rows_heads(const Tensor& t) { return {{t.stride(0), t.stride(1)}}; }                          // (rows, heads, d)
S3 batch_rows_heads(const Tensor& t) { return {{t.stride(0), t.stride(1), t.stride(2)}}; }        // (batch, rows, heads, d)
S3 grouped(const Tensor& t, int64_t group) { return {{t.stride(0), t.stride(1), group * t.stride(1)}}; }   // {token, head in group, KV head} of (T, Hq, d)

// query heads per KV head, checked against what the kernels serve
int64_t group_size(int64_t heads, int64_t heads_k) {
    TORCH_CHECK(heads_k > 0 && heads % heads_k == 0, "Number of heads in key/value must divide number of heads in query");
    const int64_t g = heads / heads_k;
    TORCH_CHECK(g == 1 || g == 2 || g == 4 || g == 8 || g == 16, "this build requires 1, 2, 4, 8 or 16 query heads per key/value head");
    return g;
}

// input checks of mha_varlen_fwd (flash_api.cpp:552-616) that apply to this build
void check_qkv(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k, bool same_kv_len) {
    require_16bit(q);
    TORCH_CHECK(k.scalar_type() == q.scalar_type(), "query and key must have the same dtype");
    TORCH_CHECK(v.scalar_type() == q.scalar_type(), "query and value must have the same dtype");
    TORCH_CHECK(cu_q.scalar_type() == at::kInt, "cu_seqlens_q must have dtype int32");
    TORCH_CHECK(cu_k.scalar_type() == at::kInt, "cu_seqlens_k must have dtype int32");
    require_gpu(q, "q"); require_gpu(k, "k"); require_gpu(v, "v");
    require_gpu(cu_q, "cu_seqlens_q"); require_gpu(cu_k, "cu_seqlens_k");
    for (const Tensor* t : {&q, &k, &v})
        TORCH_CHECK(t->numel() == 0 || t->stride(-1) == 1, "Input tensor must have contiguous last dimension");
    TORCH_CHECK(cu_q.is_contiguous(), "cu_seqlens_q must be contiguous");
    TORCH_CHECK(cu_k.is_contiguous(), "cu_seqlens_k must be contiguous");
    const int64_t batch = cu_q.numel() - 1;
    TORCH_CHECK(batch > 0, "batch size must be positive");
    TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3, "q, k, v must have shape (total, nheads, headdim)");
    const int64_t d = q.size(2);
    TORCH_CHECK(d <= 256, "FlashAttention forward only supports head dimension at most 256");
    TORCH_CHECK(d % 8 == 0, "query, key, value, and out_ must have a head_size that is a multiple of 8");
    TORCH_CHECK(k.size(1) > 0 && q.size(1) % k.size(1) == 0, "Number of heads in key/value must divide number of heads in query");
    TORCH_CHECK(k.size(2) == d && v.size(1) == k.size(1) && v.size(2) == k.size(2) && (!same_kv_len || v.size(0) == k.size(0)),
                "k and v must have shape (total_k, num_heads_k, head_size)");
    TORCH_CHECK(cu_k.numel() == batch + 1, "cu_seqlens_k must have shape (batch_size + 1)");
    TORCH_CHECK(d == kHeadDim, "this build only supports head dimension 128");
    group_size(q.size(1), k.size(1));
}

// ---- compressed keys ---------------------------------------------------------------------------------------------
int64_t windows(int64_t len, int64_t kernel_size, int64_t stride) { return len >= kernel_size ? (len - kernel_size) / stride + 1 : 0; }
// rows to allocate for compressed keys: their number for one sequence, an upper bound for a packed batch
int64_t compressed_rows_bound(int64_t batch, int64_t total_k, int64_t max_seqlen_k, int64_t kernel_size, int64_t stride) {
    return batch == 1 ? windows(max_seqlen_k, kernel_size, stride) : total_k / stride + 1;
}
void check_compress(const Tensor& k, const Tensor& cu) {
    require_gpu(k, "k");
    require_16bit(k);
    TORCH_CHECK(k.dim() == 3 && k.stride(-1) == 1, "k must have shape (total_k, num_heads_k, head_size) with a contiguous last dimension");
    TORCH_CHECK(cu.scalar_type() == at::kInt && cu.is_contiguous(), "cu_seqlens_k must be a contiguous int32 tensor");
}
Tensor compressed_buffer(const Tensor& k, int64_t rows) {                  // never a null pointer
    return at::empty({std::max<int64_t>(rows, 1), k.size(1), k.size(2)}, k.options());
}

std::tuple<Tensor, Tensor> compress_keys(const Tensor& k, const Tensor& cu, int64_t max_seqlen_k, int64_t kernel_size, int64_t stride,
                                         const OptTensor& out_, int64_t first_row) {
    check_compress(k, cu);
    TORCH_CHECK(stride > 0, "compress_keys: kernel_size and stride must be positive");
    const int64_t batch = cu.numel() - 1;
    const int64_t rows = compressed_rows_bound(batch, k.size(0), max_seqlen_k, kernel_size, stride);
    Tensor backing;
    if (out_.has_value()) {
        TORCH_CHECK(out_->dim() == 3 && out_->size(0) >= rows && out_->size(1) == k.size(1) && out_->size(2) == k.size(2) &&
                    out_->is_contiguous() && out_->scalar_type() == k.scalar_type(),
                    "out must be a contiguous (rows, num_heads_k, head_size) buffer of k's dtype");
        backing = *out_;
    } else {
        backing = compressed_buffer(k, rows);
    }
    DeviceGuard guard(k.device());
    Tensor cu_out = at::empty({batch + 1}, cu.options());
    auto fn = is_half(k) ? infllmv2_compress_keys_f16 : infllmv2_compress_keys;
    check_rc(fn(stream_of(k), ptr(k), ptr(backing), iptr(cu), static_cast<int32_t*>(ptr(cu_out)), as_int(batch), as_int(max_seqlen_k),
                as_int(k.size(1)), as_int(k.size(2)), k.stride(0), k.stride(1), as_int(kernel_size), as_int(stride), as_int(first_row)),
             "compress_keys");
    return {out_.has_value() || backing.size(0) == rows ? backing : backing.narrow(0, 0, rows), cu_out};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> compress_keys_pair(const Tensor& k, const Tensor& cu, int64_t max_seqlen_k, int64_t ks_a,
                                                              int64_t st_a, int64_t ks_b, int64_t st_b) {
    check_compress(k, cu);
    TORCH_CHECK(st_a > 0 && st_b > 0, "compress_keys_pair: kernel_size and stride must be positive");
    const int64_t batch = cu.numel() - 1;
    const int64_t rows_a = compressed_rows_bound(batch, k.size(0), max_seqlen_k, ks_a, st_a);
    const int64_t rows_b = compressed_rows_bound(batch, k.size(0), max_seqlen_k, ks_b, st_b);
    DeviceGuard guard(k.device());
    Tensor a = compressed_buffer(k, rows_a), b = compressed_buffer(k, rows_b);
    Tensor cu_a = at::empty({batch + 1}, cu.options()), cu_b = at::empty({batch + 1}, cu.options());
    auto fn = is_half(k) ? infllmv2_compress_keys_pair_f16 : infllmv2_compress_keys_pair;
    check_rc(fn(stream_of(k), ptr(k), ptr(a), ptr(b), iptr(cu), static_cast<int32_t*>(ptr(cu_a)), static_cast<int32_t*>(ptr(cu_b)),
                as_int(batch), as_int(max_seqlen_k), as_int(k.size(1)), as_int(k.size(2)), k.stride(0), k.stride(1), as_int(ks_a),
                as_int(st_a), as_int(ks_b), as_int(st_b)), "compress_keys_pair");
    return {a.size(0) == rows_a ? a : a.narrow(0, 0, rows_a), cu_a, b.size(0) == rows_b ? b : b.narrow(0, 0, rows_b), cu_b};
}

// Whether the block images of (k, v) are made where k is compressed, for attention that follows the scores of q: k and v are as the attention takes them,
// without a copy, no sequence is so long that it is walked in step (with counters that the packing clears for the one launch behind it), and the images
// are still in the 256 MB behind the L2s when the scores have read q.  Packed just before the walk, they are there in any case: with 64 blocks
// selected and 2 KV heads of 16 query heads, packing early gains 3 us of a whole prefill at 512 and 2048 tokens, 7 at 12 288 and 16 384 (128 MiB of q) and
// nothing at 20 480 to 28 672, and at 32 768 the walk is 1 to 3 % slower for it (2.81 -> 2.87 ms).
constexpr int64_t kPackEarlyBytes = 128ll << 20;
bool pack_early(const Tensor& q, const Tensor& k, const Tensor& v, int64_t max_seqlen_k) {
    if (q.numel() * q.element_size() > kPackEarlyBytes || max_seqlen_k > INFLLMV2_IN_STEP_KEYS) return false;
    const auto fits = [](const Tensor& t) {
        return t.stride(2) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
    };
    return k.dim() == 3 && k.size(2) == kHeadDim && v.dim() == 3 && v.sizes() == k.sizes() && v.scalar_type() == k.scalar_type() &&
           v.device() == k.device() && fits(k) && fits(v);
}
Tensor image_workspace(const Tensor& k, int64_t batch) { return bytes_on(k, infllmv2_kv_image_bytes(k.size(0), as_int(batch), as_int(k.size(1)))); }

// compress_keys_pair that also gives the block images of (k, v)
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> compress_keys_and_pack(const Tensor& k, const Tensor& v, const Tensor& cu, int64_t max_seqlen_k,
                                                                          int64_t ks_a, int64_t st_a, int64_t ks_b, int64_t st_b) {
    check_compress(k, cu);
    TORCH_CHECK(st_a > 0 && st_b > 0, "compress_keys_pair: kernel_size and stride must be positive");
    const int64_t batch = cu.numel() - 1;
    const int64_t rows_a = compressed_rows_bound(batch, k.size(0), max_seqlen_k, ks_a, st_a);
    const int64_t rows_b = compressed_rows_bound(batch, k.size(0), max_seqlen_k, ks_b, st_b);
    DeviceGuard guard(k.device());
    Tensor a = compressed_buffer(k, rows_a), b = compressed_buffer(k, rows_b);
    Tensor cu_a = at::empty({batch + 1}, cu.options()), cu_b = at::empty({batch + 1}, cu.options());
    Tensor images = image_workspace(k, batch);
    const S2 ks = rows_heads(k), vs = rows_heads(v);
    auto fn = is_half(k) ? infllmv2_compress_keys_and_pack_f16 : infllmv2_compress_keys_and_pack;
    check_rc(fn(stream_of(k), ptr(k), ptr(v), ptr(a), ptr(b), iptr(cu), static_cast<int32_t*>(ptr(cu_a)), static_cast<int32_t*>(ptr(cu_b)),
                ptr(images), static_cast<size_t>(images.numel()), as_int(batch), k.size(0), as_int(max_seqlen_k), as_int(k.size(1)),
                as_int(k.size(2)), ks.v, vs.v, as_int(ks_a), as_int(st_a), as_int(ks_b), as_int(st_b)), "compress_keys_and_pack");
    return {a.size(0) == rows_a ? a : a.narrow(0, 0, rows_a), cu_a, b.size(0) == rows_b ? b : b.narrow(0, 0, rows_b), cu_b, images};
}

// ---- Stage 1 (mha_varlen_fwd_stage1, flash_api.cpp:784-1049) ---------------------------------------------------------
// a key set with no rows (sequences shorter than one window) still needs a valid pointer; no row of it is read
Tensor readable(const Tensor& t) { return t.size(0) > 0 ? t : at::zeros({1, t.size(1), t.size(2)}, t.options()); }

// {batch, row, head} strides of packed keys (one "batch" for all) or of per-sequence caches
S3 key_strides(const Tensor& t, bool packed) { return packed ? S3{{0, t.stride(0), t.stride(1)}} : batch_rows_heads(t); }

struct Pool { const int32_t* cache_lens = nullptr; int64_t cache_len = 0, out_len = 0, local_blocks = 0, init_blocks = 0, block_size = kBlock, stride = 16; };

// Stage 1 with one query token per sequence: the compressed keys of every sequence are scored in parallel runs
void stage1_decode(const Tensor& q, int64_t batch, const Tensor& k, const Tensor& v, const int32_t* cu_q, const int32_t* cu_k,
                   const int32_t* k_lens, const int32_t* cu_v, const int32_t* v_lens, int64_t max_k, int64_t max_v, double scale, bool causal,
                   const Tensor& out, int64_t head_stride, int64_t row_stride, const Pool* pool) {
    const int64_t hq = q.size(-2), hk = k.size(-2), group = hq / hk;
    Tensor ws = bytes_on(q, infllmv2_stage1_decode_workspace_bytes(as_int(batch), as_int(hk), as_int(max_k), as_int(max_v)));
    const int64_t qs[3] = {q.stride(0), q.stride(-2), group * q.stride(-2)};
    const S3 ks = key_strides(k, cu_k != nullptr), vs = key_strides(v, cu_v != nullptr);
    const Pool none;
    const Pool& p = pool ? *pool : none;
    const int per = as_int(p.block_size / p.stride);
    auto fn = is_half(q) ? infllmv2_stage1_decode_f16 : infllmv2_stage1_decode;
    check_rc(fn(stream_of(q), ptr(q), ptr(k), ptr(v), ptr(out), cu_q, cu_k, k_lens, cu_v, v_lens, ptr(ws), static_cast<size_t>(ws.numel()),
                as_int(batch), as_int(hq), as_int(hk), as_int(q.size(-1)), as_int(max_k), as_int(max_v), qs, ks.v, vs.v, head_stride,
                row_stride, static_cast<float>(scale), causal ? 1 : 0, pool ? 1 : 0, p.cache_lens, as_int(p.cache_len), as_int(p.out_len),
                per + 1, per, 1, as_int(p.block_size), as_int(p.local_blocks), as_int(p.init_blocks)), "stage1_decode");
}

// the operator's signature has no max_seqlen_v: a sequence's coarse keys are never more than its fine keys, nor than all rows
int64_t max_rows_bound(const Tensor& v, int64_t batch, int64_t max_seqlen_k) { return batch > 1 ? std::min(v.size(0), max_seqlen_k) : v.size(0); }

void check_stage1(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k, const Tensor& cu_v) {
    check_qkv(q, k, v, cu_q, cu_k, false);
    TORCH_CHECK(cu_v.scalar_type() == at::kInt, "cu_seqlens_v must have dtype int32");
    TORCH_CHECK(cu_v.is_contiguous(), "cu_seqlens must be contiguous");
    TORCH_CHECK(cu_v.numel() == cu_q.numel(), "cu_seqlens_v must have shape (batch_size + 1)");
}

// Scores (Hk, total_q, max_seqlen_k).  The reference zero-fills a (Hk, T, round128(max_k)) buffer, slices it and replaces
// NaNs in a further pass (flash_api.cpp:941, infllmv2_sparse_attention.py:587-589); here the kernel defines every element
// once and produces no NaN.
Tensor stage1_scores(const Tensor& q, const Tensor& k_, const Tensor& v_, const Tensor& cu_q, const Tensor& cu_k, const Tensor& cu_v,
                     int64_t max_q, int64_t max_k, double scale, bool causal) {
    check_stage1(q, k_, v_, cu_q, cu_k, cu_v);
    DeviceGuard guard(q.device());
    const int64_t batch = cu_q.numel() - 1, total_q = q.size(0), hq = q.size(1), hk = k_.size(1);
    const Tensor k = readable(k_), v = readable(v_);
    Tensor out = at::empty({hk, total_q, max_k}, q.options());
    if (max_q == 1 && total_q > 0) {
        // decode: one query per sequence, so the parallelism has to come from the keys
        stage1_decode(q, batch, k, v, iptr(cu_q), iptr(cu_k), nullptr, iptr(cu_v), nullptr, max_k, max_rows_bound(v, batch, max_k), scale,
                      causal, out, out.stride(0), out.stride(1), nullptr);
    } else {
        const S3 qs = grouped(q, hq / hk);
        const S2 ks = rows_heads(k), vs = rows_heads(v);
        auto fn = is_half(q) ? infllmv2_varlen_fwd_stage1_f16 : infllmv2_varlen_fwd_stage1;
        check_rc(fn(stream_of(q), ptr(q), ptr(k), ptr(v), ptr(out), iptr(cu_q), iptr(cu_k), iptr(cu_v), as_int(batch), total_q, as_int(hq),
                    as_int(hk), as_int(q.size(2)), as_int(max_q), as_int(max_k), qs.v, ks.v, vs.v, out.stride(0), out.stride(1),
                    static_cast<float>(scale), causal ? 1 : 0), "varlen_fwd_stage1");
    }
    return out;
}

// Scores pooled onto key blocks in the same launch: (Hk, total_q, out_len)
Tensor stage1_pooled(const Tensor& q, const Tensor& k_, const Tensor& v_, const Tensor& cu_q, const Tensor& cu_k, const Tensor& cu_v,
                     int64_t max_q, int64_t max_k, double scale, bool causal, int64_t out_len, const OptTensor& cache_lens,
                     int64_t cache_len, int64_t local_blocks, int64_t init_blocks, int64_t block_size, int64_t stride) {
    check_stage1(q, k_, v_, cu_q, cu_k, cu_v);
    const int64_t batch = cu_q.numel() - 1, total_q = q.size(0), hq = q.size(1), hk = k_.size(1);
    TORCH_CHECK(!cache_lens.has_value() || (cache_lens->scalar_type() == at::kInt && cache_lens->numel() == batch && cache_lens->is_contiguous()),
                "cache_lens must be a contiguous int32 tensor of shape (batch_size)");
    DeviceGuard guard(q.device());
    const Tensor k = readable(k_), v = readable(v_);
    Tensor out = at::empty({hk, total_q, out_len}, q.options());
    if (max_q == 1 && total_q > 0 && out_len > 0) {
        const Pool pool{iptr(cache_lens), cache_len, out_len, local_blocks, init_blocks, block_size, stride};
        stage1_decode(q, batch, k, v, iptr(cu_q), iptr(cu_k), nullptr, iptr(cu_v), nullptr, max_k, max_rows_bound(v, batch, max_k), scale,
                      causal, out, out.stride(0), out.stride(1), &pool);
        return out;
    }
    const S3 qs = grouped(q, hq / hk);
    const S2 ks = rows_heads(k), vs = rows_heads(v);
    const int per = as_int(block_size / stride);
    auto fn = is_half(q) ? infllmv2_varlen_fwd_stage1_pooled_f16 : infllmv2_varlen_fwd_stage1_pooled;
    check_rc(fn(stream_of(q), ptr(q), ptr(k), ptr(v), ptr(out), iptr(cu_q), iptr(cu_k), iptr(cu_v), iptr(cache_lens), as_int(cache_len),
                as_int(batch), total_q, as_int(hq), as_int(hk), as_int(q.size(2)), as_int(max_q), as_int(max_k), qs.v, ks.v, vs.v,
                as_int(out_len), static_cast<float>(scale), causal ? 1 : 0, per + 1, per, 1, as_int(block_size), as_int(local_blocks),
                as_int(init_blocks)), "varlen_fwd_stage1_pooled");
    return out;
}

// The mask words of the topk best blocks of that, causal and without cached tokens, in the same launch.
Tensor stage1_selected(const Tensor& q, const Tensor& k_, const Tensor& v_, const Tensor& cu_q, const Tensor& cu_k, const Tensor& cu_v, int64_t max_q,
                       int64_t max_k, double scale, int64_t out_len, int64_t local_blocks, int64_t init_blocks, int64_t block_size, int64_t stride,
                       int64_t topk, int64_t n64) {
    check_stage1(q, k_, v_, cu_q, cu_k, cu_v);
    const int64_t batch = cu_q.numel() - 1, total_q = q.size(0), hq = q.size(1), hk = k_.size(1);
    DeviceGuard guard(q.device());
    const Tensor k = readable(k_), v = readable(v_);
    Tensor mask = at::empty({hk, total_q, n64}, q.options().dtype(at::kLong));
    const S3 qs = grouped(q, hq / hk);
    const S2 ks = rows_heads(k), vs = rows_heads(v);
    const int per = as_int(block_size / stride);
    auto fn = is_half(q) ? infllmv2_varlen_fwd_stage1_selected_f16 : infllmv2_varlen_fwd_stage1_selected;
    check_rc(fn(stream_of(q), ptr(q), ptr(k), ptr(v), static_cast<uint64_t*>(mask.data_ptr()), iptr(cu_q), iptr(cu_k), iptr(cu_v), as_int(batch), total_q,
                as_int(hq), as_int(hk), as_int(q.size(2)), as_int(max_q), as_int(max_k), qs.v, ks.v, vs.v, as_int(out_len), static_cast<float>(scale),
                per + 1, per, 1, as_int(block_size), as_int(local_blocks), as_int(init_blocks), as_int(topk), as_int(n64)), "varlen_fwd_stage1_selected");
    return mask;
}

Tensor stage1_kvcache(const Tensor& q, const Tensor& fine, const Tensor& coarse, const Tensor& fine_lens, const Tensor& coarse_lens,
                      const Tensor& cache_seqlens, int64_t local_blocks, int64_t init_blocks, std::optional<int64_t> max_cache_len,
                      int64_t block_size, int64_t stride, double scale, bool causal, bool pooled) {
    TORCH_CHECK(q.dim() == 4 && q.size(1) == 1, "q must have shape (batch_size, 1, num_heads, head_size)");
    require_16bit(q);
    TORCH_CHECK(fine.scalar_type() == q.scalar_type() && coarse.scalar_type() == q.scalar_type(), "query and key must have the same dtype");
    const int64_t batch = q.size(0), hq = q.size(2), d = q.size(3);
    require_gpu(q, "q"); require_gpu(fine, "k_fine_cache"); require_gpu(coarse, "k_coarse_cache");
    for (const Tensor* t : {&q, &fine, &coarse}) TORCH_CHECK(t->stride(-1) == 1, "Input tensor must have contiguous last dimension");
    TORCH_CHECK(fine.dim() == 4 && coarse.dim() == 4 && fine.size(0) == batch && coarse.size(0) == batch,
                "compressed-key caches must have shape (batch_size, rows, num_heads_k, head_size)");
    const int64_t hk = fine.size(2);
    group_size(hq, hk);
    TORCH_CHECK(d == kHeadDim && coarse.size(2) == hk && coarse.size(3) == d && fine.size(3) == d, "this build requires head dimension 128");
    const std::pair<const Tensor*, const char*> lens[] = {{&fine_lens, "fine_lens"}, {&coarse_lens, "coarse_lens"}, {&cache_seqlens, "cache_seqlens"}};
    for (const auto& [t, name] : lens)
        TORCH_CHECK(t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) == batch && t->is_contiguous(), name,
                    " must be a contiguous int32 tensor of shape (batch_size)");
    DeviceGuard guard(q.device());
    const int64_t rows_f = fine.size(1), rows_c = coarse.size(1);
    const Tensor q3 = q.select(1, 0);
    if (!pooled) {
        Tensor out = at::empty({batch, hk, rows_f}, q.options());
        stage1_decode(q3, batch, fine, coarse, nullptr, nullptr, iptr(fine_lens), nullptr, iptr(coarse_lens), rows_f, rows_c, scale, causal,
                      out, out.stride(1), out.stride(0), nullptr);
        return out;
    }
    const int64_t held = max_cache_len.has_value() ? *max_cache_len : (rows_f + 1) * stride + block_size;
    const int64_t out_len = (1 + held + block_size - 1) / block_size;
    Tensor out = at::empty({batch, hk, out_len}, q.options());
    const Pool pool{iptr(cache_seqlens), 0, out_len, local_blocks, init_blocks, block_size, stride};
    stage1_decode(q3, batch, fine, coarse, nullptr, nullptr, iptr(fine_lens), nullptr, iptr(coarse_lens), rows_f, rows_c, scale, causal, out,
                  out.stride(1), out.stride(0), &pool);
    return out;
}

// ---- pooling, top-k, masks ---------------------------------------------------------------------------------------
// inputs whose last dimension is dense and whose rows and heads are regularly strided are used in place
Tensor row_strided(const Tensor& x) {
    return x.stride(-1) == 1 && x.stride(1) >= x.size(2) && x.stride(0) >= 0 ? x : x.contiguous();
}

Tensor max_pooling_1d(const Tensor& input, int64_t cache_len, int64_t local_blocks, int64_t init_blocks, int64_t block_size, int64_t stride) {
    require_gpu(input, "input");
    const Tensor x = row_strided(input);
    const int s = as_int(block_size / stride);
    const int64_t out_len = (x.size(1) + cache_len + block_size - 1) / block_size;
    DeviceGuard guard(x.device());
    Tensor out = at::empty({x.size(0), x.size(1), out_len}, x.options());
    check_rc(infllmv2_max_pooling_1d_strided(stream_of(x), ptr(x), ptr(out), is_half(x) ? 0 : 1, as_int(x.size(0)), as_int(x.size(1)),
                                             as_int(x.size(2)), x.stride(0), x.stride(1), as_int(out_len), as_int(cache_len), s + 1, s, 1,
                                             as_int(block_size), as_int(local_blocks), as_int(init_blocks)), "max_pooling_1d");
    return out;
}

Tensor max_pooling_1d_varlen(const Tensor& input, const Tensor& cu_q_, const Tensor& cu_k_, const Tensor& cache_lens_, int64_t max_q,
                             int64_t local_blocks, int64_t init_blocks, int64_t block_size, int64_t stride, int64_t max_cache_len) {
    require_gpu(input, "input");
    const Tensor x = row_strided(input);
    const Tensor cu_q = cu_q_.contiguous(), cu_k = cu_k_.contiguous(), cache_lens = cache_lens_.contiguous();
    const int s = as_int(block_size / stride);
    const int64_t out_len = (max_q + max_cache_len + block_size - 1) / block_size;
    DeviceGuard guard(x.device());
    Tensor out = at::empty({x.size(0), x.size(1), out_len}, x.options());
    check_rc(infllmv2_max_pooling_1d_varlen_strided(stream_of(x), ptr(x), ptr(out), iptr(cu_q), iptr(cu_k), iptr(cache_lens), is_half(x) ? 0 : 1,
                                                    as_int(cu_q.size(0) - 1), as_int(x.size(0)), as_int(x.size(1)), as_int(max_q),
                                                    as_int(x.size(2)), x.stride(0), x.stride(1), as_int(out_len), s + 1, s, 1,
                                                    as_int(block_size), as_int(local_blocks), as_int(init_blocks)), "max_pooling_1d_varlen");
    return out;
}

std::tuple<Tensor, OptTensor> topk_blocks(const Tensor& pooled, int64_t k, bool return_mask, bool by_index, bool drop_unreachable,
                                          std::optional<int64_t> words) {
    require_gpu(pooled, "pooled");
    const Tensor x = pooled.contiguous();
    const int64_t n = x.size(-1), n64 = words.has_value() ? *words : (n + 63) / 64;
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    int64_t rows = 1;
    for (size_t i = 0; i + 1 < shape.size(); ++i) rows *= shape[i];
    DeviceGuard guard(x.device());
    shape.back() = k;
    Tensor idx = at::empty(shape, x.options().dtype(at::kInt));
    OptTensor mask;
    if (return_mask) {
        shape.back() = n64;
        mask = at::empty(shape, x.options().dtype(at::kLong));
    }
    if (!return_mask && !by_index && !drop_unreachable) {
        check_rc(infllmv2_topk_blocks(stream_of(x), ptr(x), n, static_cast<int32_t*>(ptr(idx)), rows, as_int(n), as_int(k)), "topk_blocks");
        return {idx, mask};
    }
    check_rc(infllmv2_topk_select(stream_of(x), ptr(x), n, is_half(x) ? 0 : 1, static_cast<int32_t*>(ptr(idx)),
                                  mask.has_value() ? static_cast<uint64_t*>(mask->data_ptr()) : nullptr, rows, as_int(n), as_int(k),
                                  as_int(n64), by_index ? 1 : 0, drop_unreachable ? 1 : 0), "topk_select");
    return {idx, mask};
}

// The mask of the same selection, where nobody reads the list.
Tensor topk_mask(const Tensor& pooled, int64_t k, std::optional<int64_t> words) {
    require_gpu(pooled, "pooled");
    const Tensor x = pooled.contiguous();
    const int64_t n = x.size(-1), n64 = words.has_value() ? *words : (n + 63) / 64;
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    int64_t rows = 1;
    for (size_t i = 0; i + 1 < shape.size(); ++i) rows *= shape[i];
    shape.back() = n64;
    DeviceGuard guard(x.device());
    Tensor mask = at::empty(shape, x.options().dtype(at::kLong));
    check_rc(infllmv2_topk_mask(stream_of(x), ptr(x), n, is_half(x) ? 0 : 1, static_cast<uint64_t*>(ptr(mask)), rows, as_int(n), as_int(k), as_int(n64), 0),
             "topk_mask");
    return mask;
}

std::tuple<Tensor, Tensor> window_blocks(int64_t heads, int64_t rows, const Tensor& cu_q_, const OptTensor& positions_, int64_t max_q, int64_t max_position,
                                         int64_t local_blocks, int64_t init_blocks, int64_t block_size) {
    require_gpu(cu_q_, "cu_seqlens_q");
    const Tensor cu_q = cu_q_.contiguous();
    OptTensor positions;
    if (positions_.has_value()) positions = positions_->contiguous();
    TORCH_CHECK(cu_q.scalar_type() == at::kInt && (!positions.has_value() || (positions->scalar_type() == at::kInt && positions->size(0) == cu_q.size(0) - 1)),
                "window_blocks: int32 sequence starts and positions of as many sequences");
    const int64_t n = (max_q + max_position + block_size - 1) / block_size, n64 = (n + 63) / 64;
    DeviceGuard guard(cu_q.device());
    Tensor idx = at::empty({heads, rows, init_blocks + local_blocks + 1}, cu_q.options());
    Tensor mask = at::empty({heads, rows, n64}, cu_q.options().dtype(at::kLong));
    check_rc(infllmv2_window_blocks(stream_of(cu_q), static_cast<int32_t*>(ptr(idx)), static_cast<uint64_t*>(mask.data_ptr()), iptr(cu_q),
                                    positions.has_value() ? iptr(*positions) : nullptr, as_int(cu_q.size(0) - 1), as_int(heads), rows, as_int(n), as_int(n64), as_int(block_size), as_int(local_blocks),
                                    as_int(init_blocks)), "window_blocks");
    return {idx, mask};
}

Tensor topk_to_uint64(const Tensor& topk_idx, int64_t k_blocks, const OptTensor& buffer) {
    require_gpu(topk_idx, "topk_idx");
    const Tensor idx = topk_idx.contiguous();
    const int64_t n64 = (k_blocks + 63) / 64;
    c10::SmallVector<int64_t, 5> shape(idx.sizes().begin(), idx.sizes().end());
    const int64_t k = shape.back();
    int64_t rows = 1;
    for (size_t i = 0; i + 1 < shape.size(); ++i) rows *= shape[i];
    shape.back() = n64;
    DeviceGuard guard(idx.device());
    Tensor out;
    if (buffer.has_value() && buffer->sizes() == at::IntArrayRef(shape) && buffer->scalar_type() == at::kLong &&
        buffer->device() == idx.device() && buffer->is_contiguous())
        out = *buffer;
    else
        out = at::empty(shape, idx.options().dtype(at::kLong));
    check_rc(infllmv2_topk_to_uint64(stream_of(idx), iptr(idx), static_cast<uint64_t*>(ptr(out)), rows, as_int(k), as_int(k_blocks), as_int(n64)),
             "topk_to_uint64");
    return out;
}

// the selection front end: compressed keys, fused Stage 1 and pooling, top-k with the mask words
// Block scores (Hk, total_q, blocks) of packed queries, and how many mask words a row of the selection takes.  images: where the block
// images of (k, v) go, which are then made in the same launch as the compressed keys where pack_early says so.  mask: where the mask words of the topk best go, if
// the rows are short enough for the launch that makes the scores to choose among them; there are no scores then.
std::tuple<Tensor, int64_t> block_scores(const Tensor& q_, const Tensor& k, const Tensor& cu_q, const Tensor& cu_k, int64_t max_q,
                                         int64_t max_k, int64_t local_blocks, int64_t init_blocks, const OptTensor& cache_lens,
                                         int64_t max_cache_len, double scale, bool causal, int64_t kernel_size, int64_t stride,
                                         int64_t block_size, bool exact_lse, const Tensor* v = nullptr, OptTensor* images = nullptr,
                                         int64_t topk = 0, Tensor* mask = nullptr) {
    const Tensor q = q_.stride(-1) == 1 ? q_ : q_.contiguous();
    Tensor kf, cu_f, kc, cu_c;
    if (exact_lse) {
        std::tie(kf, cu_f) = compress_keys(k, cu_k, max_k, kernel_size, stride, std::nullopt, 0);
        kc = kf; cu_c = cu_f;
    } else if (images != nullptr && pack_early(q, k, *v, max_k)) {
        Tensor packed;
        std::tie(kf, cu_f, kc, cu_c, packed) = compress_keys_and_pack(k, *v, cu_k, max_k, kernel_size, stride, 4 * kernel_size, 4 * stride);
        *images = packed;
    } else {
        std::tie(kf, cu_f, kc, cu_c) = compress_keys_pair(k, cu_k, max_k, kernel_size, stride, 4 * kernel_size, 4 * stride);
    }
    const int64_t out_len = (max_q + max_cache_len + block_size - 1) / block_size;
    int64_t n64 = ((max_k + block_size - 1) / block_size + 63) / 64;
    if (n64 * 64 < out_len) n64 = (out_len + 63) / 64;                 // cached tokens widen the pooled rows beyond max_seqlen_k
    if (mask != nullptr && out_len > 0 && out_len <= INFLLMV2_STAGE1_SELECT_BLOCKS && max_q > 1) {
        *mask = stage1_selected(q, kf, kc, cu_q, cu_f, cu_c, max_q, windows(max_k, kernel_size, stride), scale, out_len, local_blocks, init_blocks, block_size,
                                stride, topk, n64);
        return {Tensor(), n64};
    }
    const Tensor pooled = stage1_pooled(q, kf, kc, cu_q, cu_f, cu_c, max_q, windows(max_k, kernel_size, stride), scale, causal, out_len, cache_lens,
                                        0, local_blocks, init_blocks, block_size, stride);
    return {pooled, n64};
}

std::tuple<Tensor, OptTensor> select_blocks(const Tensor& q, const Tensor& k, const Tensor& cu_q, const Tensor& cu_k, int64_t max_q,
                                            int64_t max_k, int64_t topk, int64_t local_blocks, int64_t init_blocks, const OptTensor& cache_lens,
                                            int64_t max_cache_len, double scale, bool causal, int64_t kernel_size, int64_t stride,
                                            int64_t block_size, bool exact_lse, bool return_mask, bool by_index, bool drop_unreachable) {
    const auto [pooled, n64] = block_scores(q, k, cu_q, cu_k, max_q, max_k, local_blocks, init_blocks, cache_lens, max_cache_len, scale, causal,
                                            kernel_size, stride, block_size, exact_lse);
    return topk_blocks(pooled, topk, return_mask, by_index, drop_unreachable, n64);
}

// The selection of plain prefill for a caller that goes on with the mask and attends to the same k and v: {an empty list whose width says how many
// blocks a row has at most, mask, the block images of (k, v) for varlen_fwd or none}.
std::tuple<Tensor, Tensor, OptTensor> select_mask(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu, int64_t max_len, int64_t topk,
                                                  int64_t local_blocks, int64_t init_blocks, double scale, int64_t kernel_size, int64_t stride,
                                                  int64_t block_size) {
    OptTensor images;
    Tensor mask;
    const int64_t blocks = (max_len + kBlock - 1) / kBlock;
    if (max_len > 1 && blocks <= topk && topk <= 2048 && block_size == kBlock && kernel_size > 0 && stride > 0 && block_size / stride == 4 && pack_early(q, k, v, max_len)) {
        // every row takes all blocks of its sequence: nothing to score
        check_compress(k, cu);
        check_qkv(q.stride(-1) == 1 ? q : q.contiguous(), k, v, cu, cu, true);
        DeviceGuard guard(k.device());
        const int64_t batch = cu.numel() - 1, n64 = (blocks + 63) / 64;
        images = image_workspace(k, batch);
        mask = at::empty({k.size(1), q.size(0), n64}, q.options().dtype(at::kLong));
        const S2 ks = rows_heads(k), vs = rows_heads(v);
        check_rc(infllmv2_pack_kv_and_first(stream_of(q), ptr(k), ptr(v), iptr(cu), ptr(*images), static_cast<size_t>(images->numel()), as_int(batch), k.size(0),
                                            as_int(k.size(1)), as_int(k.size(2)), as_int(max_len), ks.v, vs.v, static_cast<uint64_t*>(ptr(mask)),
                                            k.size(1) * q.size(0), as_int(blocks), as_int(n64)), "pack_kv_and_first");
        return {at::empty({k.size(1), 0, topk}, q.options().dtype(at::kInt)), mask, images};
    }
    const auto [pooled, n64] = block_scores(q, k, cu, cu, max_len, max_len, local_blocks, init_blocks, std::nullopt, 0, scale, true, kernel_size,
                                            stride, block_size, false, &v, &images, topk, &mask);
    if (!mask.defined()) mask = topk_mask(pooled, topk, n64);
    return {at::empty({k.size(1), 0, topk}, q.options().dtype(at::kInt)), mask, images};
}

// ---- Stage 2 (mha_varlen_fwd, flash_api.cpp:519-782; mha_varlen_bwd, :1278-1547) ---------------------------------------
// images: of (k, v), as select_mask gives them.  Returns {out, lse, packed mask or none}.  lse: (Hk, total_q * group) on the sparse path,
// (Hq, total_q) on the dense one.
std::tuple<Tensor, Tensor, OptTensor> varlen_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k,
                                                 int64_t max_q, int64_t max_k, double scale, bool causal, const OptTensor& topk_idx,
                                                 const OptTensor& block_mask, bool alike, const OptTensor& images) {
    check_qkv(q, k, v, cu_q, cu_k, true);
    DeviceGuard guard(q.device());
    const int64_t batch = cu_q.numel() - 1, total_q = q.size(0), hq = q.size(1), d = q.size(2), total_k = k.size(0), hk = k.size(1);
    const int64_t group = hq / hk;
    OptTensor mask, packed = images;                           // packed: the block images of (k, v), where there are any before the walk's launch
    if (block_mask.has_value()) {
        // rows may be wider than max_seqlen_k needs (select_blocks widens them for cached tokens): the kernels take
        // the width as a row stride and never look at a block beyond the sequence
        const int64_t n64 = ((max_k + kBlock - 1) / kBlock + 63) / 64;
        TORCH_CHECK(block_mask->scalar_type() == at::kLong && block_mask->dim() == 3 && block_mask->size(0) == hk &&
                    block_mask->size(1) == total_q && block_mask->size(2) >= n64,
                    "block_mask must be int64 of shape (num_heads_k, total_q, words) with words >= ceil(ceil(max_seqlen_k / 64) / 64)");
        require_gpu(*block_mask, "block_mask");
        mask = block_mask->contiguous();
    } else if (topk_idx.has_value()) {
        TORCH_CHECK(topk_idx->dim() == 3 && topk_idx->size(0) == hk && topk_idx->size(1) == total_q,
                    "topk_idx must have shape (num_heads_k, total_q, k)");
        const int64_t k_blocks = (max_k + kBlock - 1) / kBlock, n64 = (k_blocks + 63) / 64;
        if (max_k <= INFLLMV2_IN_STEP_KEYS && total_q > 0 && max_q > 0 && !images.has_value()) {
            // The mask words are made by the launch that packs k and v (2049 queries behind 17 962 keys, from the compressed keys on, 325.2 -> 323.4 us, 512 behind each of three
            // prompts 219.6 -> 217.2, 2000 tokens 85.4 -> 83.9).  Not for sequences that are
            // walked in step: the packing clears the counters of the one launch behind it, and is then part of that call.
            require_gpu(*topk_idx, "topk_idx");
            const Tensor idx = topk_idx->contiguous();
            mask = at::empty({hk, total_q, n64}, idx.options().dtype(at::kLong));
            packed = image_workspace(k, batch);
            const S2 ks = rows_heads(k), vs = rows_heads(v);
            check_rc(infllmv2_pack_kv_and_topk(stream_of(q), ptr(k), ptr(v), iptr(cu_k), ptr(*packed), static_cast<size_t>(packed->numel()), as_int(batch),
                                               total_k, as_int(hk), as_int(d), as_int(max_k), ks.v, vs.v, iptr(idx), static_cast<uint64_t*>(mask->data_ptr()),
                                               hk * total_q, as_int(idx.size(2)), as_int(n64)), "pack_kv_and_topk");
        } else {
            mask = topk_to_uint64(*topk_idx, k_blocks, std::nullopt);
        }
    }
    Tensor out = at::empty_like(q);
    const bool sparse = mask.has_value();
    Tensor lse = sparse ? at::empty({hk, total_q * group}, q.options().dtype(at::kFloat))             // flash_api.cpp:665
                        : at::empty({hq, total_q}, q.options().dtype(at::kFloat));
    const int64_t lse_strides[3] = {sparse ? group : 1, sparse ? 1 : total_q, group * total_q};
    TORCH_CHECK(!images.has_value() || (images->device() == k.device() && images->is_contiguous() && images->scalar_type() == at::kByte &&
                                        images->numel() >= static_cast<int64_t>(infllmv2_kv_image_bytes(total_k, as_int(batch), as_int(hk)))),
                "images must hold the block images of k and v");
    Tensor ws = packed.has_value() ? *packed : image_workspace(k, batch);
    const S3 qs = grouped(q, group), os = grouped(out, group);
    const S2 ks = rows_heads(k), vs = rows_heads(v);
    auto fn = is_half(q) ? infllmv2_varlen_fwd_selected_f16 : infllmv2_varlen_fwd_selected;
    // a mask that came with its indices has at most so many blocks to a row (negative: neighbouring rows are alike)
    const int listed = sparse && topk_idx.has_value() && topk_idx->dim() > 0 ? as_int(topk_idx->size(-1)) : 0, most_selected = alike ? -listed : listed;
    check_rc(fn(stream_of(q), ptr(q), ptr(k), ptr(v), ptr(out), static_cast<float*>(ptr(lse)), iptr(cu_q), iptr(cu_k),
                sparse ? static_cast<const uint64_t*>(mask->data_ptr()) : nullptr, ptr(ws), static_cast<size_t>(ws.numel()),
                packed.has_value() ? 1 : 0, as_int(batch), total_q, total_k, as_int(hq), as_int(hk), as_int(d), as_int(max_q), as_int(max_k), qs.v,
                ks.v, vs.v, os.v, lse_strides, sparse ? as_int(mask->size(-1)) : 0, static_cast<float>(scale), causal ? 1 : 0, most_selected), "varlen_fwd");
    return {out, lse, mask};
}

// Returns (dq, dk, dv) with the shapes and dtype of (q, k, v).  most_selected: blocks in a row of the mask at most, 0 where that is not known
std::tuple<Tensor, Tensor, Tensor> varlen_bwd(const Tensor& dout_, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                                              const Tensor& lse, const Tensor& cu_q, const Tensor& cu_k, int64_t max_q, int64_t max_k,
                                              double scale, bool causal, const OptTensor& mask, bool lse_expanded, bool deterministic,
                                              int64_t most_selected) {
    const Tensor dout = dout_.stride(-1) == 1 ? dout_ : dout_.contiguous();
    TORCH_CHECK(dout.scalar_type() == q.scalar_type() && dout.sizes() == q.sizes(), "dout must have the shape and dtype of q");
    DeviceGuard guard(q.device());
    const int64_t batch = cu_q.numel() - 1, total_q = q.size(0), hq = q.size(1), total_k = k.size(0), hk = k.size(1), group = hq / hk;
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const int64_t lse_strides[3] = {lse_expanded ? group : 1, lse_expanded ? 1 : total_q, group * total_q};
    auto size_query = deterministic ? infllmv2_varlen_bwd_deterministic_workspace_bytes : infllmv2_varlen_bwd_workspace_bytes;
    Tensor ws = bytes_on(q, size_query(as_int(batch), total_q, total_k, as_int(hk), as_int(max_k)));
    const S3 qs = grouped(q, group), os = grouped(out, group), dos = grouped(dout, group), dqs = grouped(dq, group);
    const S2 ks = rows_heads(k), vs = rows_heads(v), dks = rows_heads(dk), dvs = rows_heads(dv);
    auto fn = is_half(q) ? infllmv2_varlen_bwd_selected_f16 : infllmv2_varlen_bwd_selected;
    check_rc(fn(stream_of(q), ptr(dout), ptr(q), ptr(k), ptr(v), ptr(out), static_cast<float*>(ptr(lse)), ptr(dq), ptr(dk), ptr(dv), iptr(cu_q),
                iptr(cu_k), static_cast<const uint64_t*>(ptr(mask)), ptr(ws), static_cast<size_t>(ws.numel()), as_int(batch), total_q, total_k,
                as_int(hq), as_int(hk), as_int(q.size(2)), as_int(max_q), as_int(max_k), qs.v, ks.v, vs.v, os.v, dos.v, dqs.v, dks.v, dvs.v,
                lse_strides, mask.has_value() ? as_int(mask->size(-1)) : 0, static_cast<float>(scale), causal ? 1 : 0, deterministic ? 1 : 0,
                as_int(most_selected)), "varlen_bwd");
    return {dq, dk, dv};
}

// ---- decode (mha_fwd_kvcache, flash_api.cpp:1549-1843) -------------------------------------------------------------------
OptTensor int32_vec(const OptTensor& t, int64_t batch, const char* name) {
    if (!t.has_value()) return t;
    TORCH_CHECK(t->scalar_type() == at::kInt, name, " must have dtype int32");
    require_gpu(*t, name);
    TORCH_CHECK(t->dim() == 1 && t->size(0) == batch, name, " must have shape (batch_size)");
    return t->contiguous();
}

// splits of rows of at most `blocks` blocks: no more than leave each of a workgroup's four wavefronts one
int decode_splits(int64_t batch, int64_t hk, int64_t blocks) {
    return as_int(std::min<int64_t>(infllmv2_fwd_kvcache_num_splits(as_int(batch), as_int(hk), 0), std::max<int64_t>(1, (blocks + 3) / 4)));
}

// topk_idx (batch, Hk, 1, k) int32 or block_mask (batch, Hk, 1, words) int64, or neither (dense).  Returns {out, lse}.
std::tuple<Tensor, Tensor> fwd_kvcache(const Tensor& q, const Tensor& kc, const Tensor& vc, const OptTensor& kn, const OptTensor& vn,
                                       const OptTensor& seqlens_, double scale, int64_t num_splits, const OptTensor& topk_idx_,
                                       const OptTensor& block_mask_, const OptTensor& batch_idx_, const OptTensor& leftpad_,
                                       const OptTensor& table, const OptTensor& rot_cos, const OptTensor& rot_sin, bool interleaved) {
    require_gpu(q, "q"); require_gpu(kc, "k_cache"); require_gpu(vc, "v_cache");
    require_16bit(q);
    TORCH_CHECK(kc.scalar_type() == q.scalar_type(), "query and key must have the same dtype");
    TORCH_CHECK(vc.scalar_type() == q.scalar_type(), "query and value must have the same dtype");
    TORCH_CHECK(q.dim() == 4 && kc.dim() == 4 && vc.dim() == 4, "q, k_cache, v_cache must have 4 dimensions");
    const int64_t batch = q.size(0), hq = q.size(2), d = q.size(3), hk = kc.size(2);
    const bool paged = table.has_value();
    int64_t cap = kc.size(1), page = 0, batch_c = kc.size(0);
    if (paged) {
        TORCH_CHECK(!batch_idx_.has_value(), "Paged KVcache does not support cache_batch_idx");
        TORCH_CHECK(!leftpad_.has_value(), "We don't support Paged KV and leftpad_k running at the same time yet");
        require_gpu(*table, "block_table");
        TORCH_CHECK(table->scalar_type() == at::kInt, "block_table must have dtype torch.int32");
        TORCH_CHECK(table->stride(-1) == 1, "block_table must have contiguous last dimension");
        TORCH_CHECK(table->dim() == 2 && table->size(0) == batch, "block_table must have shape (batch_size, max_num_blocks_per_seq)");
        page = kc.size(1);
        TORCH_CHECK(page % kBlock == 0, "Paged KV cache block size must be divisible by 64");
        cap = table->size(1) * page;
        batch_c = batch;
    }
    TORCH_CHECK(batch > 0, "batch size must be positive");
    TORCH_CHECK(d == kHeadDim, "this build only supports head dimension 128");
    group_size(hq, hk);
    TORCH_CHECK(q.size(1) == 1, "this build only supports seqlen_q == 1 in infllmv2_attn_with_kvcache");
    if (paged) {
        TORCH_CHECK(kc.size(3) == d && vc.sizes() == kc.sizes(),
                    "paged k_cache and v_cache must have shape (num_blocks, page_block_size, num_heads_k, head_size)");
    } else {
        TORCH_CHECK(kc.size(3) == d && vc.sizes() == kc.sizes() && (batch_idx_.has_value() || batch_c == batch),
                    "k_cache and v_cache must have shape (batch_size, seqlen_cache, num_heads_k, head_size)");
    }
    int64_t seqlen_new = 0;
    S3 kns{{0, 0, 0}}, vns{{0, 0, 0}};
    if (kn.has_value()) {
        TORCH_CHECK(vn.has_value(), "If key is supplied, value must also be passed in");
        TORCH_CHECK(kn->scalar_type() == q.scalar_type() && vn->scalar_type() == q.scalar_type(), "Key and value must have the same dtype as query");
        TORCH_CHECK(kn->dim() == 4 && kn->size(0) == batch && kn->size(2) == hk && kn->size(3) == d && vn->sizes() == kn->sizes(),
                    "k and v must have shape (batch_size, seqlen_new, num_heads_k, head_size)");
        seqlen_new = kn->size(1);
        kns = batch_rows_heads(*kn); vns = batch_rows_heads(*vn);
    }
    OptTensor seqlens = seqlens_;
    if (seqlens.has_value()) {
        TORCH_CHECK(seqlens->scalar_type() == at::kInt, "seqlens_k must have dtype int32");
        TORCH_CHECK(seqlens->dim() == 1 && seqlens->size(0) == batch, "seqlens_k must have shape (batch_size)");
        seqlens = seqlens->contiguous();
    }
    TORCH_CHECK(!kn.has_value() || seqlens.has_value(), "If key is supplied, seqlens_k must also be passed in");
    const OptTensor batch_idx = int32_vec(batch_idx_, batch, "cache_batch_idx"), leftpad = int32_vec(leftpad_, batch, "leftpad_k");
    int64_t rotary_dim = 0;
    if (rot_cos.has_value()) {
        TORCH_CHECK(kn.has_value(), "If rotary cos/sin are provided, new key / value to be appended to KV cache must also be provided");
        TORCH_CHECK(rot_sin.has_value(), "If rotary cos is provided, rotary sin must also be provided");
        require_gpu(*rot_cos, "rotary_cos"); require_gpu(*rot_sin, "rotary_sin");
        rotary_dim = rot_cos->size(1) * 2;
        TORCH_CHECK(rotary_dim <= d, "rotary_dim must be <= headdim");
        TORCH_CHECK(rotary_dim % 16 == 0, "Only rotary dimensions divisible by 16 are currently supported");
        TORCH_CHECK(rot_cos->size(0) >= cap, "cos/sin seqlen must be at least the seqlen of KV cache");
        TORCH_CHECK(rot_sin->sizes() == rot_cos->sizes() && rot_cos->is_contiguous() && rot_sin->is_contiguous(),
                    "rotary_cos and rotary_sin must be contiguous (seqlen_ro, rotary_dim / 2) tensors");
        TORCH_CHECK(rot_cos->scalar_type() == q.scalar_type() && rot_sin->scalar_type() == q.scalar_type(),
                    "rotary_cos must have the same dtype as query");
    }
    OptTensor mask, idx;
    if (block_mask_.has_value()) {
        require_gpu(*block_mask_, "block_mask");
        TORCH_CHECK(block_mask_->scalar_type() == at::kLong && block_mask_->dim() == 4 && block_mask_->size(0) == batch &&
                    block_mask_->size(2) == 1 && block_mask_->size(1) == hk && block_mask_->device() == q.device(),
                    "block_mask must be an int64 tensor of shape (batch_size, num_heads_k, 1, words) on q's device");
        mask = block_mask_->contiguous();
    } else if (topk_idx_.has_value()) {
        require_gpu(*topk_idx_, "topk_idx");
        TORCH_CHECK(topk_idx_->dim() == 4 && topk_idx_->size(0) == batch && topk_idx_->size(1) == hk && topk_idx_->size(2) == 1,
                    "topk_idx must have shape (batch_size, num_heads_k, 1, k)");
        idx = topk_idx_->contiguous();
    }
    DeviceGuard guard(q.device());
    Tensor out = at::empty_like(q);
    Tensor lse = at::empty({batch, hq, 1}, q.options().dtype(at::kFloat));
    const int splits = num_splits <= 0 && idx.has_value() ? decode_splits(batch, hk, idx->size(3))
                                                          : infllmv2_fwd_kvcache_num_splits(as_int(batch), as_int(hk), as_int(num_splits));
    Tensor ws = bytes_on(q, infllmv2_fwd_kvcache_workspace_bytes(as_int(batch), as_int(hk), splits));
    const int64_t qs[2] = {q.stride(0), q.stride(2)}, os[2] = {out.stride(0), out.stride(2)};
    const S3 kcs = batch_rows_heads(kc), vcs = batch_rows_heads(vc);
    const int64_t table_stride = paged ? table->stride(0) : 0;
    if (idx.has_value() && idx->size(3) > 0) {
        auto fn = is_half(q) ? infllmv2_fwd_kvcache_topk_f16 : infllmv2_fwd_kvcache_topk;
        check_rc(fn(stream_of(q), ptr(q), ptr(kc), ptr(vc), ptr(kn), ptr(vn), iptr(seqlens), ptr(out), static_cast<float*>(ptr(lse)), iptr(idx),
                    as_int(idx->size(3)), ptr(ws), static_cast<size_t>(ws.numel()), as_int(batch), 1, as_int(hq), as_int(hk), as_int(d),
                    as_int(cap), as_int(seqlen_new), qs, kcs.v, vcs.v, kns.v, vns.v, os, splits, static_cast<float>(scale), iptr(batch_idx),
                    iptr(leftpad), iptr(table), table_stride, as_int(page), ptr(rot_cos), ptr(rot_sin), as_int(rotary_dim),
                    interleaved ? 1 : 0), "fwd_kvcache_topk");
        return {out, lse};
    }
    if (idx.has_value()) mask = at::zeros({batch, hk, 1, ((cap + kBlock - 1) / kBlock + 63) / 64}, q.options().dtype(at::kLong));  // an empty list selects nothing
    auto fn = is_half(q) ? infllmv2_fwd_kvcache_f16 : infllmv2_fwd_kvcache;
    check_rc(fn(stream_of(q), ptr(q), ptr(kc), ptr(vc), ptr(kn), ptr(vn), iptr(seqlens), ptr(out), static_cast<float*>(ptr(lse)),
                static_cast<const uint64_t*>(ptr(mask)), ptr(ws), static_cast<size_t>(ws.numel()), as_int(batch), 1, as_int(hq), as_int(hk),
                as_int(d), as_int(cap), as_int(seqlen_new), qs, kcs.v, vcs.v, kns.v, vns.v, os, mask.has_value() ? as_int(mask->size(-1)) : 0,
                splits, static_cast<float>(scale), iptr(batch_idx), iptr(leftpad), iptr(table), table_stride, as_int(page), ptr(rot_cos),
                ptr(rot_sin), as_int(rotary_dim), interleaved ? 1 : 0), "fwd_kvcache");
    return {out, lse};
}

// What a decode step asks of its tensors.
void check_step(const Tensor& q, const Tensor& kn, const Tensor& vn, const Tensor& kc, const Tensor& vc,
                const Tensor& fine, const Tensor& coarse, const OptTensor& lens, int64_t host_len,
                const OptTensor& fine_lens_, const OptTensor& coarse_lens_, int64_t kernel_size,
                int64_t stride, int64_t block_size, bool scores) {
    require_gpu(q, "q"); require_gpu(kc, "k_cache");
    require_16bit(q);
    for (const Tensor* t : {&kn, &vn, &kc, &vc, &fine, &coarse}) {
        TORCH_CHECK(t->scalar_type() == q.scalar_type(), "query and key must have the same dtype");
        TORCH_CHECK(t->device() == q.device(), "the caches and the new token must be on q's device");
        TORCH_CHECK(t->dim() == 4 && t->stride(-1) == 1, "Input tensor must have contiguous last dimension");
    }
    TORCH_CHECK(q.dim() == 4 && q.size(1) == 1 && q.stride(-1) == 1, "q must have shape (batch_size, 1, num_heads, head_size)");
    const int64_t batch = q.size(0), hq = q.size(2), d = q.size(3), hk = kc.size(2);
    TORCH_CHECK(d == kHeadDim, "this build only supports head dimension 128");
    group_size(hq, hk);
    TORCH_CHECK(kc.size(0) == batch && kc.size(3) == d && vc.sizes() == kc.sizes(),
                "k_cache and v_cache must have shape (batch_size, seqlen_cache, num_heads_k, head_size)");
    TORCH_CHECK(kn.size(0) == batch && kn.size(1) == 1 && kn.size(2) == hk && kn.size(3) == d && vn.sizes() == kn.sizes(),
                "k and v must have shape (batch_size, seqlen_new, num_heads_k, head_size)");
    for (const Tensor* t : {&fine, &coarse})
        TORCH_CHECK(t->size(0) == batch && t->size(2) == hk && t->size(3) == d,
                    "compressed-key caches must have shape (batch_size, rows, num_heads_k, head_size)");
    for (const OptTensor* t : {&lens, &fine_lens_, &coarse_lens_})
        TORCH_CHECK(!t->has_value() || ((*t)->scalar_type() == at::kInt && (*t)->dim() == 1 && (*t)->size(0) == batch && (*t)->is_contiguous() &&
                (*t)->device() == q.device()), "lengths must be contiguous int32 tensors of shape (batch_size)");
    // four compressed keys per block, as the pooling of stage1_pooled and stage1_kvcache; without scores nothing looks at the blocks
    TORCH_CHECK(!scores || (block_size == kBlock && stride > 0 && block_size / stride == 4),
                "only 64-token blocks over stride-16 compressed keys are fused");
    // with the length at hand, as compress_keys checks it: a compressed key that has no row is refused, not dropped
    for (const auto& [t, kernel, st] : {std::tuple(&fine, kernel_size, stride), std::tuple(&coarse, 4 * kernel_size, 4 * stride)})
        TORCH_CHECK(lens.has_value() || st <= 0 || windows(host_len + 1, kernel, st) == windows(host_len, kernel, st) ||
                    t->size(1) >= windows(host_len + 1, kernel, st), "out must be a contiguous (rows, num_heads_k, head_size) buffer of k's dtype");
}

// The front of a decode step of a layer for a batch of sequences: append the token, extend the compressed keys, and - with
// scores - Stage 1 and pooling.  lens: tokens held (device), or none: host_len for every sequence.  max_len bounds the
// lengths after the step.  Returns {lengths after the step, block scores (batch, Hk, blocks) or an undefined tensor}.
std::tuple<Tensor, Tensor> decode_front(const Tensor& q, const Tensor& kn, const Tensor& vn, const Tensor& kc, const Tensor& vc,
                                        const Tensor& fine, const Tensor& coarse, const OptTensor& lens, int64_t host_len,
                                        const OptTensor& fine_lens_, const OptTensor& coarse_lens_, int64_t max_len, int64_t kernel_size,
                                        int64_t stride, int64_t block_size, bool scores, int64_t local_blocks, int64_t init_blocks,
                                        double scale) {
    check_step(q, kn, vn, kc, vc, fine, coarse, lens, host_len, fine_lens_, coarse_lens_, kernel_size, stride, block_size, scores);
    const int64_t batch = q.size(0), hq = q.size(2), d = q.size(3), hk = kc.size(2), cap = kc.size(1), group = hq / hk;
    const auto ints = q.options().dtype(at::kInt);
    Tensor new_lens = at::empty({batch}, ints);
    const Tensor fine_lens = fine_lens_.has_value() ? *fine_lens_ : at::empty({batch}, ints);
    const Tensor coarse_lens = coarse_lens_.has_value() ? *coarse_lens_ : at::empty({batch}, ints);
    const int64_t out_len = scores ? (max_len + block_size - 1) / block_size : 0;
    Tensor pooled, ws;
    if (scores) {
        pooled = at::empty({batch, hk, out_len}, q.options());
        const int64_t max_f = std::min(windows(max_len, kernel_size, stride), fine.size(1));
        const int64_t max_c = std::min(windows(max_len, 4 * kernel_size, 4 * stride), coarse.size(1));
        ws = bytes_on(q, infllmv2_stage1_decode_workspace_bytes(as_int(batch), as_int(hk), as_int(max_f), as_int(max_c)));
    }
    const int64_t qs[3] = {q.stride(0), q.stride(2), group * q.stride(2)};
    const int64_t kns[2] = {kn.stride(0), kn.stride(2)}, vns[2] = {vn.stride(0), vn.stride(2)};
    const S3 kcs = batch_rows_heads(kc), vcs = batch_rows_heads(vc), fs = batch_rows_heads(fine), cs = batch_rows_heads(coarse);
    auto fn = is_half(q) ? infllmv2_decode_step_scores_f16 : infllmv2_decode_step_scores;
    check_rc(fn(stream_of(q), ptr(q), ptr(kn), ptr(vn), ptr(kc), ptr(vc), ptr(fine), ptr(coarse), iptr(lens), as_int(host_len),
                static_cast<int32_t*>(ptr(new_lens)), static_cast<int32_t*>(ptr(fine_lens)), static_cast<int32_t*>(ptr(coarse_lens)),
                scores ? ptr(pooled) : nullptr, scores ? ptr(ws) : nullptr, scores ? static_cast<size_t>(ws.numel()) : 0, as_int(batch),
                as_int(hq), as_int(hk), as_int(d), as_int(cap), as_int(fine.size(1)), as_int(coarse.size(1)), as_int(max_len), qs, kns, vns,
                kcs.v, vcs.v, fs.v, cs.v, as_int(kernel_size), as_int(stride), as_int(4 * kernel_size), as_int(4 * stride),
                static_cast<float>(scale), as_int(out_len), as_int(local_blocks), as_int(init_blocks)), "decode_step_scores");
    return {new_lens, pooled};
}

// The front and, with topk > 0, the selection.  Returns {lengths after the step, mask (batch, Hk, 1, words) or none}.
std::tuple<Tensor, OptTensor> decode_step(const Tensor& q, const Tensor& kn, const Tensor& vn, const Tensor& kc, const Tensor& vc,
                                          const Tensor& fine, const Tensor& coarse, const OptTensor& lens, int64_t host_len,
                                          const OptTensor& fine_lens, const OptTensor& coarse_lens, int64_t max_len, int64_t kernel_size,
                                          int64_t stride, int64_t block_size, int64_t topk, int64_t local_blocks, int64_t init_blocks,
                                          double scale) {
    require_gpu(q, "q");
    DeviceGuard guard(q.device());
    auto [new_lens, pooled] = decode_front(q, kn, vn, kc, vc, fine, coarse, lens, host_len, fine_lens, coarse_lens, max_len, kernel_size,
                                           stride, block_size, topk > 0, local_blocks, init_blocks, scale);
    if (topk <= 0) return {new_lens, std::nullopt};
    return {new_lens, topk_mask(pooled, topk, std::nullopt).unsqueeze(2)};
}

// A whole decode step on selected blocks: the front, the selection and the attention.  The selection is made by the
// attention's own launch where that serves it (a workgroup per CU at most, rows of 2048 block scores at most: see
// infllmv2_fwd_kvcache_scores), by a top-k launch otherwise.  Returns {out, lengths after the step}; a step of one sequence whose length the
// host gives has no lengths to return.
std::tuple<Tensor, Tensor> decode_sparse(const Tensor& q, const Tensor& kn, const Tensor& vn, const Tensor& kc, const Tensor& vc,
                                         const Tensor& fine, const Tensor& coarse, const OptTensor& lens, int64_t host_len,
                                         const OptTensor& fine_lens, const OptTensor& coarse_lens, int64_t max_len, int64_t kernel_size,
                                         int64_t stride, int64_t block_size, int64_t topk, int64_t local_blocks, int64_t init_blocks,
                                         double scale) {
    TORCH_CHECK(topk > 0, "decode_sparse: topk must be positive");
    require_gpu(q, "q");
    TORCH_CHECK(q.dim() == 4 && kc.dim() == 4, "q, k_cache, v_cache must have 4 dimensions");
    check_step(q, kn, vn, kc, vc, fine, coarse, lens, host_len, fine_lens, coarse_lens, kernel_size, stride, block_size, true);
    DeviceGuard guard(q.device());
    const int64_t batch = q.size(0), hq = q.size(2), hk = kc.size(2);
    const int splits = decode_splits(batch, hk, topk);
    const int64_t blocks = (max_len + block_size - 1) / block_size;
    const bool all = blocks <= topk;                           // nothing to select: no scores
    if (batch * hk * splits > 256 || max_len > INFLLMV2_DECODE_MAX_SCORES * kBlock) {
        if (all && topk <= INFLLMV2_DECODE_MAX_SCORES) {
            const Tensor new_lens = std::get<0>(decode_front(q, kn, vn, kc, vc, fine, coarse, lens, host_len, fine_lens, coarse_lens, max_len, kernel_size,
                                                             stride, block_size, false, local_blocks, init_blocks, scale));
            return {std::get<0>(fwd_kvcache(q, kc, vc, std::nullopt, std::nullopt, new_lens, scale, 0, std::nullopt, std::nullopt, std::nullopt, std::nullopt,
                                            std::nullopt, std::nullopt, std::nullopt, false)), new_lens};
        }
        auto [new_lens, mask] = decode_step(q, kn, vn, kc, vc, fine, coarse, lens, host_len, fine_lens, coarse_lens, max_len, kernel_size, stride,
                                            block_size, topk, local_blocks, init_blocks, scale);
        return {std::get<0>(fwd_kvcache(q, kc, vc, std::nullopt, std::nullopt, new_lens, scale, 0, std::nullopt, mask, std::nullopt, std::nullopt,
                                        std::nullopt, std::nullopt, std::nullopt, false)), new_lens};
    }
    // What lives inside the step shares one allocation, and lengths that the host has get no tensor of their own: a step that the device finishes in 19 to 20 us was
    // bound by the host that issues it (one sequence, seven allocations 22.6 us to issue, two 19.6; six sequences 19.2 and 17.3).
    Tensor new_lens, out = at::empty_like(q);
    if (lens.has_value()) new_lens = at::empty({batch}, q.options().dtype(at::kInt));
    const int64_t max_f = std::min(windows(max_len, kernel_size, stride), fine.size(1)), max_c = std::min(windows(max_len, 4 * kernel_size, 4 * stride), coarse.size(1));
    size_t at_byte = 0;
    auto take = [&](size_t bytes) { const size_t start = at_byte; at_byte += (bytes + 255) / 256 * 256; return start; };
    const size_t record_bytes = infllmv2_stage1_decode_workspace_bytes(as_int(batch), as_int(hk), as_int(max_f), as_int(max_c));
    const size_t partial_bytes = infllmv2_fwd_kvcache_workspace_bytes(as_int(batch), as_int(hk), splits);
    const size_t scores = take(2 * static_cast<size_t>(batch * hk * blocks)), records = take(std::max<size_t>(record_bytes, 16)), partials = take(partial_bytes);
    const size_t lse = take(sizeof(float) * static_cast<size_t>(batch * hq)), own_lens = take(3 * sizeof(int32_t) * static_cast<size_t>(batch));
    Tensor ws = bytes_on(q, at_byte);
    char* base = static_cast<char*>(ptr(ws));
    int32_t* own = reinterpret_cast<int32_t*>(base + own_lens);
    int32_t* new_ptr = lens.has_value() ? static_cast<int32_t*>(ptr(new_lens)) : own;
    int32_t* fine_ptr = fine_lens.has_value() ? static_cast<int32_t*>(ptr(*fine_lens)) : own + batch;
    int32_t* coarse_ptr = coarse_lens.has_value() ? static_cast<int32_t*>(ptr(*coarse_lens)) : own + 2 * batch;
    const int64_t group = hq / hk, qs[3] = {q.stride(0), q.stride(2), group * q.stride(2)}, os[2] = {out.stride(0), out.stride(2)};
    const int64_t kns[2] = {kn.stride(0), kn.stride(2)}, vns[2] = {vn.stride(0), vn.stride(2)};
    const S3 kcs = batch_rows_heads(kc), vcs = batch_rows_heads(vc), fs = batch_rows_heads(fine), cs = batch_rows_heads(coarse);
    void* stream = stream_of(q);
    if (all) {
        auto step = is_half(q) ? infllmv2_decode_step_all_f16 : infllmv2_decode_step_all;
        check_rc(step(stream, ptr(q), ptr(kn), ptr(vn), ptr(kc), ptr(vc), ptr(fine), ptr(coarse), iptr(lens), as_int(host_len), new_ptr, fine_ptr, coarse_ptr, ptr(out),
                      reinterpret_cast<float*>(base + lse), base + partials, partial_bytes, as_int(batch), as_int(hq), as_int(hk), as_int(kHeadDim),
                      as_int(kc.size(1)), as_int(fine.size(1)), as_int(coarse.size(1)), as_int(max_len), qs, kns, vns, kcs.v, vcs.v, fs.v, cs.v, os,
                      as_int(kernel_size), as_int(stride), as_int(4 * kernel_size), as_int(4 * stride), splits, static_cast<float>(scale)), "decode_step_all");
        return {out, new_lens};
    }
    auto front = is_half(q) ? infllmv2_decode_step_scores_f16 : infllmv2_decode_step_scores;
    check_rc(front(stream, ptr(q), ptr(kn), ptr(vn), ptr(kc), ptr(vc), ptr(fine), ptr(coarse), iptr(lens), as_int(host_len), new_ptr, fine_ptr, coarse_ptr,
                   base + scores, base + records, record_bytes, as_int(batch), as_int(hq), as_int(hk), as_int(kHeadDim), as_int(kc.size(1)),
                   as_int(fine.size(1)), as_int(coarse.size(1)), as_int(max_len), qs, kns, vns, kcs.v, vcs.v, fs.v, cs.v, as_int(kernel_size),
                   as_int(stride), as_int(4 * kernel_size), as_int(4 * stride), static_cast<float>(scale), as_int(blocks), as_int(local_blocks),
                   as_int(init_blocks)), "decode_step_scores");
    auto attend = is_half(q) ? infllmv2_fwd_kvcache_scores_f16 : infllmv2_fwd_kvcache_scores;
    check_rc(attend(stream, ptr(q), ptr(kc), ptr(vc), new_ptr, ptr(out), reinterpret_cast<float*>(base + lse), base + scores, as_int(blocks), as_int(topk),
                    base + partials, partial_bytes, as_int(batch), as_int(hq), as_int(hk), as_int(kHeadDim), as_int(kc.size(1)), qs, kcs.v, vcs.v, os,
                    splits, static_cast<float>(scale)), "fwd_kvcache_scores");
    return {out, new_lens};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "native host side of infllmv2_cuda_impl_amd's operators";
    m.def("compress_keys", &compress_keys);
    m.def("compress_keys_pair", &compress_keys_pair);
    m.def("stage1_scores", &stage1_scores);
    m.def("stage1_pooled", &stage1_pooled);
    m.def("stage1_kvcache", &stage1_kvcache);
    m.def("max_pooling_1d", &max_pooling_1d);
    m.def("max_pooling_1d_varlen", &max_pooling_1d_varlen);
    m.def("topk_blocks", &topk_blocks);
    m.def("window_blocks", &window_blocks);
    m.def("topk_to_uint64", &topk_to_uint64);
    m.def("select_blocks", &select_blocks);
    m.def("select_mask", &select_mask);
    m.def("varlen_fwd", &varlen_fwd);
    m.def("varlen_bwd", &varlen_bwd);
    m.def("fwd_kvcache", &fwd_kvcache);
    m.def("decode_step", &decode_step);
    m.def("decode_sparse", &decode_sparse);
}
