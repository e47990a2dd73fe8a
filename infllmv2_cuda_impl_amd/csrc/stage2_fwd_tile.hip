// Stage-2 forward without a mask (gfx950): dense attention over packed sequences as a flash tile of 256 query rows.
//
// Where every token attends its whole prefix nothing is left to fetch per token, and the hybrid walk (stage2_fwd_hybrid.hip) only
// keeps its costs: 16 query rows per K / V fragment read from LDS, softmax and MFMAs of a wavefront one after the other.  Here a workgroup of 8
// wavefronts owns 256 rows (16 tokens of 16 heads, 32 of 8) and a wavefront 32 of them, the N side of v_mfma_f32_32x32x16: a fragment feeds
// twice the rows in half the instructions.  K and V come from the same block images through the same 4-tile LDS ring.
//
// What bounds it: per block a SIMD's two wavefronts need 64 MFMAs of 32 clocks and about 250 vector instructions (64 of them
// exponentials), which share the issue port: neither may wait for the other.  So the walk is one block ahead with its scores, and the order
// inside a block is written out: one MFMA of the next block's S, two exponentials of this block's, the LDS reads of the operands that come
// next.  Left to the compiler, which forms clumps of MFMAs and of exponentials, the same work takes 2310 us for 16384 tokens of 2 KV heads
// instead of 1980.  Counters at 2500 + 6001 + 4096 tokens: matrix pipe busy 48 % of the kernel, vector pipe 37 %, LDS reads free of conflicts.
// Operator with 2 KV heads, us, hybrid walk -> this one: 2000 tokens 62 -> 61, 3800 156 -> 125, 16384 2430 -> 1980 (1.11 PFLOP/s), 50000
// 20370 -> 17100 (1.2 PFLOP/s), 2500 + 6001 + 4096 566 -> 472, 777 + 5003 + 1291 + 9173 1160 -> 950.
//
// Operands.  S^T = K Q^T: lane (n = lane % 32, h = lane / 32) holds key n of a 32-key chunk, d = 16 ks + 8 h + j: one 16-byte unit of
// the K image.  The accumulators hold keys 8 i + 4 h + e (register 4 i + e) of row n; a V image unit holds keys 4 g + e and
// 16 + 4 g + e of its chunk, so registers i = jj and i = jj + 2 are, converted, the B operand that goes with the V units of
// g = 2 jj + h: P moves nowhere.
#include "common.h"
#include "kv_image.h"
#include "block_walker.h"
#include "lds_dma.h"
#include "stage2_fwd.h"
#include "infllmv2_hip.h"
#include <math.h>

namespace IV2_NS {

constexpr int kTileRows = 256;                                 // query rows of a workgroup, 32 per wavefront
constexpr int kRingTiles = 4;
constexpr int kTileBytes = 32768;                              // K image | V image of one block
constexpr float kLazyLimit = 64.f;                             // as in the hybrid walk: a lane's sum of P that the reference exponent has to keep to

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

template <bool kCausal>
__global__ __launch_bounds__(512)
void stage2_fwd_tile_kernel(const FwdParams p, const TileExtra x) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    uint4* ring = reinterpret_cast<uint4*>(smem_raw);                               // [kRingTiles][2048]: K units 0..1023, V units 1024..2047

    // ---- which tile: sequence by sequence, longest prefixes first, the KV heads of a tile next to each other (on the XCDs of a chip
    //      that shares work round robin: each keeps to one head where there are two, four or eight).  Tiles behind the end of a sequence
    //      are then a run of workgroups that return at once.  With the sequences innermost instead (all longest prefixes first) the live
    //      workgroups came at a fixed distance, which the dispatcher maps to the same few shader engines: 1890 us instead of
    //      950 for 777, 5003, 1291 and 9173 tokens. ----
    int G = blockIdx.x;
    if (G >= x.sequences * x.tiles_per_seq) return;                                 // uniform per workgroup
    const int h_kv = G % x.heads_k;
    G /= x.heads_k;
    const int level = x.tiles_per_seq - 1 - G % x.tiles_per_seq;
    const int b = x.batch - 1 - G / x.tiles_per_seq;
    const int q0 = p.cu_seqlens_q[b];
    const int Sq = p.cu_seqlens_q[b + 1] - q0;
    const int i_first = level * (kTileRows >> x.row_shift);
    if (i_first >= Sq) return;                                                      // uniform per workgroup
    const int Sk = p.cu_seqlens_k[b + 1] - p.cu_seqlens_k[b];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const int n = lane & 31, h = lane >> 5;
    const int per_wave = 32 >> x.row_shift;                                         // tokens of a wavefront
    const int i_wave = i_first + wave * per_wave;
    auto last_of = [&](int t) {                                                     // last key token t attends
        const int lk = kCausal ? t + Sk - Sq : Sk - 1;
        return lk > Sk - 1 ? Sk - 1 : lk;
    };
    const int wave_first_key = i_wave + per_wave <= Sq ? last_of(i_wave) : -1;      // of the wavefront's first token; -1: it has rows without a token

    elem8 qf[8];
    {
        const int i = i_wave + (n >> x.row_shift), head = n & ((1 << x.row_shift) - 1);
        const int64_t tok = static_cast<int64_t>(q0) + (i < Sq ? i : Sq - 1);
        const elem_bits* qp = p.q + tok * p.q_tok_stride + h_kv * p.q_kvh_stride + (head < p.group ? head : p.group - 1) * p.q_grp_stride + 8 * h;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const elem8*>(qp + 16 * ks);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                // before the first LDS-DMA (see the hybrid walk)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+v"(qf[ks]));

    const int64_t slot0 = static_cast<int64_t>(h_kv) * p.n_slots + image_slot0(p.cu_seqlens_k, b);
    const elem_bits* src = (wave < 4 ? p.kimg : p.vimg) + slot0 * kImageElems + (wave & 3) * 2048;   // this wavefront's quarter of K or V
    const uint32_t ring_base = __builtin_amdgcn_readfirstlane(lds_address_of(ring) + wave * 4096);
    auto issue = [&](int j, int tile) { dma_copy_4k(src + static_cast<int64_t>(j) * kImageElems, 16 * lane, ring_base + tile * kTileBytes); };
    int blocks = 0;                                                                 // of the tile's last token
    {
        const int i_end = i_first + (kTileRows >> x.row_shift) - 1;
        const int lk = last_of(i_end < Sq ? i_end : Sq - 1);
        blocks = lk < 0 ? 0 : (lk >> 6) + 1;
        if (blocks > x.max_blocks) blocks = x.max_blocks;                           // a sequence longer than the announced max_seqlen_k
    }

    // m: reference exponent as in softmax_step, but finite from the start (a row whose keys are all hidden so far has P = 0 by itself)
    float m = -3.4028234e38f, l = 0.f;
    floatx16 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

    // 16-byte units of this lane inside a tile: K unit (2 cc + n/16, ks/2, n%16 + 16 (2 (ks%2) + h)), V unit (2 t + n/16, cc, n%16 + 16 (2 jj + h))
    const int k_unit = (n >> 4) * 256 + (n & 15) + 16 * h;
    const int v_unit = 1024 + (n >> 4) * 128 + (n & 15) + 16 * h;
    elem8 kf[16];                                              // K of the next block, kf[2 ks + cc]
    auto load_k = [&](int tile, int half) {                    // half the depth at a time: 4 of 8 ks
        const uint4* kb = ring + tile * 2048 + k_unit;
#pragma unroll
        for (int ks = 4 * half; ks < 4 * half + 4; ++ks)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                const uint4 raw = kb[cc * 512 + (ks >> 1) * 64 + (ks & 1) * 32];
                __builtin_memcpy(&kf[2 * ks + cc], &raw, 16);
            }
    };
    auto scores = [&](floatx16 (&s)[2]) {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[cc][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) s[cc] = IV2_MFMA32(kf[2 * ks + cc], qf[ks], s[cc]);
    };
    auto hide = [&](floatx16 (&s)[2], int j) {                 // keys behind the row's last one
        const int i = i_wave + (n >> x.row_shift);
        const int lim = (i < Sq ? last_of(i) : -1) - j * kBlockN;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * cc + 8 * (r >> 2) + 4 * h + (r & 3) > lim) s[cc][r] = -INFINITY;
    };
    elem8 pf[4];
    auto exponentials = [&](floatx16 (&s)[2]) -> float {       // s becomes P; returns the lane's sum
        float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[cc][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[cc][r], p.scale_log2, -m));
                part[r & 3] += s[cc][r];
            }
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pf[2 * cc + jj][e] = static_cast<elem_t>(s[cc][4 * jj + e]);
                    pf[2 * cc + jj][4 + e] = static_cast<elem_t>(s[cc][4 * (jj + 2) + e]);
                }
        return (part[0] + part[1]) + (part[2] + part[3]);
    };

    // One barrier per block.  Behind the one of block j the tiles of j, j + 1 and j + 2 are in LDS and the fourth is free: V of j and K of
    // j + 1 and j + 2 are read from LDS, j + 3 is requested.  S of j + 1 is formed between the exponentials of j.
    for (int j = 0; j < 3 && j < blocks; ++j) issue(j, j);
    floatx16 sa[2], sb[2];
    if (blocks > 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        load_k(0, 0);
        load_k(0, 1);
        scores(sa);
        load_k(1, 0);                                          // whatever lies there where there is no second block: its scores are not used
    }
    auto step = [&](int j, floatx16 (&sc)[2], floatx16 (&sn)[2]) {
        const int slot = j & 3;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wavefront's part of tile j + 2
        __syncthreads();
        if (j + 3 < blocks) issue(j + 3, (j + 3) & 3);
        const bool edge = j * kBlockN + kBlockN - 1 > wave_first_key;              // the last block or two
        if (edge) hide(sc, j);
        const uint4* vb = ring + slot * 2048 + v_unit;
        elem8 vf[16];
        // Region A: S of the next block, MFMA by MFMA, and beside each MFMA two of this block's exponentials and its share of LDS reads
        // (the rest of K for the coming MFMAs, then V).  The order is fixed by hand: the compiler's own clumps both sides.
        auto read_k = [&](int f) {
            const uint4 raw = ring[((slot + 1) & 3) * 2048 + k_unit + (f & 1) * 512 + (f >> 2) * 64 + ((f >> 1) & 1) * 32];
            __builtin_memcpy(&kf[f], &raw, 16);
        };
        auto read_v = [&](int f) {                             // f = 8 cc + 4 jj + t
            const uint4 raw = vb[(f & 3) * 256 + (f >> 3) * 64 + ((f >> 2) & 1) * 32];
            __builtin_memcpy(&vf[f], &raw, 16);
        };
        float part[2] = {0.f, 0.f};
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r) sn[cc][r] = 0.f;
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            sn[f & 1] = IV2_MFMA32(kf[f], qf[f >> 1], sn[f & 1]);
            if (f < 4) {
                read_k(8 + 2 * f);
                read_k(9 + 2 * f);
            } else if (f < 12) {
                read_v(f - 4);
            }
            const int cc = f >> 3, r = 2 * (f & 7);
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[cc][r], p.scale_log2, -m));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[cc][r + 1], p.scale_log2, -m));
            part[0] += p0;
            part[1] += p1;
            asm volatile("" : "+v"(part[0]), "+v"(part[1]));   // here, not all at the end
            pf[2 * cc + ((r >> 2) & 1)][(r >> 3) * 4 + (r & 3)] = static_cast<elem_t>(p0);
            pf[2 * cc + ((r >> 2) & 1)][(r >> 3) * 4 + (r & 3) + 1] = static_cast<elem_t>(p1);
            __builtin_amdgcn_sched_barrier(0);
        }
        float rs = part[0] + part[1];
        asm volatile("" : "+v"(pf[0]), "+v"(pf[1]), "+v"(pf[2]), "+v"(pf[3]), "+v"(rs));
        if (__ballot(!(rs <= kLazyLimit)) != 0ull) {           // a row without a reference yet, one that grew, or NaN: the block's scores once more
            load_k(slot, 0);
            load_k(slot, 1);
            scores(sc);
            if (edge) hide(sc, j);
            float mx = -INFINITY;
#pragma unroll
            for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[cc][r]);
            const float m_new = fmaxf(m, half_max(mx) * p.scale_log2);
            const float alpha = __builtin_amdgcn_exp2f(m - m_new);
            l *= alpha;
            m = m_new;
#pragma unroll
            for (int t = 0; t < 4; ++t) o[t] *= alpha;
            rs = exponentials(sc);
        }
        l += rs;
        // Region B: P V, the rest of V ahead of the MFMAs that need it, the first half of the next K behind them.
#pragma unroll
        for (int f = 0; f < 16; ++f) {                         // f = 8 cc + 4 jj + t
            o[f & 3] = IV2_MFMA32(vf[f], pf[f >> 2], o[f & 3]);
            if (f < 8) {
                read_v(8 + f);
            } else {
                const uint4 raw = ring[((slot + 2) & 3) * 2048 + k_unit + (f & 1) * 512 + ((f - 8) >> 2) * 64 + ((f >> 1) & 1) * 32];
                __builtin_memcpy(&kf[f - 8], &raw, 16);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int j = 0; j < blocks; j += 2) {                      // uniform over the workgroup
        step(j, sa, sb);
        if (j + 1 < blocks) step(j + 1, sb, sa);
    }

    const float l_tot = half_sum(l);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    int row = n;
    asm volatile("" : "+v"(row));                              // computed again: the walk has no registers to spare
    const int i = i_wave + (row >> x.row_shift), head = row & ((1 << x.row_shift) - 1);
    if (i >= Sq || head >= p.group) return;
    const int64_t tok = static_cast<int64_t>(q0) + i;
    elem_bits* op = p.out + tok * p.o_tok_stride + h_kv * p.o_kvh_stride + head * p.o_grp_stride + 4 * h;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            uint2 wv;
            wv.x = pack_elem2(o[t][4 * i4] * inv, o[t][4 * i4 + 1] * inv);
            wv.y = pack_elem2(o[t][4 * i4 + 2] * inv, o[t][4 * i4 + 3] * inv);
            *reinterpret_cast<uint2*>(op + 32 * t + 8 * i4) = wv;
        }
    if (h == 0) {
        const float lse = l_tot > 0.f ? m * 0.69314718055994530942f + logf(l_tot) : INFINITY;
        p.lse[h_kv * p.lse_kvh_stride + tok * p.lse_tok_stride + head * p.lse_grp_stride] = lse;
    }
}

// Time of a dense launch whose workgroups take `tokens` tokens each, one workgroup per CU at a time: in microseconds, but for what all
// launches share.  A workgroup costs `fixed` and `block` per key block; a launch takes as long as its longest walk, or as the
// work of all of them on 256 CUs with a last round that is `partial` of one more; workgroups behind the end of a sequence, which
// return at once, 1.7 ns each.  The host knows the longest sequence and the totals: the others are taken to be of equal length.
static double dense_walk_time(int tokens, double fixed, double block, double partial, int batch, int num_heads_k, int64_t total_q,
                              int64_t total_k, int max_seqlen_q, int max_seqlen_k, bool causal) {
    auto blocks = [&](double q, double k) {                    // of a workgroup of a sequence, on average
        const double first = causal ? (k > q ? k - q : 0.) : k;
        return q > tokens ? (first + k) / (2 * kBlockN) + 0.5 : ceil(k / kBlockN);
    };
    const int others = batch - 1;
    const double q = others > 0 && total_q > max_seqlen_q ? static_cast<double>(total_q - max_seqlen_q) / others : 0.;
    const double k = others > 0 && total_k > max_seqlen_k ? static_cast<double>(total_k - max_seqlen_k) / others : 0.;
    const double of_longest = ceil(static_cast<double>(max_seqlen_q) / tokens), of_others = others * ceil(q / tokens);
    const double rounds = num_heads_k * (of_longest + of_others) / 256.;
    const double each = fixed + block * (of_longest * blocks(max_seqlen_q, max_seqlen_k) + of_others * blocks(q, k)) / (of_longest + of_others);
    const double chain = fixed + block * ceil(static_cast<double>(max_seqlen_k) / kBlockN);
    const double all = each * (rounds + (rounds > 1. ? partial : 0.));
    return (chain > all ? chain : all) + 0.0017 * num_heads_k * batch * of_longest;
}

// Whether a forward without a mask goes by tiles: a tile walks a block in 1.5 us, the hybrid walk's group of 8 tokens in 1.0, so tiles
// win where there is more work than the longest chain and lose where that chain, or the rounding up to whole tiles, decides.
// The constants are a fit to 359 launches of 1 to 300 sequences of 4 to 20000 tokens over up to 16000 keys, 1 to 8 KV heads, groups of 8 and
// 16 (within 15 to 17 %); the choice costs 0.3 % of the better walk's time on average and over 10 % in one of them.  A number of
// tiles alone, 240, cost 3.3 % and up to 45 (us, hybrid walk | tiles; * the one taken here):
//   1 KV head:  3800 tokens 88 * | 101, 5000 143 | 136 *, 16000 1080 | 894 *
//   2 KV heads: 1000 tokens 27 * | 37, 2000 62 | 61 *, 16000 2132 | 1769 *; with groups of 8 3800 tokens 152 | 105 *
//   2 KV heads: 1000 and 3 x 16 tokens 30 * | 39; 4000 and 100 x 16 316 | 233 *; 80 x 24 21 * | 31; 2 x 300 over 6300 keys (4 heads) 209 | 163 *
bool dense_tiles_pay(int batch, int num_heads_k, int group, int64_t total_q, int64_t total_k, int max_seqlen_q, int max_seqlen_k, bool causal) {
    if (max_seqlen_q <= 0) return false;
    const double tiles = dense_walk_time(kTileRows >> tile_row_shift(group), 10., 1.5, 0.75, batch, num_heads_k, total_q, total_k, max_seqlen_q, max_seqlen_k, causal);
    const double groups = dense_walk_time(8, 6., 1., 0.7, batch, num_heads_k, total_q, total_k, max_seqlen_q, max_seqlen_k, causal);
    return tiles < groups + 1.;
}

int launch_stage2_fwd_tile(hipStream_t st, const FwdParams& p, int batch, int num_heads_k, int max_seqlen_q, int max_seqlen_k, bool causal) {
    TileExtra x{};
    x.batch = batch;
    x.heads_k = num_heads_k;
    x.sequences = num_heads_k * batch;
    x.row_shift = tile_row_shift(p.group);
    x.tiles_per_seq = tiles_per_sequence(p.group, max_seqlen_q);
    x.max_blocks = (max_seqlen_k + kBlockN - 1) / kBlockN;
    const int64_t total = static_cast<int64_t>(x.sequences) * x.tiles_per_seq;
    IV2_CHECK(total <= 0x3fffffff, "varlen_fwd: too many token groups");
    const int64_t grid = (total + 7) / 8 * 8;
    const size_t lds = kRingTiles * kTileBytes;
    const auto kernel = causal ? &stage2_fwd_tile_kernel<true> : &stage2_fwd_tile_kernel<false>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    IV2_CHECK(e == hipSuccess, "varlen_fwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(512), lds, st, p, x);
    IV2_LAUNCH_CHECK();
    return 0;
}

}  // namespace IV2_NS

#ifndef IV2_F16        // element-type independent: defined once
extern "C" int infllmv2_varlen_fwd_dense_tiles(int batch, int64_t total_q, int64_t total_k, int num_heads, int num_heads_k, int max_seqlen_q,
                                               int max_seqlen_k, int is_causal) {
    return num_heads_k > 0 && batch > 0 && IV2_NS::dense_tiles_pay(batch, num_heads_k, num_heads / num_heads_k, total_q, total_k, max_seqlen_q,
                                                                   max_seqlen_k, is_causal != 0) ? 1 : 0;
}
#endif
