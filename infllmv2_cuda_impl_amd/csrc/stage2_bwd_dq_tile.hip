// Stage-2 backward, dQ by tiles of 256 query rows (gfx950): without a mask, or for a window, whose neighbouring rows select nearly the same.
//
// The mathematics of stage2_bwd_dq.hip on the walk of stage2_fwd_tile.hip: a workgroup of 4 wavefronts owns 256 rows and walks the blocks that any of
// its tokens selected; a row has P = 0 in a block it did not select.  The hybrid walk reads 48 KiB of LDS per (token, common block) for 16 query rows,
// and 32 KiB through the L1 path per block of a token's own; here the three operands of a block (K, V and K transposed) are read from LDS once per 64
// rows.
//
// 16384 dense tokens of 2 KV heads: 3810 us by the hybrid walk, 2760 here (1.2 PFLOP/s, where the forward's tiles stand too: power).
//
// What bounds it: 96 MFMAs of 32 clocks per wavefront and block, and what stands beside them: one wavefront per SIMD issues a vector instruction
// about every five clocks.  So the work of a step is spread by hand: with j the block whose gradient is formed and j + 1 the next,
//   A  S of j + 1      beside it the second half of dS of j, then the first exponentials of j + 1
//   B  dQ of j         beside it the exponentials of j + 1
//   C  dP of j + 1     beside it the last exponentials, then the first half of dS of j + 1
// 512 registers: dQ (128), Q and dO (64 each) in accumulation registers, S and dP (64 each), dS (32).
//
// Operands.  As in the forward, S^T and dP^T leave keys 8 i + 4 h + e (register 4 i + e) of row n in lane (n, h), and registers i = jj and i = jj + 2
// are, converted, the B operand of dQ^T = K^T dS^T; its A operand, four keys of one column, is a transposing read of the K image.  In LDS the 16-byte
// units (g', r') of a kilobyte of the image lie at 16 g' + (r' + 4 g') % 16: transposing reads of four rows then use every bank once.
#include "common.h"
#include "kv_image.h"
#include "block_walker.h"
#include "lds_dma.h"
#include "tile_walk.h"
#include "stage2_bwd.h"
#include "infllmv2_hip.h"
#include <math.h>

namespace IV2_NS {

constexpr int kDqSlots = 4;                                    // of the ring

typedef short short4t __attribute__((ext_vector_type(4)));
typedef int int4t __attribute__((ext_vector_type(4)));

#ifdef IV2_F16
#define IV2_MFMA32_ASM "v_mfma_f32_32x32x16_f16"
#else
#define IV2_MFMA32_ASM "v_mfma_f32_32x32x16_bf16"
#endif

// acc[hf] += a * b[hf] for both halves, accumulators in AGPRs.  The compiler does not see that these are MFMAs: the block opens with the wait states
// between a vector instruction's result and an MFMA that reads it, and inside the walk only MFMAs touch the accumulators.
__device__ __forceinline__ void mfma_both(floatx16& acc0, floatx16& acc1, const elem8& a, const int4t& b0, const int4t& b1) {
    int4t ai;
    __builtin_memcpy(&ai, &a, 16);
    asm volatile("s_nop 1\n\t" IV2_MFMA32_ASM " %0, %2, %3, %0\n\t" IV2_MFMA32_ASM " %1, %2, %4, %1"
                 : "+a"(acc0), "+a"(acc1) : "v"(ai), "v"(b0), "v"(b1));
}

template <bool kCausal>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(1, 1)))
void bwd_dq_tile_kernel(const BwdParams p, const TileExtra x) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];        // [kDqSlots]: K image, V in K-image order

    // ---- which tile: as in the forward ----
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
    const int per_half = 32 >> x.row_shift;                                         // tokens of half a wavefront
    const int i_wave = i_first + wave * 2 * per_half;
    auto last_of = [&](int t) {                                                     // last key token t attends
        const int lk = kCausal ? t + Sk - Sq : Sk - 1;
        return lk > Sk - 1 ? Sk - 1 : lk;
    };
    const int wave_first_key = last_of(i_wave);

    // ---- the rows' operands, LSE and D = rowsum(dO * O) (compute_dot_do_o, flash_bwd_preprocess_kernel.h:56-137) ----
    elem8 qf[2][8], dof[2][8];
    float lse2[2], dsum[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        const int i = i_wave + hf * per_half + (n >> x.row_shift), head = n & ((1 << x.row_shift) - 1), headc = head < p.group ? head : p.group - 1;
        const int64_t tok = static_cast<int64_t>(q0) + (i < Sq ? i : Sq - 1);
        const elem_bits* qp = p.q + tok * p.q_tok + h_kv * p.q_kvh + headc * p.q_grp + 8 * h;
        const elem_bits* dp = p.dout + tok * p.do_tok + h_kv * p.do_kvh + headc * p.do_grp + 8 * h;
        const elem_bits* op = p.out + tok * p.o_tok + h_kv * p.o_kvh + headc * p.o_grp + 8 * h;
        elem8 of[8];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            qf[hf][ks] = *reinterpret_cast<const elem8*>(qp + 16 * ks);
            dof[hf][ks] = *reinterpret_cast<const elem8*>(dp + 16 * ks);
            of[ks] = *reinterpret_cast<const elem8*>(op + 16 * ks);
        }
        lse2[hf] = p.lse[h_kv * p.lse_kvh + tok * p.lse_tok + headc * p.lse_grp] * kLog2e;
        float sum = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += static_cast<float>(dof[hf][ks][e]) * static_cast<float>(of[ks][e]);
        dsum[hf] = half_sum(sum);
        if (head >= p.group) {                                 // spare rows: P = exp2(x - inf) and dS = P (dP - D) vanish, here and in the dK/dV kernel
            lse2[hf] = INFINITY;
            dsum[hf] = 0.f;
        }
    }

    typedef TileWalk<kCausal> Walk;
    Walk walk;
    {
        const int left = Sq - i_first, all = kTileRows >> x.row_shift;
        walk.tokens = left < all ? left : all;
        const int lk = last_of(i_first + walk.tokens - 1);                          // of the tile's last token
        walk.blocks = lk < 0 ? 0 : (lk >> 6) + 1;
        if (walk.blocks > x.max_blocks) walk.blocks = x.max_blocks;                 // a sequence longer than the announced max_seqlen_k
        walk.rows = p.fwd_mask ? p.fwd_mask + (static_cast<int64_t>(h_kv) * p.total_q + q0 + i_first) * p.n64_fwd : nullptr;
        walk.n64 = p.n64_fwd;
        walk.mine = wave * 2 * per_half;
        walk.per_wave = 2 * per_half;
        walk.last_key = last_of(i_first);
        walk.init();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                // before the first LDS-DMA (see the hybrid walk)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+a"(qf[0][ks]), "+a"(qf[1][ks]), "+a"(dof[0][ks]), "+a"(dof[1][ks]));

    const int64_t slot0 = static_cast<int64_t>(h_kv) * p.n_slots + image_slot0(p.cu_seqlens_k, b);
    const elem_bits* kimg = p.kimg + slot0 * kImageElems;
    const elem_bits* vimg = p.vimg_r + slot0 * kImageElems;
    const uint32_t ring_base = __builtin_amdgcn_readfirstlane(lds_address_of(smem_raw) + wave * 4096);  // this wavefront copies a quarter of every image
    // the unit that lands in this lane's place of a kilobyte
    const uint32_t dma_lane = static_cast<uint32_t>(((lane >> 4) * 16 + (((lane & 15) - 4 * (lane >> 4)) & 15)) * 16);
    auto issue_part = [&](int block, int slot, int part) {     // 1 KiB of 8
        const elem_bits* src = (part < 4 ? kimg : vimg) + static_cast<int64_t>(Walk::index(block)) * kImageElems + wave * 2048 + (part & 3) * 512;
        dma_copy_1k(src, dma_lane, ring_base + slot * kSlotBytes + (part >> 2) * (kSlotBytes / 2) + (part & 3) * 1024);
    };
    auto issue = [&](int block, int slot) {
#pragma unroll
        for (int part = 0; part < 8; ++part) issue_part(block, slot, part);
    };

    // places of this lane's operands inside an image in LDS, for even and odd steps of the depth (fragment (cc, ks)) ...
    const int frag_even = ((n >> 4) * 256 + 16 * h + (((n & 15) + 4 * h) & 15)) * 16;
    const int frag_odd = ((n >> 4) * 256 + 16 * (2 + h) + (((n & 15) + 8 + 4 * h) & 15)) * 16;
    // ... and of its piece of a transposing read, for jj = 0 and 1: key 4 h + rho / 4 (+ 8 jj), columns 16 (lane / 16 % 2) + 4 (rho % 4) ..
    const int rho = lane & 15, tr_g = 2 * ((lane >> 4) & 1) + ((rho & 3) >> 1), tr_r = 4 * h + (rho >> 2) + 4 * tr_g;
    const int tr_0 = (tr_g * 16 + (tr_r & 15)) * 16 + (rho & 1) * 8, tr_1 = (tr_g * 16 + ((tr_r + 8) & 15)) * 16 + (rho & 1) * 8;

    floatx16 acc[2][4];                                        // dQ^T: column 32 t + 8 (r / 4) + 4 h + r % 4 of row n
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[hf][t][r] = 0.f;
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    floatx16 s[2][2], dp[2][2];                                // [half][32-key chunk]; s holds P from the exponentials on
    int4t ds[2][4];                                            // dS, two elements to a word: [half][2 cc + jj]
    typedef __attribute__((__vector_size__(2 * sizeof(elem_t)))) elem_t elem2;
    auto two_elems = [](float lo, float hi) -> int {
        const elem2 v = {static_cast<elem_t>(lo), static_cast<elem_t>(hi)};
        int w;
        __builtin_memcpy(&w, &v, 4);
        return w;
    };
    const int token_bit = kTokenBits + (n >> x.row_shift);     // of this lane's token of the first half, in a block's bits
    auto against = [&](int hf, int block) -> float { return (block >> (token_bit + hf * per_half)) & 1 ? lse2[hf] : INFINITY; };
    auto hide = [&](int cc, int block) {                       // keys behind the rows' last ones
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int lim = last_of(i_wave + hf * per_half + (n >> x.row_shift)) - Walk::index(block) * kBlockN;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * cc + 8 * (r >> 2) + 4 * h + (r & 3) > lim) s[hf][cc][r] = -INFINITY;
        }
    };
    auto edge = [&](int block) { return Walk::index(block) * kBlockN + kBlockN - 1 > wave_first_key; };   // the last block or two

    // ---- operands: 48 a step, each read three uses ahead ----
    elem8 fr[4];
    auto read_frag = [&](int base, int u, int buf) {           // fragment u = 8 cc + ks of an image
        const unsigned char* at = smem_raw + base + ((u & 1) ? frag_odd : frag_even) + ((u >> 3) * 512 + ((u & 7) >> 1) * 64) * 16;
        const uint4 raw = *reinterpret_cast<const uint4*>(at);
        __builtin_memcpy(&fr[buf], &raw, 16);
    };
    auto read_tr = [&](int base, int u, int buf) {             // fragment u = 8 cc + 4 jj + t of K transposed
        const unsigned char* at = smem_raw + base + (((u >> 2) & 1) ? tr_1 : tr_0) + (u >> 3) * 8192 + (u & 3) * 1024;
        typedef __attribute__((address_space(3))) short4t* Lds;
        const short4t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)at), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(at + 4096));
        __builtin_memcpy(&fr[buf], &lo, 8);
        __builtin_memcpy(reinterpret_cast<unsigned char*>(&fr[buf]) + 8, &hi, 8);
    };
    // use u of a step: 0..15 A (K of the next block), 16..31 B (K of the current one, transposed), 32..47 C (V of the next), 48.. A of the step behind
    auto read_ahead = [&](int u, int cur, int next, int after) {
        if (u < 16) read_frag(next, u, u & 3);
        else if (u < 32) read_tr(cur, u - 16, u & 3);
        else if (u < 48) read_frag(next + kSlotBytes / 2, u - 32, u & 3);
        else read_frag(after, u - 48, u & 3);
    };
    // ---- vector work, element i = 16 hf + r of chunk cc ----
    auto exponential = [&](int cc, int i, float a0, float a1) {
        float v = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i >> 4][cc][i & 15], p.scale_log2, i < 16 ? -a0 : -a1));
        asm volatile("" : "+v"(v));
        s[i >> 4][cc][i & 15] = v;
    };
    auto ds_pair = [&](int cc, int i) {                        // elements i and i + 1
        const int hf = i >> 4, r = i & 15;
        int w = two_elems(s[hf][cc][r] * (dp[hf][cc][r] - dsum[hf]), s[hf][cc][r + 1] * (dp[hf][cc][r + 1] - dsum[hf]));
        asm volatile("" : "+v"(w));
        ds[hf][2 * cc + ((r >> 2) & 1)][(r >> 3) * 2 + ((r & 3) >> 1)] = w;
    };
    auto form_s = [&](int u) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) s[hf][u >> 3] = IV2_MFMA32(fr[u & 3], qf[hf][u & 7], (u & 7) == 0 ? zero : s[hf][u >> 3]);
    };
    auto form_dp = [&](int u) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) dp[hf][u >> 3] = IV2_MFMA32(fr[u & 3], dof[hf][u & 7], (u & 7) == 0 ? zero : dp[hf][u >> 3]);
    };
    auto form_dq = [&](int u) { mfma_both(acc[0][u & 3], acc[1][u & 3], fr[u & 3], ds[0][u >> 2], ds[1][u >> 2]); };

    // ---- the walk ----
    // j0: the block whose gradient is next; j1 is in LDS, j2 and j3 are there or on their way.  The barrier stands between B and C: behind it nobody
    // reads j0 any more, its slot takes the block after j3, and j2 has landed.
    int j0 = walk.next(), j1 = walk.next(), j2 = walk.next(), j3 = j2 >= 0 ? walk.next() : -1;
    int at0 = 0;                                               // slot of j0
    int every = ~0;                                            // bits of the tokens that selected all blocks so far
    if (j0 >= 0) {
        issue(j0, 0);
        issue(j1 >= 0 ? j1 : j0, 1);
        issue(j2 >= 0 ? j2 : j0, 2);
        issue(j3 >= 0 ? j3 : j0, 3);
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");      // j0 and j1
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 3; ++u) read_frag(0, u, u & 3);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            form_s(u);
            if (u < 13) read_frag(0, u + 3, (u + 3) & 3); else read_frag(kSlotBytes / 2, u - 13, (u + 3) & 3);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (edge(j0)) { hide(0, j0); hide(1, j0); }
        const float a0 = against(0, j0), a1 = against(1, j0);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            form_dp(u);
            if (u < 13) read_frag(kSlotBytes / 2, u + 3, (u + 3) & 3); else read_frag(kSlotBytes, u - 13, (u + 3) & 3);
            if (u < 8) {
#pragma unroll
                for (int i = 8 * u; i < 8 * u + 8; ++i) exponential(i >> 5, i & 31, a0, a1);
            } else {
                ds_pair(0, 4 * (u - 8));
                ds_pair(0, 4 * (u - 8) + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    while (j1 >= 0) {                                          // uniform over the workgroup
        const int at1 = (at0 + 1) & 3, at2 = (at0 + 2) & 3;
        const int cur = at0 * kSlotBytes, next = at1 * kSlotBytes, after = at2 * kSlotBytes;
        every &= j0;
        const int j4 = j3 >= 0 ? walk.next() : -1;
        const float a0 = against(0, j1), a1 = against(1, j1);
#pragma unroll
        for (int u = 0; u < 8; ++u) {                          // A
            form_s(u);
            read_ahead(u + 3, cur, next, after);
            ds_pair(1, 4 * u);
            ds_pair(1, 4 * u + 2);
            __builtin_amdgcn_sched_barrier(0);
        }
        const bool cut = edge(j1);
        if (cut) hide(0, j1);
#pragma unroll
        for (int u = 8; u < 16; ++u) {
            form_s(u);
            read_ahead(u + 3, cur, next, after);
            if (u > 8) {
                exponential(0, 2 * (u - 9), a0, a1);
                exponential(0, 2 * (u - 9) + 1, a0, a1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (cut) hide(1, j1);
#pragma unroll
        for (int u = 16; u < 32; ++u) {                        // B
            form_dq(u - 16);
            read_ahead(u + 3, cur, next, after);
#pragma unroll
            for (int i = 14 + (u - 16) * 21 / 8; i < 14 + (u - 15) * 21 / 8; ++i) exponential(i >> 5, i & 31, a0, a1);   // 14 .. 55
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");       // this wavefront's part of j2; j3's may be on its way
        __syncthreads();
#pragma unroll
        for (int u = 32; u < 48; ++u) {                        // C
            form_dp(u - 32);
            read_ahead(u + 3, cur, next, after);
            if (u & 1) issue_part(j4 >= 0 ? j4 : j1, at0, (u - 33) / 2);             // behind the last block the slot takes anything
            if (u < 40) {
                exponential((56 + u - 32) >> 5, (56 + u - 32) & 31, a0, a1);
            } else {
                ds_pair(0, 4 * (u - 40));
                ds_pair(0, 4 * (u - 40) + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        at0 = at1;
        j0 = j1; j1 = j2; j2 = j3; j3 = j4;
    }
    every &= j0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // nothing is on its way to LDS when the workgroup ends
    if (j0 >= 0) {                                             // the last block
        const int cur = at0 * kSlotBytes;
#pragma unroll
        for (int i = 0; i < 32; i += 2) ds_pair(1, i);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            read_tr(cur, u, u & 3);
            form_dq(u);
        }
    }
    // the last MFMAs' results must be out of the matrix pipeline before ordinary instructions read them
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int t = 0; t < 4; ++t) asm volatile("" : "+a"(acc[hf][t]));

    // from here on the arguments are read again: what only the end needs would take registers from the walk
    typedef const __attribute__((address_space(4))) BwdParams* Arguments;
    Arguments late = reinterpret_cast<Arguments>(reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
    asm volatile("" : "+s"(late));
    auto store = [&](const floatx16 (&a)[4], int hf, bool rows) {
        int row = n;
        asm volatile("" : "+v"(row));
        const int i = i_wave + hf * per_half + (row >> x.row_shift), head = row & ((1 << x.row_shift) - 1);
        if (i >= Sq || head >= late->group || !rows) return;
        elem_bits* to = late->dq + (static_cast<int64_t>(q0) + i) * late->dq_tok + h_kv * late->dq_kvh + head * late->dq_grp + 4 * h;
        const float scale = late->scale;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                uint2 wv;
                wv.x = pack_elem2(a[t][4 * i4] * scale, a[t][4 * i4 + 1] * scale);
                wv.y = pack_elem2(a[t][4 * i4 + 2] * scale, a[t][4 * i4 + 3] * scale);
                *reinterpret_cast<uint2*>(to + 32 * t + 8 * i4) = wv;
            }
    };
    // what the dK/dV kernel fetches of a token with one 128-byte transfer: [LSE * log2(e) x 16 | D x 16]
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        const int i = i_wave + hf * per_half + (n >> x.row_shift), head = n & ((1 << x.row_shift) - 1);
        if (i < Sq) {
            float* to = late->rowstat + (static_cast<int64_t>(h_kv) * late->total_q + q0 + i) * 32 + 16 * h + head;
            *to = h == 0 ? lse2[hf] : dsum[hf];
            if (x.row_shift == 3) to[8] = h == 0 ? INFINITY : 0.f;                  // rows of the 16 that a group of 8 does not fill
        }
    }
    const int full = (1 << 2 * per_half) - 1;
    if ((every >> kTokenBits & full) != full) {                            // uniform per wavefront: a block was walked for some rows only
        // An infinity or a NaN in a block passes to rows that did not select it (0 x inf).  Where the result shows one, this wavefront's tokens are
        // walked once more, one at a time and each over its own blocks alone.
        float sum = 0.f;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += __builtin_fabsf(acc[hf][t][r]);
        if (__ballot(!(sum < INFINITY)) != 0ull) {
            for (int t = 0; t < 2 * per_half && i_wave + t < Sq; ++t) {
                const int hf = t >= per_half ? 1 : 0, lk = last_of(i_wave + t);
                const int64_t tok = static_cast<int64_t>(q0) + i_wave + t;
                const int head = n & ((1 << x.row_shift) - 1), headc = head < late->group ? head : late->group - 1;   // every token's rows hold this token's heads
                const elem_bits* qp = late->q + tok * late->q_tok + h_kv * late->q_kvh + headc * late->q_grp + 8 * h;
                const elem_bits* dop = late->dout + tok * late->do_tok + h_kv * late->do_kvh + headc * late->do_grp + 8 * h;
                // this token's LSE and D, from the lanes that hold its rows
                const int from = (n & ((1 << x.row_shift) - 1)) + ((t - hf * per_half) << x.row_shift);
                const float lse_t = __shfl(hf ? lse2[1] : lse2[0], from), d_t = __shfl(hf ? dsum[1] : dsum[0], from);
                BlockWalker own;
                own.init(late->fwd_mask ? late->fwd_mask + (static_cast<int64_t>(h_kv) * late->total_q + tok) * late->n64_fwd : nullptr, late->n64_fwd,
                         lk < 0 ? -1 : lk >> 6);
                floatx16 a[4] = {zero, zero, zero, zero};
                for (int j = own.next(); j >= 0 && j < x.max_blocks; j = own.next()) {
                    const elem_bits* kb = kimg + static_cast<int64_t>(j) * kImageElems;
                    const elem_bits* vb = vimg + static_cast<int64_t>(j) * kImageElems;
                    s[0][0] = s[0][1] = dp[0][0] = dp[0][1] = zero;
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int unit = (n >> 4) * 256 + (n & 15) + 16 * (2 * (u & 1) + h) + (u >> 3) * 512 + ((u & 7) >> 1) * 64;
                        const elem8 kq = *reinterpret_cast<const elem8*>(kb + unit * 8), vq = *reinterpret_cast<const elem8*>(vb + unit * 8);
                        const elem8 qq = *reinterpret_cast<const elem8*>(qp + 16 * (u & 7)), dd = *reinterpret_cast<const elem8*>(dop + 16 * (u & 7));
                        s[0][u >> 3] = IV2_MFMA32(kq, qq, s[0][u >> 3]);
                        dp[0][u >> 3] = IV2_MFMA32(vq, dd, dp[0][u >> 3]);
                    }
                    const int lim = lk - j * kBlockN;
#pragma unroll
                    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                        for (int r = 0; r < 16; r += 2) {
                            float v[2];
#pragma unroll
                            for (int e = 0; e < 2; ++e) {
                                const bool seen = 32 * cc + 8 * (r >> 2) + 4 * h + (r & 3) + e <= lim;
                                const float pr = seen ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[0][cc][r + e], late->scale_log2, -lse_t)) : 0.f;
                                v[e] = pr * (dp[0][cc][r + e] - d_t);
                            }
                            ds[0][2 * cc + ((r >> 2) & 1)][(r >> 3) * 2 + ((r & 3) >> 1)] = two_elems(v[0], v[1]);
                        }
#pragma unroll
                    for (int u = 0; u < 16; ++u) {             // 8 cc + 4 jj + t'
                        const int cc = u >> 3, jj = (u >> 2) & 1, d = 32 * (u & 3) + n;
                        uint32_t w[4];
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const int key = 32 * cc + 16 * (e >> 2) + 8 * jj + 4 * h + (e & 3);
                            const uint32_t bits = kb[(((key >> 4) * 4 + (d >> 5)) * 64 + ((d & 31) >> 3) * 16 + (key & 15)) * 8 + (d & 7)];
                            w[e >> 1] = (e & 1) ? w[e >> 1] | bits << 16 : bits;
                        }
                        elem8 kt, dq;
                        __builtin_memcpy(&kt, w, 16);
                        __builtin_memcpy(&dq, &ds[0][u >> 2], 16);
                        a[u & 3] = IV2_MFMA32(kt, dq, a[u & 3]);
                    }
                }
                store(a, hf, (n >> x.row_shift) == t - hf * per_half);
            }
            return;
        }
    }
    store(acc[0], 0, true);
    store(acc[1], 1, true);
}

// Whether the backward forms dQ by tiles.
// Without a mask by an estimate: a tile walks a block in 2.3 us, a group of 8 tokens in 1.6.  The constants are a fit to 134 backward passes of 1 to 5 sequences of 130 to
// 12000 tokens, 1 to 4 KV heads, groups of 8 and 16.  Near the line the estimate errs by a few per cent: it asks for 7 % more than a tie, with which none of those passes
// became slower than by groups.  Whole backward in us, groups of 8 tokens | tiles (* the one taken here): 2 KV heads of 16, 2048 tokens 231 * | 220; 4 heads of 8, 6000
// tokens 2095 | 1617 *.
// Under a mask, as in the forward, only by what a chunk, a KV head and a batch of the same rows have in common: blocks chosen by score by groups, windows by tiles where
// tiles are the faster walk in a launch that they fill.  Whole backward in us, groups | tiles, groups of 16 unless said otherwise: 33 blocks: 9000 tokens, 2 KV heads 1049 |
// 974, 40000, 1 head 2434 | 2262 (2000, 1 head 133 | 154); 6 blocks: 40000 860 | 862, 60000 1303 | 1313 (1000, 2 heads 84 | 93), groups of 8 40000 804 | 680, 1000, 4 heads 105 |
// 103.
bool dq_tiles_pay(int batch, int num_heads_k, int group, int64_t total_q, int64_t total_k, int max_seqlen_q, int max_seqlen_k, bool causal,
                  int most_selected) {
    if (most_selected != kNoMask) return most_selected < 0 && (group == 8 || most_selected <= -16);
    if (max_seqlen_q <= 0 || max_seqlen_k <= 0) return false;
    const double tiles = walk_time(kTileRows >> tile_row_shift(group), [](double b) { return 18. + 2.3 * b; }, 0.5, batch, num_heads_k, total_q, total_k, max_seqlen_q,
                                   max_seqlen_k, causal);
    const double groups = walk_time(8, [](double b) { return 8. + 1.6 * b; }, 0.7, batch, num_heads_k, total_q, total_k, max_seqlen_q, max_seqlen_k, causal);
    return tiles < 0.93 * groups;
}

int launch_bwd_dq_tile(hipStream_t st, const BwdParams& p, int batch, int max_seqlen_q, bool causal) {
    TileExtra x{};
    x.batch = batch;
    x.heads_k = p.num_heads_k;
    x.sequences = p.num_heads_k * batch;
    x.row_shift = tile_row_shift(p.group);
    x.tiles_per_seq = tiles_per_sequence(p.group, max_seqlen_q);
    x.max_blocks = p.k_blocks;
    const int64_t total = static_cast<int64_t>(x.sequences) * x.tiles_per_seq;
    IV2_CHECK(total <= max_workgroups(64 * kTileWaves) - 8, "varlen_bwd: too many token groups");
    IV2_CHECK(p.k_blocks <= 16384, "varlen_bwd: more than %d key blocks per sequence", 16384);      // what the hybrid walk's mask rows hold: accepted by either or by none
    const int64_t grid = (total + 7) / 8 * 8;
    const size_t lds = kDqSlots * kSlotBytes;
    const auto kernel = causal ? &bwd_dq_tile_kernel<true> : &bwd_dq_tile_kernel<false>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    IV2_CHECK(e == hipSuccess, "varlen_bwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * kTileWaves), lds, st, p, x);
    IV2_LAUNCH_CHECK();
    return 0;
}

}  // namespace IV2_NS

#ifndef IV2_F16        // element-type independent: defined once
extern "C" int infllmv2_varlen_bwd_dq_tiles(int batch, int64_t total_q, int64_t total_k, int num_heads, int num_heads_k, int max_seqlen_q,
                                            int max_seqlen_k, int is_causal, int most_selected) {
    return num_heads_k > 0 && batch > 0 && IV2_NS::dq_tiles_pay(batch, num_heads_k, num_heads / num_heads_k, total_q, total_k, max_seqlen_q,
                                                                max_seqlen_k, is_causal != 0, most_selected) ? 1 : 0;
}
#endif
