// Stage-2 forward by flash tiles of 256 query rows (gfx950): without a mask, or for a window, whose neighbouring rows select nearly the same.
//
// Where every token attends its whole prefix nothing is left to fetch per token, and the hybrid walk (stage2_fwd_hybrid.hip) only
// keeps its costs: 16 query rows per K / V fragment read from LDS, softmax and MFMAs of a wavefront one after the other; where the rows differ a
// little it fetches the rest per token, 32 KiB through the L1 path for 16 rows.  Here a workgroup of 4 wavefronts owns 256 rows (16 tokens of 16
// heads, 32 of 8) and walks the blocks that any of its tokens selected; a row that did not select one has P = 0 there.  K and V come from
// the same block images, through an LDS ring of three blocks.
//
// What bounds it: the power the matrix pipe draws.  16384 dense tokens of 2 KV heads take 1825 us (1.2 PFLOP/s) with random inputs and 1460 with zeros, where
// only the clock differs; a library product of 8192^3 in bf16 makes 1.40 and 1.80 PFLOP/s with both operands in rows, 1.62 and 2.25 with the right one
// transposed.  What a step does beside the MFMAs counts in energy more than in issue slots, and the operand reads from LDS are the largest part: so a
// wavefront takes 64 rows, in two halves of 32 (the N side of v_mfma_f32_32x32x16), and a fragment feeds both.  That is one wavefront per SIMD with 512
// registers (128 of O, 64 each of Q, S, K and V, 32 of P), and the overlap of MFMAs and exponentials is written out: while one half's P V and scores are on
// the matrix pipe, the other half's exponentials are formed.  Before, eight wavefronts of 32 rows, two to a SIMD, read twice the LDS bytes: 1910 us; four
// wavefronts of 32 rows in workgroups of two to a CU 1993; this shape with copies and scalar work at the head of a step instead of between its MFMAs 1979.
// Operator, us, eight wavefronts -> this one: 2500 + 6001 + 4096 tokens 481 -> 455, 777 + 5003 + 1291 + 9173 865 -> 816, 50000 17000 -> 16600.
//
// Operands.  S^T = K Q^T: lane (n = lane % 32, h = lane / 32) holds key n of a 32-key chunk, d = 16 ks + 8 h + j: one 16-byte unit of
// the K image.  The accumulators hold keys 8 i + 4 h + e (register 4 i + e) of row n; a V image unit holds keys 4 g + e and
// 16 + 4 g + e of its chunk, so registers i = jj and i = jj + 2 are, converted, the B operand that goes with the V units of
// g = 2 jj + h: P moves nowhere.
#include "common.h"
#include "kv_image.h"
#include "block_walker.h"
#include "lds_dma.h"
#include "tile_walk.h"
#include "stage2_fwd.h"
#include "infllmv2_hip.h"
#include <math.h>

namespace IV2_NS {

constexpr int kSlots = 3;                                      // of the ring
constexpr float kLazyLimit = 64.f;                             // as in the hybrid walk: a lane's sum of P that the reference exponent has to keep to
constexpr float kNoReference = -3.4028234e38f;

template <bool kCausal>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(1, 1)))
void stage2_fwd_tile_kernel(const FwdParams p, const TileExtra x) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const uint4* ring = reinterpret_cast<const uint4*>(smem_raw);                   // [kSlots][2048]: K units 0..1023, V units 1024..2047

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
    const int per_half = 32 >> x.row_shift;                                         // tokens of half a wavefront
    const int i_wave = i_first + wave * 2 * per_half;
    auto last_of = [&](int t) {                                                     // last key token t attends
        const int lk = kCausal ? t + Sk - Sq : Sk - 1;
        return lk > Sk - 1 ? Sk - 1 : lk;
    };
    const int wave_first_key = last_of(i_wave);                                     // of the wavefront's first token

    elem8 qf[2][8];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        const int i = i_wave + hf * per_half + (n >> x.row_shift), head = n & ((1 << x.row_shift) - 1);
        const int64_t tok = static_cast<int64_t>(q0) + (i < Sq ? i : Sq - 1);
        const elem_bits* qp = p.q + tok * p.q_tok_stride + h_kv * p.q_kvh_stride + (head < p.group ? head : p.group - 1) * p.q_grp_stride + 8 * h;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qf[hf][ks] = *reinterpret_cast<const elem8*>(qp + 16 * ks);
    }

    typedef TileWalk<kCausal> Walk;
    Walk walk;
    {
        const int left = Sq - i_first, all = kTileRows >> x.row_shift;
        walk.tokens = left < all ? left : all;
        const int lk = last_of(i_first + walk.tokens - 1);                          // of the tile's last token
        walk.blocks = lk < 0 ? 0 : (lk >> 6) + 1;
        if (walk.blocks > x.max_blocks) walk.blocks = x.max_blocks;                 // a sequence longer than the announced max_seqlen_k
        walk.rows = p.mask ? p.mask + (static_cast<int64_t>(h_kv) * p.total_q + q0 + i_first) * p.n64 : nullptr;
        walk.n64 = p.n64;
        walk.mine = wave * 2 * per_half;
        walk.per_wave = 2 * per_half;
        walk.last_key = last_of(i_first);
        walk.init();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                // before the first LDS-DMA (see the hybrid walk)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+a"(qf[0][ks]), "+a"(qf[1][ks]));

    const int64_t slot0 = static_cast<int64_t>(h_kv) * p.n_slots + image_slot0(p.cu_seqlens_k, b);
    const elem_bits* kimg = p.kimg + slot0 * kImageElems;
    const elem_bits* vimg = p.vimg + slot0 * kImageElems;
    const uint32_t ring_base = __builtin_amdgcn_readfirstlane(lds_address_of(ring) + wave * 4096);      // this wavefront copies a quarter of every image
    auto issue_part = [&](int block, int slot, int part) {     // 1 KiB of 8
        const elem_bits* src = (part < 4 ? kimg : vimg) + static_cast<int64_t>(Walk::index(block)) * kImageElems + wave * 2048 + (part & 3) * 512;
        dma_copy_1k(src, 16 * lane, ring_base + slot * kSlotBytes + (part >> 2) * (kSlotBytes / 2) + (part & 3) * 1024);
    };
    auto issue = [&](int block, int slot) {
#pragma unroll
        for (int part = 0; part < 8; ++part) issue_part(block, slot, part);
    };

    // m: reference exponent as in softmax_step, but finite from the start (a row whose keys are all hidden so far has P = 0 by itself)
    float m[2] = {kNoReference, kNoReference}, l[2] = {0.f, 0.f};
    floatx16 o[2][4];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[hf][t][r] = 0.f;

    // 16-byte units of this lane inside an image: K unit (2 cc + n/16, ks/2, n%16 + 16 (2 (ks%2) + h)), V unit (2 t + n/16, cc, n%16 + 16 (2 jj + h))
    const int k_unit = (n >> 4) * 256 + (n & 15) + 16 * h;
    const int v_unit = (n >> 4) * 128 + (n & 15) + 16 * h;
    auto k_at = [](int f) { return (f & 1) * 512 + (f >> 2) * 64 + ((f >> 1) & 1) * 32; };               // fragment f = 2 ks + cc
    auto v_at = [](int f) { return (f & 3) * 256 + (f >> 3) * 64 + ((f >> 2) & 1) * 32; };               // fragment f = 8 cc + 4 jj + t
    elem8 kf[16], vf[16];
    auto read_k = [&](int slot, int f) {
        const uint4 raw = ring[slot * 2048 + k_unit + k_at(f)];
        __builtin_memcpy(&kf[f], &raw, 16);
    };
    auto read_v = [&](int slot, int f) {
        const uint4 raw = ring[slot * 2048 + 1024 + v_unit + v_at(f)];
        __builtin_memcpy(&vf[f], &raw, 16);
    };
    floatx16 s[2][2];
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto hide = [&](int hf, int j) {                           // keys behind the row's last one
        const int lim = last_of(i_wave + hf * per_half + (n >> x.row_shift)) - j * kBlockN;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * cc + 8 * (r >> 2) + 4 * h + (r & 3) > lim) s[hf][cc][r] = -INFINITY;
    };
    auto largest = [&](int hf) -> float {                      // of the row, log2 units
        float mx = -INFINITY;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[hf][cc][r]);
        return half_max(mx) * p.scale_log2;
    };
    typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t words4;
    typedef __attribute__((__vector_size__(2 * sizeof(elem_t)))) elem_t elem2;
    auto two_elems = [](float lo, float hi) -> uint32_t {       // one conversion instruction
        const elem2 v = {static_cast<elem_t>(lo), static_cast<elem_t>(hi)};
        uint32_t w;
        __builtin_memcpy(&w, &v, 4);
        return w;
    };
    words4 pf[2][4];                                           // P, two elements to a word
    auto operand = [](const words4& w) {
        elem8 v;
        __builtin_memcpy(&v, &w, 16);
        return v;
    };
    auto exponentials = [&](int hf, float against) -> float {   // P of a block at once; returns the lane's sum
        float sum = 0.f;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float lo = __builtin_amdgcn_exp2f(__builtin_fmaf(s[hf][cc][r], p.scale_log2, -against));
                const float hi = __builtin_amdgcn_exp2f(__builtin_fmaf(s[hf][cc][r + 1], p.scale_log2, -against));
                sum += lo;
                sum += hi;
                pf[hf][2 * cc + ((r >> 2) & 1)][(r >> 3) * 2 + ((r & 3) >> 1)] = two_elems(lo, hi);
            }
        return sum;
    };
    auto rescale = [&](int hf, float m_new) {
        const float alpha = __builtin_amdgcn_exp2f(m[hf] - m_new);
        l[hf] *= alpha;
        m[hf] = m_new;
#pragma unroll
        for (int t = 0; t < 4; ++t) o[hf][t] *= alpha;
    };
    // Half a step: 32 MFMAs for one half of the rows and, spread between them, the exponentials of a block for the other half, each in three
    // places (multiply-add, exp2, sum), so that none waits for its predecessor.  They start a group late, when the last scores have left the matrix pipe, and are through
    // before the last MFMA, so that the branch on their sum costs nothing.  `beside` adds LDS reads, copies and scalar work.  The order is fixed by
    // hand: the compiler's own clumps both sides.
    auto half_step = [&](auto&& mfma, auto&& beside, int hf, float against) -> float {
        float e[32], sum = 0.f;
        auto upto = [](int group) { return group < 1 ? 0 : (group - 1) * 9 / 8 < 32 ? (group - 1) * 9 / 8 : 32; };
#pragma unroll
        for (int g = 0; g < 32; ++g) {
            mfma(g);
            beside(g);
#pragma unroll
            for (int i = upto(g - 1); i < upto(g); ++i) {
                sum += e[i];
                asm volatile("" : "+v"(sum));                  // here, not all at the end
                if (i & 1) {
                    uint32_t two = two_elems(e[i - 1], e[i]);
                    asm volatile("" : "+v"(two));
                    const int r = i & 15;
                    pf[hf][2 * (i >> 4) + ((r >> 2) & 1)][(r >> 3) * 2 + ((r & 3) >> 1)] = two;
                }
            }
#pragma unroll
            for (int i = upto(g); i < upto(g + 1); ++i) {
                e[i] = __builtin_amdgcn_exp2f(e[i]);
                asm volatile("" : "+v"(e[i]));
            }
#pragma unroll
            for (int i = upto(g + 1); i < upto(g + 2); ++i) {
                e[i] = __builtin_fmaf(s[hf][i >> 4][i & 15], p.scale_log2, -against);
                asm volatile("" : "+v"(e[i]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return sum;
    };
    auto form_s = [&](int hf) { return [&, hf](int f) { s[hf][f & 1] = IV2_MFMA32(kf[f], qf[hf][f >> 1], f < 2 ? zero : s[hf][f & 1]); }; };
    auto form_o = [&](int hf) { return [&, hf](int f) { o[hf][f & 3] = IV2_MFMA32(vf[f], operand(pf[hf][f >> 2]), o[hf][f & 3]); }; };
    const int token_bit = kTokenBits + (n >> x.row_shift);     // of this lane's token of the first half, in a block's bits
    auto selects = [&](int hf, int block) -> bool { return (block >> (token_bit + hf * per_half)) & 1; };
    auto against = [&](int hf, int block) -> float { return selects(hf, block) ? m[hf] : INFINITY; };     // rows that did not select the block: P = exp2(-inf)
    auto settle = [&](int hf, int block, float sum) {           // the sum of a block's P, or the block once more
        if (__ballot(!(sum <= kLazyLimit)) != 0ull) {          // a row without a reference yet, one that grew, or NaN
            const float mx = largest(hf);
            const bool selected = selects(hf, block);
            rescale(hf, selected ? fmaxf(m[hf], mx) : m[hf]);
            sum = exponentials(hf, selected ? m[hf] : INFINITY);
        }
        l[hf] += sum;
    };
    auto edge = [&](int block) { return Walk::index(block) * kBlockN + kBlockN - 1 > wave_first_key; };   // the last block or two

    // The walk: j0 is the current block, j1 the next; j1 and j2 are in the ring or on their way, j3 is requested.  The two halves of the rows take turns: while
    // the matrix pipe works on one, the exponentials of the other are formed.  At the top of a step P of j0 is there for the first half, its scores
    // for the second, and V of j0 is in registers.
    int j0 = walk.next(), j1 = walk.next(), j2 = walk.next();
    int at1 = 1;                                               // slot of j1
    int every = ~0;                                            // bits of the tokens that selected all blocks so far
    if (j0 >= 0) {
        issue(j0, 0);
        if (j1 >= 0) issue(j1, 1);
        if (j2 >= 0) issue(j2, 2);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
#pragma unroll
        for (int f = 0; f < 16; ++f) read_k(0, f);
#pragma unroll
        for (int f = 0; f < 16; ++f) read_v(0, f);
#pragma unroll
        for (int f = 0; f < 16; ++f) form_s(0)(f);
#pragma unroll
        for (int f = 0; f < 16; ++f) form_s(1)(f);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            // rows that selected the first block take their reference from it
            if (edge(j0)) hide(hf, Walk::index(j0));
            const float mx = largest(hf);
            if (selects(hf, j0) && mx > kNoReference && mx < INFINITY) m[hf] = mx;
        }
        settle(0, j0, exponentials(0, against(0, j0)));
    }
    while (j1 >= 0) {                                          // uniform over the workgroup
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");       // this wavefront's part of j1; j2's may be on its way
        __syncthreads();
        const int slot = at1, freed = at1 == 0 ? 2 : at1 - 1;  // of j1, of j0
        every &= j0;
        const int j3 = j2 >= 0 ? walk.next() : -1;
        settle(1, j0, half_step([&](int g) { if (g < 16) form_o(0)(g); else form_s(0)(g - 16); }, [&](int g) {
            if (g < 24 && g % 3 != 2) read_k(slot, 2 * (g / 3) + g % 3);
            if (g >= 24 && g % 2 == 0) issue_part(j3 >= 0 ? j3 : j1, freed, (g - 24) / 2);   // behind the last block the slot takes anything
        }, 1, against(1, j0)));
        if (edge(j1)) hide(0, Walk::index(j1));
        settle(0, j1, half_step([&](int g) { if (g < 16) form_o(1)(g); else form_s(1)(g - 16); }, [&](int g) {
            if (g < 8 && g % 2 == 0) issue_part(j3 >= 0 ? j3 : j1, freed, 4 + g / 2);
            if (g >= 8 && (g - 8) % 3 != 2) read_v(slot, 2 * ((g - 8) / 3) + (g - 8) % 3);
        }, 0, against(0, j1)));
        if (edge(j1)) hide(1, Walk::index(j1));
        at1 = at1 == 2 ? 0 : at1 + 1;
        j0 = j1; j1 = j2; j2 = j3;
    }
    every &= j0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // nothing is on its way to LDS when the workgroup ends
    if (j0 >= 0) {                                             // the last block
#pragma unroll
        for (int f = 0; f < 16; ++f) form_o(0)(f);
        settle(1, j0, exponentials(1, against(1, j0)));
#pragma unroll
        for (int f = 0; f < 16; ++f) form_o(1)(f);
    }

    // from here on the arguments are read again: what only the end needs would take registers from the walk
    typedef const __attribute__((address_space(4))) FwdParams* Arguments;
    Arguments late = reinterpret_cast<Arguments>(reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
    asm volatile("" : "+s"(late));
    auto store = [&](const floatx16 (&oo)[4], float mm, float ll, int hf, bool lanes) {
        const float l_tot = half_sum(ll);
        const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        int row = n;
        asm volatile("" : "+v"(row));                          // computed again: the walk has no registers to spare
        const int i = i_wave + hf * per_half + (row >> x.row_shift), head = row & ((1 << x.row_shift) - 1);
        if (i < Sq && head < late->group && lanes) {
            const int64_t tok = static_cast<int64_t>(q0) + i;
            elem_bits* op = late->out + tok * late->o_tok_stride + h_kv * late->o_kvh_stride + head * late->o_grp_stride + 4 * h;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    uint2 wv;
                    wv.x = pack_elem2(oo[t][4 * i4] * inv, oo[t][4 * i4 + 1] * inv);
                    wv.y = pack_elem2(oo[t][4 * i4 + 2] * inv, oo[t][4 * i4 + 3] * inv);
                    *reinterpret_cast<uint2*>(op + 32 * t + 8 * i4) = wv;
                }
            if (h == 0) {
                const float lse = l_tot > 0.f ? mm * 0.69314718055994530942f + logf(l_tot) : INFINITY;
                late->lse[h_kv * late->lse_kvh_stride + tok * late->lse_tok_stride + head * late->lse_grp_stride] = lse;
            }
        }
    };
    const int full = (1 << 2 * per_half) - 1;
    if ((every >> kTokenBits & full) != full) {                            // uniform per wavefront: a block was walked for some rows only
        // An infinity or a NaN in a block passes to rows that did not select it (0 x inf).  Where the result shows one, this wavefront's tokens are
        // walked once more, one at a time and each over its own blocks alone.
        float sum = l[0] + l[1];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += __builtin_fabsf(o[hf][t][r]);
        if (__ballot(!(sum < INFINITY)) != 0ull) {
            for (int t = 0; t < 2 * per_half && i_wave + t < Sq; ++t) {
                const int hf = t >= per_half ? 1 : 0, lk = last_of(i_wave + t);
                {
                    const int head = n & ((1 << x.row_shift) - 1);                  // every token's rows hold this token's heads: the copies are not stored
                    const elem_bits* qp = late->q + (static_cast<int64_t>(q0) + i_wave + t) * late->q_tok_stride + h_kv * late->q_kvh_stride +
                                          (head < late->group ? head : late->group - 1) * late->q_grp_stride + 8 * h;
#pragma unroll
                    for (int ks = 0; ks < 8; ++ks) vf[ks] = *reinterpret_cast<const elem8*>(qp + 16 * ks);
                }
                BlockWalker own;
                own.init(late->mask ? late->mask + (static_cast<int64_t>(h_kv) * late->total_q + q0 + i_wave + t) * late->n64 : nullptr, late->n64,
                         lk < 0 ? -1 : lk >> 6);
                float mm = kNoReference, ll = 0.f;
#pragma unroll
                for (int u = 0; u < 4; ++u) o[0][u] = zero;
                for (int j = own.next(); j >= 0 && j < x.max_blocks; j = own.next()) {
                    const uint4* ks_src = reinterpret_cast<const uint4*>(kimg + static_cast<int64_t>(j) * kImageElems) + k_unit;
                    const uint4* vs_src = reinterpret_cast<const uint4*>(vimg + static_cast<int64_t>(j) * kImageElems) + v_unit;
                    s[0][0] = s[0][1] = zero;
#pragma unroll
                    for (int f = 0; f < 16; ++f) {
                        const uint4 raw = ks_src[k_at(f)];
                        __builtin_memcpy(&kf[0], &raw, 16);
                        s[0][f & 1] = IV2_MFMA32(kf[0], vf[f >> 1], s[0][f & 1]);
                    }
                    const int lim = lk - j * kBlockN;
                    float mx = -INFINITY;
#pragma unroll
                    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            if (32 * cc + 8 * (r >> 2) + 4 * h + (r & 3) > lim) s[0][cc][r] = -INFINITY;
                            mx = fmaxf(mx, s[0][cc][r]);
                        }
                    const float m_new = fmaxf(mm, half_max(mx) * late->scale_log2), alpha = __builtin_amdgcn_exp2f(mm - m_new);
                    mm = m_new;
                    ll = ll * alpha + exponentials(0, mm);
#pragma unroll
                    for (int u = 0; u < 4; ++u) o[0][u] *= alpha;
#pragma unroll
                    for (int f = 0; f < 16; ++f) {
                        const uint4 raw = vs_src[v_at(f)];
                        __builtin_memcpy(&kf[0], &raw, 16);
                        o[0][f & 3] = IV2_MFMA32(kf[0], operand(pf[0][f >> 2]), o[0][f & 3]);
                    }
                }
                store(o[0], mm, ll, hf, (n >> x.row_shift) == t - hf * per_half);
            }
            return;
        }
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) store(o[hf], m[hf], l[hf], hf, true);
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
    const double tiles = walk_time(kTileRows >> tile_row_shift(group), [](double b) { return 10. + 1.5 * b; }, 0.75, batch, num_heads_k, total_q, total_k, max_seqlen_q,
                                   max_seqlen_k, causal);
    const double groups = walk_time(8, [](double b) { return 6. + b; }, 0.7, batch, num_heads_k, total_q, total_k, max_seqlen_q, max_seqlen_k, causal);
    return tiles < groups + 1.;
}

// Whether a forward under a mask goes by tiles.  Masked rows are the same bit for bit whatever else is in their launch (a chunk of the queries, a KV head on
// its own, other sequences), and the two walks round apart: so the choice may use only what all of those have in common, never the size of the launch.
// Blocks chosen by score go by groups of 8 tokens, whatever tiles would gain in a launch that they fill.  A window (neighbouring rows alike) goes by tiles: a tile
// walks what one row has and a little.  Layer prefill in us, groups | tiles, groups of 16 unless said otherwise: 60000 tokens, 1 KV head, 6 blocks 381 | 338; 40000, 33
// blocks 776 | 649; 40000, 6 blocks, groups of 8 224 | 125; 9000, 2 heads, 33 blocks 322 | 268; 30 x 600, 2 heads, 6 blocks 187 | 165.  Launches that do not fill the chip
// pay for it: 1000 tokens, 2 heads, 6 blocks 20.9 | 26.2; 2000, 1 head, 33 blocks 43.5 | 57.7.
bool masked_by_tiles(int most_selected) { return most_selected < 0; }

int launch_stage2_fwd_tile(hipStream_t st, const FwdParams& p, int batch, int num_heads_k, int max_seqlen_q, int max_seqlen_k, bool causal) {
    TileExtra x{};
    x.batch = batch;
    x.heads_k = num_heads_k;
    x.sequences = num_heads_k * batch;
    x.row_shift = tile_row_shift(p.group);
    x.tiles_per_seq = tiles_per_sequence(p.group, max_seqlen_q);
    x.max_blocks = (max_seqlen_k + kBlockN - 1) / kBlockN;
    const int64_t total = static_cast<int64_t>(x.sequences) * x.tiles_per_seq;
    IV2_CHECK(total <= max_workgroups(64 * kTileWaves) - 8, "varlen_fwd: too many token groups");
    const int64_t grid = (total + 7) / 8 * 8;
    const size_t lds = kSlots * kSlotBytes;
    const auto kernel = causal ? &stage2_fwd_tile_kernel<true> : &stage2_fwd_tile_kernel<false>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    IV2_CHECK(e == hipSuccess, "varlen_fwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * kTileWaves), lds, st, p, x);
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
extern "C" int infllmv2_varlen_fwd_masked_tiles(int batch, int64_t /*total_q*/, int64_t /*total_k*/, int /*num_heads*/, int num_heads_k, int /*max_seqlen_q*/,
                                                int /*max_seqlen_k*/, int /*is_causal*/, int most_selected) {
    return num_heads_k > 0 && batch > 0 && IV2_NS::masked_by_tiles(most_selected) ? 1 : 0;
}
#endif
