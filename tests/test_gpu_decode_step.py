"""The kernels of a decode step at the sizes where they can go wrong: the workgroup-per-row top-k at its row lengths and with
ties, the index-list form of the decode attention, and the launch that appends a token, extends the compressed keys and
scores, around the lengths at which windows and 64-key tiles complete."""
import numpy as np
import pytest
import torch

from oracle import infllmv2_oracle as O
from conftest import bf16_np, words_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [257, 511, 512, 513, 1024, 1025, 2047, 2048, 2049, 4097, 8192])
@pytest.mark.parametrize("k", [1, 16, 64, 65, 300])
def test_topk_with_a_workgroup_per_row(n, k):
    from infllmv2_cuda_impl_amd import topk_blocks
    g = torch.Generator(device="cpu").manual_seed(n * 7 + k)
    rows = torch.stack([torch.randn(n, generator=g), torch.randint(0, 3, (n,), generator=g).float(), torch.zeros(n),
                        torch.where(torch.rand(n, generator=g) < 0.995, torch.tensor(float("-inf")), torch.randn(n, generator=g)),
                        torch.where(torch.rand(n, generator=g) < 0.02, torch.tensor(float("inf")), torch.randn(n, generator=g).abs())])
    pooled = rows.to(torch.bfloat16)
    ref = O.topk_blocks(bf16_np(pooled), k)
    idx, mask = topk_blocks(pooled.cuda(), k, return_mask=True)
    assert np.array_equal(idx.cpu().numpy(), ref)
    words = O.topk_to_uint64(ref, n * 64, 64)[0]
    assert np.array_equal(words_np(mask), words)
    by_index = topk_blocks(pooled.cuda(), k, by_index=True).cpu().numpy()
    srt = np.sort(np.where(ref < 0, 1 << 30, ref), axis=-1)
    assert np.array_equal(by_index, np.where(srt == 1 << 30, -1, srt))
    kept = topk_blocks(pooled.cuda(), k, drop_unreachable=True).cpu().numpy()
    vals = bf16_np(pooled)
    for r in range(len(ref)):
        want = [c for c in ref[r] if c >= 0 and vals[r, c] > -np.inf]
        assert kept[r].tolist() == want + [-1] * (k - len(want))


@pytest.mark.parametrize("splits", [0, 1, 3, 64])
@pytest.mark.parametrize("new", [0, 1, 2])
def test_decode_with_an_index_list_equals_the_mask(splits, new):
    """Unsorted, repeated and unused (-1) slots; lengths at block and cache edges (the last sequence's cache is full)."""
    import infllmv2_cuda_impl_amd as ops
    B, cap, Hk = 5, 4288, 2
    lens = [4288 - new, 64 - new, 1, 4160, 4288]
    g = torch.Generator(device="cpu").manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()
    q, kc, vc = mk(B, 1, 32, 128), mk(B, cap, Hk, 128), mk(B, cap, Hk, 128)
    kn, vn = (mk(B, new, Hk, 128), mk(B, new, Hk, 128)) if new else (None, None)
    idx = torch.randint(-1, cap // 64 + 2, (B, Hk, 1, 70), generator=g).to(torch.int32)
    idx[:, :, :, 40:50] = idx[:, :, :, :10]
    idx[1, 0] = -1                                             # nothing selected
    idx[:, 1, 0, 3] = ((torch.tensor(lens) + max(new, 1) - 1).clamp(max=cap - 1) // 64).to(torch.int32)    # the newest block
    words = torch.from_numpy(O.topk_to_uint64(idx.numpy(), cap, 64)[0].view(np.int64)).cuda()
    L = torch.tensor(lens, dtype=torch.int32).cuda()
    res = []
    for opt in ({"topk_idx": idx.cuda()}, {"block_mask": words}):
        k2, v2 = kc.clone(), vc.clone()
        out, lse = ops.infllmv2_attn_with_kvcache(q, k2, v2, k=kn, v=vn, cache_seqlens=L, num_splits=splits, return_softmax_lse=True, **opt)
        res.append((out, lse, k2, v2))
    # the two forms may cut the row into different numbers of runs
    assert (res[0][0].float() - res[1][0].float()).abs().max() <= 8e-3 and torch.equal(res[0][2], res[1][2]) and torch.equal(res[0][3], res[1][3])
    kr, vr = bf16_np(kc).copy(), bf16_np(vc).copy()
    ro, rl = O.decode_forward(bf16_np(q), kr, vr, np.minimum(np.array(lens), cap - new), words_np(words), 128 ** -0.5,
                              None if kn is None else bf16_np(kn), None if vn is None else bf16_np(vn))
    ok = [b for b in range(B) if lens[b] + new <= cap]         # a full cache takes no key: compared between the two forms only
    err = np.abs(bf16_np(res[0][0]) - ro)[ok]
    assert err.max() <= 2e-2 and err.mean() <= 1e-3
    assert np.array_equal(bf16_np(res[0][2])[ok], kr[ok]) and np.array_equal(bf16_np(res[0][3])[ok], vr[ok])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hk,G", [(2, 16), (1, 8)])
def test_step_launch_equals_the_separate_operators(dtype, Hk, G):
    """Append + compressed keys + scores + top-k of one step, per sequence, against compress_keys_cache_pair,
    infllmv2_attn_stage1_kvcache and topk_blocks; with per-sequence lengths on the device and with one host length."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    lens = [30, 31, 32, 47, 126, 127, 128, 191, 64 * 128 + 63, 64 * 64 * 2 + 127, 8703, 5000]
    cap = 8704
    g = torch.Generator(device="cuda").manual_seed(11)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    B = len(lens)
    q, kn, vn = mk(B, 1, Hk * G, 128), mk(B, 1, Hk, 128), mk(B, 1, Hk, 128)
    k, v = mk(B, cap, Hk, 128), mk(B, cap, Hk, 128)
    L = torch.tensor(lens, dtype=torch.int32, device="cuda")
    fine, coarse = mk(B, cap // 16 + 1, Hk, 128), mk(B, cap // 64 + 1, Hk, 128)
    fl, cl = ops.compress_keys_cache_pair(k, L, (32, 16, fine), (128, 64, coarse))
    # what the step has to leave behind
    k2, v2, f2, c2, n2 = k.clone(), v.clone(), fine.clone(), coarse.clone(), L + 1
    for b, n in enumerate(lens):
        k2[b, n], v2[b, n] = kn[b, 0], vn[b, 0]
    fl2, cl2 = ops.compress_keys_cache_pair(k2, n2, (32, 16, f2), (128, 64, c2), old_lens=L, max_new_rows=1)
    pooled = ops.infllmv2_attn_stage1_kvcache(q, f2, c2, fl2, cl2, L, 2, 1, max_cache_len=cap - 1)
    _, want = ops.topk_blocks(pooled, 16, return_mask=True, by_index=True)
    got_n, mask = _lib.host.decode_step(q, kn, vn, k, v, fine, coarse, L, 0, fl, cl, cap, 32, 16, 64, 16, 2, 1, 128 ** -0.5)
    for a, b in ((got_n, n2), (k, k2), (v, v2), (fine, f2), (coarse, c2), (fl, fl2), (cl, cl2)):
        assert torch.equal(a, b)
    assert torch.equal(mask[:, :, 0, :want.shape[-1]], want)
    # one sequence, its length on the host
    for b in (1, 5, 10):
        s = slice(b, b + 1)
        k[b, lens[b]] = 0
        n1, m1 = _lib.host.decode_step(q[s], kn[s], vn[s], k[s], v[s], fine[s], coarse[s], None, lens[b], None, None, lens[b] + 1,
                                       32, 16, 64, 16, 2, 1, 128 ** -0.5)
        assert int(n1) == lens[b] + 1 and torch.equal(k[s], k2[s]) and torch.equal(fine[s], f2[s]) and torch.equal(coarse[s], c2[s])
        w = m1.shape[-1]
        blocks = (lens[b] + 64) // 64
        bits = lambda m: ops.uint64_to_bool(m.contiguous(), blocks)
        assert torch.equal(bits(m1[:, :, 0]), bits(want[s]))


@pytest.mark.parametrize("held", [64 * 64 * 4 - 1, 64 * 64 * 4 + 65, 64 * 64 * 8 + 1, 40])
@pytest.mark.parametrize("masked", [False, True])
def test_decode_runs_longer_than_one_look_up(held, masked):
    """Workgroups of four wavefronts and of one, runs of up to and over 64 blocks per wavefront, the new row in the last of them."""
    import infllmv2_cuda_impl_amd as ops
    g = torch.Generator(device="cuda").manual_seed(held)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    cap, Hk = (held + 64) // 64 * 64, 1
    q, kc, vc, kn, vn = mk(1, 1, 16, 128), mk(1, cap, Hk, 128), mk(1, cap, Hk, 128), mk(1, 1, Hk, 128), mk(1, 1, Hk, 128)
    L = torch.tensor([held], dtype=torch.int32, device="cuda")
    words = torch.randint(-2 ** 62, 2 ** 62, (1, Hk, 1, (cap // 64 + 63) // 64), generator=g, device="cuda") | -(2 ** 63) | 1 if masked else None
    kr, vr = kc.clone(), vc.clone()
    kr[:, held], vr[:, held] = kn[:, 0], vn[:, 0]
    s = (q[0, 0].float() @ kr[0, :held + 1, 0].float().t()) * 128 ** -0.5
    if masked:
        j = torch.arange(held + 1, device="cuda") // 64
        s = s.masked_fill(((words[0, 0, 0][j // 64] >> (j % 64)) & 1) == 0, float("-inf"))
    ref = torch.softmax(s, -1) @ vr[0, :held + 1, 0].float()
    for splits in (0, 1, 2, 64):
        k2, v2 = kc.clone(), vc.clone()
        out = ops.infllmv2_attn_with_kvcache(q, k2, v2, k=kn, v=vn, cache_seqlens=L, num_splits=splits, block_mask=words)
        assert torch.equal(k2, kr) and torch.equal(v2, vr)
        assert (out[0, 0].float() - ref).abs().max() <= 1e-2 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("topk", [1, 3, 64, 300])
@pytest.mark.parametrize("tied", [False, True])
def test_selection_inside_the_attention_equals_topk(dtype, topk, tied):
    """Whole steps against decode_step (top-k launch, mask) + infllmv2_attn_with_kvcache: rows of 1 to 2048 block scores, lengths
    at the edges of 64 words and of 256 columns, and all scores equal (a zero query)."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    lens = [0, 62, 63, 64 * 64 - 2, 64 * 64 - 1, 64 * 256 - 1, 64 * 256, 64 * 512 + 5, 131070]
    cap, Hk, B = 131072, 1, len(lens)
    g = torch.Generator(device="cuda").manual_seed(topk)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dtype)
    q, kn, vn = mk(B, 1, 16, 128) * (0 if tied else 1), mk(B, 1, Hk, 128), mk(B, 1, Hk, 128)
    k, v = mk(B, cap, Hk, 128), mk(B, cap, Hk, 128)
    L = torch.tensor(lens, dtype=torch.int32, device="cuda")
    fine, coarse = mk(B, cap // 16 + 1, Hk, 128), mk(B, cap // 64 + 1, Hk, 128)
    fl, cl = ops.compress_keys_cache_pair(k, L, (32, 16, fine), (128, 64, coarse))
    for s, max_len in ((slice(0, B), cap), (slice(0, 1), 1), (slice(3, 4), 64 * 64 - 1), (slice(5, 6), 64 * 256), (slice(6, 7), 64 * 256 + 1)):
        step = (q[s], kn[s], vn[s], k[s], v[s], fine[s], coarse[s], L[s], 0, fl[s].clone(), cl[s].clone(), max_len, 32, 16, 64, topk, 2, 1,
                128 ** -0.5)
        out, n1 = _lib.host.decode_sparse(*step)
        n2, mask = _lib.host.decode_step(*step[:9], fl[s].clone(), cl[s].clone(), *step[11:])
        splits = min(_lib.lib.infllmv2_fwd_kvcache_num_splits(mask.shape[0], Hk, 0), (topk + 3) // 4)
        want = ops.infllmv2_attn_with_kvcache(q[s], k[s], v[s], cache_seqlens=n2, block_mask=mask, num_splits=splits)
        assert torch.equal(n1, n2) and torch.equal(out, want)


@pytest.mark.parametrize("opt", [{"selection": "dense", "block_size": 128}, {"selection": "dense", "block_size": 32, "stride": 8, "kernel_size": 16},
                                 {"selection": "sparse", "dense_len": 1 << 20, "block_size": 128}, {"selection": "sparse", "stride": 15}])
def test_steps_of_layers_with_other_block_sizes_and_strides(opt):
    """Where nothing is scored the block size is not looked at; where blocks are scored, the strides that put four compressed keys on a
    block.  Against the operators called one by one."""
    import infllmv2_cuda_impl_amd as ops
    layer = ops.InfLLMv2Attention(topk=4, local_blocks=1, **opt)
    ks, st = layer.kernel_size, layer.stride
    g = torch.Generator(device="cuda").manual_seed(3)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    n, Hk = 1000, 2
    one, batch = [c.empty(*a, n + 64, Hk, 128, "cuda", stride=st) for c, a in ((ops.SequenceCache, ()), (ops.BatchCache, (2,)))]
    k, v = mk(2 * n, Hk, 128), mk(2 * n, Hk, 128)
    layer.fill_cache(batch, k, v, [n, n])
    one.k[0, :n], one.v[0, :n], one.length = k[:n], v[:n], n
    layer._extend_compressed(one, 0)
    for step in range(3):
        q, kn, vn = mk(2, 1, 32, 128), mk(2, 1, Hk, 128), mk(2, 1, Hk, 128)
        out1, out2 = layer.decode(q[:1], kn[:1], vn[:1], one), layer.decode_batch(q, kn, vn, batch)
        held = batch.lengths - 1
        assert torch.equal(one.k[0, n + step], kn[0, 0]) and torch.equal(batch.k[:, n + step], kn[:, 0]) and int(held[0]) == n + step
        idx = None
        if layer.selection == "sparse" and layer.dense_len == 0:
            f, c = torch.zeros_like(batch.k_fine), torch.zeros_like(batch.k_coarse)
            fl, cl = ops.compress_keys_cache_pair(batch.k, batch.lengths, (ks, st, f), (4 * ks, 4 * st, c))
            assert torch.equal(fl, batch.fine_lens) and torch.equal(cl, batch.coarse_lens)
            pooled = ops.infllmv2_attn_stage1_kvcache(q, f, c, fl, cl, held, layer.local_blocks, layer.init_blocks, max_cache_len=n + step, stride=st)
            idx = ops.topk_blocks(pooled, layer.topk).unsqueeze(2)
        want = ops.infllmv2_attn_with_kvcache(q, batch.k, batch.v, cache_seqlens=batch.lengths, topk_idx=idx)
        assert (out2.float() - want.float()).abs().max() <= 8e-3          # the runs may be cut differently
        assert (out1.float() - want[:1].float()).abs().max() <= 8e-3


@pytest.mark.parametrize("selection", ["sparse", "dense"])
@pytest.mark.parametrize("which, rows, last", [("k_fine", 3, 79), ("k_coarse", 1, 191)])
def test_a_compressed_cache_without_room_is_refused(selection, which, rows, last):
    """One sequence: the step that completes a window (the fourth of 32/16 with token 80, the second of 128/64 with token 192) finds no
    row for its mean."""
    import infllmv2_cuda_impl_amd as ops
    layer = ops.InfLLMv2Attention(topk=2, local_blocks=0, selection=selection)
    cache = ops.SequenceCache.empty(256, 1, 128, "cuda")
    setattr(cache, which, getattr(cache, which)[:rows])
    mk = lambda h: torch.randn(1, 1, h, 128, device="cuda").to(torch.bfloat16)
    cache.length = last - 1
    layer.decode(mk(16), mk(1), mk(1), cache)
    with pytest.raises(RuntimeError, match="out must be a contiguous"):
        layer.decode(mk(16), mk(1), mk(1), cache)
    assert cache.length == last


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [70, 700])
@pytest.mark.parametrize("topk", [1, 5, 64, 800])
def test_selection_inside_the_attention_takes_signed_zeros(dtype, n, topk):
    """Rows of -0 alone, of both zeros, with -inf and +inf among them: -0 and +0 tie, as in topk_blocks."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    g = torch.Generator(device="cpu").manual_seed(n + topk)
    z = torch.where(torch.rand(4, n, generator=g) < 0.5, -0.0, 0.0)
    z[0] = -0.0
    z[2] = torch.where(torch.rand(n, generator=g) < 0.3, torch.tensor(float("-inf")), z[2])
    z[3] = torch.where(torch.rand(n, generator=g) < 0.1, torch.rand(n, generator=g), z[3])
    z[3, 0], z[3, n - 1] = float("inf"), float("inf")
    scores = z.to(dtype).cuda()
    B, L = 4, 64 * n - 3
    gc = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, generator=gc, device="cuda", dtype=dtype)
    q, kc, vc = mk(B, 1, 16, 128), mk(B, 64 * n, 1, 128), mk(B, 64 * n, 1, 128)
    lens = torch.full((B,), L, dtype=torch.int32, device="cuda")
    splits = 4
    out, lse = torch.empty_like(q), torch.empty((B, 16, 1), dtype=torch.float32, device="cuda")
    ws = torch.empty(_lib.lib.infllmv2_fwd_kvcache_workspace_bytes(B, 1, splits), dtype=torch.uint8, device="cuda")
    two, s3 = lambda t: _lib.i64_array([t.stride(0), t.stride(2)]), lambda t: _lib.i64_array(t.stride()[:3])
    _lib.call_for(dtype, "infllmv2_fwd_kvcache_scores", torch.cuda.current_stream().cuda_stream, q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                  lens.data_ptr(), out.data_ptr(), lse.data_ptr(), scores.data_ptr(), n, topk, ws.data_ptr(), ws.numel(), B, 16, 1, 128, 64 * n,
                  two(q), s3(kc), s3(vc), two(out), splits, 128 ** -0.5)
    _, mask = ops.topk_blocks(scores, topk, return_mask=True)
    want, want_lse = ops.infllmv2_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, block_mask=mask.view(B, 1, 1, -1), num_splits=splits,
                                                    return_softmax_lse=True)
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("batch", [1, 130])                    # workgroups of four wavefronts and, from 257 on, of one
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("held", [63, 64, 129])
def test_cache_rows_far_apart(batch, both, held):
    """Row strides of 2^24 elements, beyond what a 32-bit offset inside a block reaches; K alone, and K and V.  Equal to a dense cache bit
    for bit.  All sequences of the larger batch read the same cache row."""
    import infllmv2_cuda_impl_amd as ops
    cap, Hk, far = 130, 2, 1 << 24
    g = torch.Generator(device="cuda").manual_seed(held)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    k, v, q = mk(1, cap, Hk, 128), mk(1, cap, Hk, 128), mk(batch, 1, 32, 128)
    kn, vn = (mk(1, 1, Hk, 128), mk(1, 1, Hk, 128)) if batch == 1 else (None, None)
    room = torch.empty((cap - 1) * far + 2 * Hk * 128, dtype=torch.bfloat16, device="cuda")      # a row holds K, then V
    part = lambda at: room[at:].as_strided((1, cap, Hk, 128), (cap * far, far, 128, 1))
    k_far, v_far = part(0).copy_(k), part(Hk * 128).copy_(v) if both else v.clone()
    opt = dict(k=kn, v=vn, cache_seqlens=torch.full((batch,), held, dtype=torch.int32, device="cuda"), return_softmax_lse=True,
               cache_batch_idx=torch.zeros(batch, dtype=torch.int32, device="cuda"), num_splits=1)
    out, lse = ops.infllmv2_attn_with_kvcache(q, k_far, v_far, **opt)
    want, want_lse = ops.infllmv2_attn_with_kvcache(q, k, v, **opt)
    assert torch.equal(out, want) and torch.equal(lse, want_lse) and torch.equal(k_far, k) and torch.equal(v_far, v)


@pytest.mark.parametrize("held", [64, 127])
def test_cache_rows_stored_backwards(held):
    """Negative row strides, which the C ABI takes: row 0 of the cache is the last one in memory."""
    from infllmv2_cuda_impl_amd import _lib
    cap, Hk = 128, 2
    g = torch.Generator(device="cuda").manual_seed(held)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    k, v, q = mk(1, cap, Hk, 128), mk(1, cap, Hk, 128), mk(1, 1, 32, 128)
    L = torch.tensor([held], dtype=torch.int32, device="cuda")
    back_k, back_v = k.flip(1).contiguous(), v.flip(1).contiguous()
    zero3, row = _lib.i64_array([0, 0, 0]), Hk * 128

    def call(kt, vt, sign):
        first = 0 if sign > 0 else (cap - 1) * row * 2         # bytes
        out, lse = torch.empty_like(q), torch.empty((1, 32, 1), dtype=torch.float32, device="cuda")
        strides = lambda: _lib.i64_array([cap * row, sign * row, 128])
        _lib.call("infllmv2_fwd_kvcache", torch.cuda.current_stream().cuda_stream, q.data_ptr(), kt.data_ptr() + first, vt.data_ptr() + first, None,
                  None, L.data_ptr(), out.data_ptr(), lse.data_ptr(), None, None, 0, 1, 1, 32, Hk, 128, cap, 0, _lib.i64_array([32 * 128, 128]),
                  strides(), strides(), zero3, zero3, _lib.i64_array([32 * 128, 128]), 0, 1, 128 ** -0.5, None, None, None, 0, 0, None, None, 0, 0)
        return out, lse
    for a, b in zip(call(k, v, 1), call(back_k, back_v, -1)):
        assert torch.equal(a, b)


def test_a_mask_of_more_words_than_lds_holds():
    """A paged cache of 8193 x 64 blocks (33.6 million rows, a few pages behind all of its table): the first sequence is that long, with
    blocks selected in the first and the last words; the second has 70 words, the third one.  Equal to the same blocks as short sequences."""
    import infllmv2_cuda_impl_amd as ops
    Hk, pages, words = 1, 8, 8193
    g = torch.Generator(device="cuda").manual_seed(3)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    kc, vc, q = mk(pages, 64, Hk, 128), mk(pages, 64, Hk, 128), mk(3, 1, 16, 128)
    blocks = words * 64
    table = (torch.arange(blocks, dtype=torch.int32, device="cuda") % pages).expand(3, -1).contiguous()
    picked = [[0, 7, 64 * 8192 + 5, blocks - 2, blocks - 1], [3, 4000, 4479], [1, 2]]
    lens = [blocks * 64 - 17, 4480 * 64, 130]                  # the third's blocks beyond its end do not count
    mask = torch.zeros(3, Hk, 1, words, dtype=torch.int64)
    for b, js in enumerate(picked):
        for j in js + [blocks - 3] * (b > 0):
            mask[b, 0, 0, j // 64] |= -(2 ** 63) if j % 64 == 63 else 1 << (j % 64)
    L = torch.tensor(lens, dtype=torch.int32, device="cuda")
    for splits in (1, 2):
        out, lse = ops.infllmv2_attn_with_kvcache(q, kc, vc, cache_seqlens=L, block_table=table, block_mask=mask.cuda(), num_splits=splits,
                                                  return_softmax_lse=True)
        for b, js in enumerate(picked):
            js = [j for j in js if j * 64 < lens[b]]
            rows = lambda t: torch.cat([t[j % pages, :min(64, lens[b] - 64 * j)] for j in js])[:, 0].float()
            s = q[b, 0].float() @ rows(kc).t().contiguous() * 128 ** -0.5
            want = torch.softmax(s, -1) @ rows(vc)
            assert (out[b, 0].float() - want).abs().max() <= 2e-2 and (lse[b, :, 0] - torch.logsumexp(s, -1)).abs().max() <= 2e-3


@pytest.mark.parametrize("batch, cap, max_len", [(129, 256, 200), (2, 64 * 2049, 64 * 2048), (2, 64 * 2049, 64 * 2048 + 1)])
def test_steps_on_both_sides_of_the_selecting_launch(batch, cap, max_len):
    """More (sequence, KV head) pairs than CUs, and rows of 2048 and of 2049 block scores: a top-k launch and a mask where the attention's
    launch does not select, through the layer."""
    import infllmv2_cuda_impl_amd as ops
    g = torch.Generator(device="cuda").manual_seed(batch)
    Hk, layer = 2, ops.InfLLMv2Attention(topk=3, local_blocks=1)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    lens = [max_len - 1 - 7 * (b % 9) for b in range(batch)]
    cache = ops.BatchCache.empty(batch, cap, Hk, 128, "cuda")
    layer.fill_cache(cache, mk(sum(lens), Hk, 128), mk(sum(lens), Hk, 128), lens)
    held, q, kn, vn = cache.lengths.clone(), mk(batch, 1, 32, 128), mk(batch, 1, Hk, 128), mk(batch, 1, Hk, 128)
    out = layer.decode_batch(q, kn, vn, cache)
    pooled = ops.infllmv2_attn_stage1_kvcache(q, cache.k_fine, cache.k_coarse, cache.fine_lens, cache.coarse_lens, held, 1, 1, max_cache_len=max_len - 1)
    want = ops.infllmv2_attn_with_kvcache(q, cache.k, cache.v, cache_seqlens=held + 1, topk_idx=ops.topk_blocks(pooled, 3).unsqueeze(2))
    assert torch.equal(cache.lengths, held + 1) and (out.float() - want.float()).abs().max() <= 8e-3
