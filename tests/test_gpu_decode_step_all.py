"""Decode steps whose rows hold no more blocks than the selection takes: no scores, and attention, append and compressed keys in one launch.  Outputs, caches and
lengths are, bit for bit, those of the step operator by operator, around the tokens that complete a window, with the keepers in workgroups
of their own and in the attention's, with one split, and with more (sequence, KV head) pairs than CUs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype, Hk, G, lens, topk", [
    (torch.bfloat16, 2, 16, [1, 30, 31, 32, 126, 127, 128, 191, 1022], 16), (torch.float16, 1, 8, [0], 1), (torch.bfloat16, 1, 16, [63, 62], 1),
    (torch.bfloat16, 2, 16, [2047], 64), (torch.bfloat16, 2, 1, [511, 4094], 64), (torch.float16, 2, 16, [127 + 16 * i for i in range(32)], 64),
    (torch.bfloat16, 4, 16, [255 - i for i in range(64)], 4), (torch.bfloat16, 2, 16, [191 + 3 * i for i in range(130)], 300)])
def test_step_equals_the_separate_operators(dtype, Hk, G, lens, topk):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    B, most = len(lens), max(lens) + 1
    cap = (most + 63) // 64 * 64 + 64
    g = torch.Generator(device="cuda").manual_seed(B + most)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    q, kn, vn = mk(B, 1, Hk * G, 128), mk(B, 1, Hk, 128), mk(B, 1, Hk, 128)
    k, v = mk(B, cap, Hk, 128), mk(B, cap, Hk, 128)
    L = torch.tensor(lens, dtype=torch.int32, device="cuda")
    fine, coarse = mk(B, cap // 16 + 1, Hk, 128), mk(B, cap // 64 + 1, Hk, 128)
    fl, cl = ops.compress_keys_cache_pair(k, L, (32, 16, fine), (128, 64, coarse))
    k2, v2, f2, c2, fl2, cl2 = (t.clone() for t in (k, v, fine, coarse, fl, cl))
    n2, mask = _lib.host.decode_step(q, kn, vn, k2, v2, f2, c2, L, 0, fl2, cl2, most, 32, 16, 64, topk, 2, 1, 128 ** -0.5)
    splits = min(_lib.lib.infllmv2_fwd_kvcache_num_splits(B, Hk, 0), (topk + 3) // 4) if B * Hk <= 256 else 0
    want = ops.infllmv2_attn_with_kvcache(q, k2, v2, cache_seqlens=n2, block_mask=mask, num_splits=splits)
    one = B == 1
    got, n = _lib.host.decode_sparse(q, kn, vn, k, v, fine, coarse, None if one else L, lens[0] if one else 0, None if one else fl, None if one else cl, most,
                                     32, 16, 64, topk, 2, 1, 128 ** -0.5)
    for a, b in ((got, want), (k, k2), (v, v2), (fine, f2), (coarse, c2)) + (() if one else ((n, n2), (fl, fl2), (cl, cl2))):
        assert torch.equal(a, b)


@pytest.mark.parametrize("block_size", [0, 32, 128])
@pytest.mark.parametrize("lens", [[100], [100, 5000]])
def test_other_block_sizes_are_refused(block_size, lens):
    """Before anything is divided by them."""
    import infllmv2_cuda_impl_amd as ops
    layer, cap, B = ops.InfLLMv2Attention(topk=16, block_size=block_size), 8192, len(lens)
    rand = lambda *s: torch.randn(*s, device="cuda").to(torch.bfloat16)
    cache = ops.BatchCache.empty(B, cap, 2, 128, "cuda")
    layer.fill_cache(cache, rand(sum(lens), 2, 128), rand(sum(lens), 2, 128), lens)
    with pytest.raises(RuntimeError, match="only 64-token blocks"):
        layer.decode_batch(rand(B, 1, 32, 128), rand(B, 1, 2, 128), rand(B, 1, 2, 128), cache)
