"""Block images and the mask words of an index list in one launch: the bytes of the launches that make them apart, with ragged and empty sequences, rows that
do not fill a workgroup, unused and out-of-range indices, lists of no entry and words beyond the keys; and an operator call with indices, on both sides of
the length where the two are made apart, bit for bit the call with the mask words."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens, hk, rows, topk, n64", [
    ([1, 64, 65, 0, 130], 2, 1, 5, 1),
    ([700], 1, 4, 16, 1),
    ([700, 5000], 3, 1027, 64, 2),
    ([64], 2, 6, 0, 3),                                          # lists of no entry
    ([33], 1, 259, 200, 512),                                    # many words: more than the images' LDS
    ([100, 100], 2, 0, 8, 2),
])
def test_same_bytes_as_apart(lens, hk, rows, topk, n64):
    from infllmv2_cuda_impl_amd import _lib
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(5)
    total, batch, stream = sum(lens), len(lens), torch.cuda.current_stream(dev).cuda_stream
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device=dev)
    size = _lib.lib.infllmv2_kv_image_bytes(total, batch, hk)
    kv = torch.randn(total, 2, hk, 128, generator=g).to(torch.bfloat16).to(dev)
    k, v = kv[:, 0], kv[:, 1].contiguous()
    ks, vs = _lib.i64_array(k.stride()[:2]), _lib.i64_array(v.stride()[:2])
    idx = torch.randint(-3, n64 * 64 + 5, (max(rows, 1), max(topk, 1)), generator=g).to(torch.int32).to(dev)
    images = [torch.zeros(size, dtype=torch.uint8, device=dev) for _ in range(2)]
    words = [torch.full((rows + 3, n64), -7, dtype=torch.int64, device=dev) for _ in range(2)]
    args = lambda n: (stream, k.data_ptr(), v.data_ptr(), cu.data_ptr(), images[n].data_ptr(), size, batch, total, hk, 128, max(lens), ks, vs)
    _lib.call("infllmv2_pack_kv", *args(0))
    _lib.call("infllmv2_topk_to_uint64", stream, idx.data_ptr(), words[0].data_ptr(), rows, topk, n64 * 64, n64)
    _lib.call("infllmv2_pack_kv_and_topk", *args(1), idx.data_ptr(), words[1].data_ptr(), rows, topk, n64)
    assert torch.equal(images[0], images[1]) and torch.equal(words[0], words[1])
    assert (words[1][rows:] == -7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq, sk", [([300, 0, 65], [300, 40, 777]), ([9], [32768]), ([9], [32769])])
def test_operator_with_indices_equals_words(sq, sk, dtype):
    import infllmv2_cuda_impl_amd as ops
    dev, hk = torch.device("cuda:0"), 2
    g = torch.Generator(device="cpu").manual_seed(6)
    r = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(dev)
    cu = lambda ns: torch.tensor(np.cumsum([0] + ns), dtype=torch.int32, device=dev)
    q, kv = r(sum(sq), 16 * hk, 128), r(sum(sk), 2, hk, 128)
    k, v = kv[:, 0], kv[:, 1]
    idx = torch.randint(-1, (max(sk) + 63) // 64, (hk, sum(sq), 12), generator=g).to(torch.int32).to(dev)
    words, _ = ops.topk_to_uint64(idx, max(sk), 64)
    more = dict(causal=True)
    want = ops.infllmv2_attn_varlen_func(q, k, v, cu(sq), cu(sk), max(sq), max(sk), topk_idx=idx, block_mask=words, **more)
    got = ops.infllmv2_attn_varlen_func(q, k, v, cu(sq), cu(sk), max(sq), max(sk), topk_idx=idx, **more)
    wide = ops.infllmv2_attn_varlen_func(q, k, v, cu(sq), cu(sk), max(sq), max(sk), topk_idx=idx.transpose(0, 1).contiguous().transpose(0, 1), **more)
    assert torch.equal(got, want) and torch.equal(wide, want)
    leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
    out = ops.infllmv2_attn_varlen_func(*leaves, cu(sq), cu(sk), max(sq), max(sk), topk_idx=idx, deterministic=True, **more)
    grads = torch.autograd.grad(out, leaves, torch.ones_like(out))
    out2 = ops.infllmv2_attn_varlen_func(*leaves, cu(sq), cu(sk), max(sq), max(sk), topk_idx=idx, block_mask=words, deterministic=True, **more)
    for a, b in zip(grads, torch.autograd.grad(out2, leaves, torch.ones_like(out2))):
        assert torch.equal(a, b)
