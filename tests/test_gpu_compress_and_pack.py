"""Compressed keys and block images in one launch: the bytes of the launches that make them apart, at sequences around a block, a window and
the rows one workgroup takes, empty ones, dense and strided k and v; and the layer with k and v in every order it accepts, packed along with the
selection or not, bit for bit the selection followed by an attention that packs for itself."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, hk, sets", [
    ([1, 63, 64, 65, 127, 128, 129], 2, [(32, 16), (128, 64)]),
    ([0, 5, 0, 31], 1, [(32, 16), (128, 64)]),                   # no window at all
    ([1000, 33], 3, [(16, 8), (64, 32)]),                        # windows whose staging is smaller than a block's rows
    ([700], 2, [(300, 7), (1200, 28)]),                          # ... and larger than the LDS holds
    ([33000, 64], 1, [(32, 16), (128, 64)]),
])
def test_same_bytes_as_apart(lens, hk, sets, dtype):
    from infllmv2_cuda_impl_amd import _lib
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(5)
    total, batch, stream = sum(lens), len(lens), torch.cuda.current_stream(dev).cuda_stream
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device=dev)
    size = _lib.lib.infllmv2_kv_image_bytes(total, batch, hk)
    both = torch.randn(total, 2, hk, 128, generator=g).to(dtype).to(dev)
    for k, v in ((both[:, 0], both[:, 1]), (both[:, 0].contiguous(), both[:, 1].transpose(0, 1).contiguous().transpose(0, 1))):
        ks, vs = _lib.i64_array(k.stride()[:2]), _lib.i64_array(v.stride()[:2])
        fresh = lambda: [torch.full((total // st + 1, hk, 128), 7.0, dtype=dtype, device=dev) for _, st in sets] + \
                        [torch.full((batch + 1,), -1, dtype=torch.int32, device=dev) for _ in sets] + [torch.zeros(size, dtype=torch.uint8, device=dev)]
        a, b, cu_a, cu_b, images = want = fresh()
        _lib.call_for(dtype, "infllmv2_compress_keys_pair", stream, k.data_ptr(), a.data_ptr(), b.data_ptr(), cu.data_ptr(), cu_a.data_ptr(),
                      cu_b.data_ptr(), batch, max(lens), hk, 128, *k.stride()[:2], *sets[0], *sets[1])
        _lib.call("infllmv2_pack_kv", stream, k.data_ptr(), v.data_ptr(), cu.data_ptr(), images.data_ptr(), size, batch, total, hk, 128, max(lens), ks, vs)
        a, b, cu_a, cu_b, images = got = fresh()
        _lib.call_for(dtype, "infllmv2_compress_keys_and_pack", stream, k.data_ptr(), v.data_ptr(), a.data_ptr(), b.data_ptr(), cu.data_ptr(),
                      cu_a.data_ptr(), cu_b.data_ptr(), images.data_ptr(), size, batch, total, max(lens), hk, 128, ks, vs, *sets[0], *sets[1])
        for x, y in zip(want, got):
            assert torch.equal(x, y)
        with pytest.raises(RuntimeError, match="workspace too small"):
            _lib.call_for(dtype, "infllmv2_compress_keys_and_pack", stream, k.data_ptr(), v.data_ptr(), a.data_ptr(), b.data_ptr(), cu.data_ptr(),
                          cu_a.data_ptr(), cu_b.data_ptr(), images.data_ptr(), size - 1025, batch, total, max(lens), hk, 128, ks, vs, *sets[0], *sets[1])


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("lens", [[300, 1, 777], [32768], [32769]])
def test_layer_takes_every_order(lens, d):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    from infllmv2_cuda_impl_amd.attention import attend_varlen, pad_head_dim
    dev, total, hk = torch.device("cuda:0"), sum(lens), 1
    g = torch.Generator(device="cpu").manual_seed(6)
    r = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).to(dev)
    q, kv = r(total, 16 * hk, d), r(total, 2, hk, d)
    k, v = kv[:, 0].contiguous(), kv[:, 1].contiguous()
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device=dev)
    layer = ops.InfLLMv2Attention(topk=8, local_blocks=2)
    args = (cu, max(lens), 8, 2, 1, d ** -0.5, 32, 16, 64)
    shifted = torch.empty(v.numel() + 4, dtype=v.dtype, device=dev)[4:].view(v.shape).copy_(v)
    idx, mask, _ = _lib.host.select_mask(*pad_head_dim(q, k), v, *args)
    want = attend_varlen(q, k, v, cu, cu, max(lens), max(lens), causal=True, topk_idx=idx, block_mask=mask)
    for kk, vv, packed in ((k, v, True), (kv[:, 0], kv[:, 1], True), (k, v.transpose(0, 2).contiguous().transpose(0, 2), False), (k, shifted, False)):
        images = _lib.host.select_mask(*pad_head_dim(q, kk), vv, *args)[2]
        assert (images is not None) == (packed and d == 128 and max(lens) <= 32768)
        if vv is shifted and d == 128:                           # refused by the attention, as without a selection
            with pytest.raises(RuntimeError, match="16-byte aligned"):
                layer(q, kk, vv, cu, max(lens))
            continue
        assert torch.equal(layer(q, kk, vv, cu, max(lens)), want)
        leaves = [t.detach().requires_grad_(True) for t in (q, kk, vv)]
        out = layer(*leaves, cu, max(lens))
        assert torch.equal(out.detach(), want)
        grads = torch.autograd.grad(out, leaves, torch.ones_like(out))
        assert all(torch.isfinite(x).all() for x in grads)
    wrong = v[:-1]                                               # other errors are the attention's as before
    with pytest.raises(RuntimeError, match="k and v must have shape"):
        layer(q, k, wrong, cu, max(lens))
