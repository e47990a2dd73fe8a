"""Block images and mask words of rows that take every block, in one launch: the images of infllmv2_pack_kv byte for byte, words of ones up to the last block, nothing
behind them, with ragged and empty sequences, one and several words to a row, and no rows; and a prefill of such sequences bit for bit the one with a mask from top-k."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens, hk, rows, blocks, n64", [([1, 64, 65, 0, 130], 2, 1, 3, 1), ([700], 1, 2048, 11, 1), ([5000, 33], 3, 1027, 79, 2), ([64], 2, 683, 128, 3), ([64], 1, 5, 0, 1),
                                                          ([100, 100], 2, 0, 2, 1)])
def test_same_bytes_as_apart(lens, hk, rows, blocks, n64):
    from infllmv2_cuda_impl_amd import _lib
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(7)
    total, batch, stream = sum(lens), len(lens), torch.cuda.current_stream(dev).cuda_stream
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device=dev)
    size = _lib.lib.infllmv2_kv_image_bytes(total, batch, hk)
    kv = torch.randn(total, 2, hk, 128, generator=g).to(torch.bfloat16).to(dev)
    k, v = kv[:, 0], kv[:, 1].contiguous()
    ks, vs = _lib.i64_array(k.stride()[:2]), _lib.i64_array(v.stride()[:2])
    images = [torch.zeros(size, dtype=torch.uint8, device=dev) for _ in range(2)]
    words = torch.full((rows + 3, n64), -7, dtype=torch.int64, device=dev)
    args = lambda n: (stream, k.data_ptr(), v.data_ptr(), cu.data_ptr(), images[n].data_ptr(), size, batch, total, hk, 128, max(lens), ks, vs)
    _lib.call("infllmv2_pack_kv", *args(0))
    _lib.call("infllmv2_pack_kv_and_first", *args(1), words.data_ptr(), rows, blocks, n64)
    want = [(1 << max(0, min(64, blocks - 64 * w))) - 1 for w in range(n64)]
    want = torch.tensor([x - (1 << 64) if x >> 63 else x for x in want], dtype=torch.int64, device=dev)
    assert torch.equal(images[0], images[1]) and (words[:rows] == want).all() and (words[rows:] == -7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, topk", [([2], 1), ([1024, 1000, 0, 63], 16), ([4096], 64), ([4160, 5], 65)])
def test_prefill(lens, topk, dtype):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    r = lambda heads: torch.randn(sum(lens), heads, 128, generator=g, device="cuda").to(dtype)
    q, k, v = r(32), r(2), r(2)
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device="cuda")
    held = torch.zeros(len(lens), dtype=torch.int32, device="cuda")
    with torch.no_grad():
        got = ops.InfLLMv2Attention(topk=topk, local_blocks=0)(q, k, v, cu, max(lens))
        idx, mask = ops.select_blocks(q, k, cu, cu, max(lens), max(lens), topk, 0, 1, cache_lens=held, max_cache_len=0, return_mask=True)
        want = attend_varlen(q, k, v, cu, cu, max(lens), max(lens), causal=True, topk_idx=idx, block_mask=mask)
    assert torch.equal(got, want)
