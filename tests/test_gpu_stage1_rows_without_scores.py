"""Rows that take as many blocks as they can score: the selecting Stage 1 forms no scores for them, and its mask words are still those of Stage 1, pooling
and top-k one after the other, on either side of the line, with forced blocks behind a row's last one, windows wider than
the selection, scores that are all equal or zero, and one token to a wavefront or, beyond 10 240, two."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, hk", [([2], 1), ([30, 33, 65], 1), ([1023], 1), ([1040, 0, 1025], 2), ([4097], 1), ([4096, 2100, 700], 4), ([10300, 1100], 1)])
def test_same_words_as_with_scores(lens, hk, dtype):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(sum(lens))
    r = lambda heads: torch.randn(sum(lens), heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = r(16 * hk), r(hk), r(hk)
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device="cuda")
    held = torch.zeros(len(lens), dtype=torch.int32, device="cuda")
    blocks = -(-max(lens) // 64)
    for topk in sorted({1, 2, 15, 16, 17, max(1, blocks - 1), blocks, blocks + 1, 200}):
        for local, init in ((0, 0), (1, 1), (topk + 3, 0), (0, topk + 2), (2, blocks + 5)):
            for scaled in (q, q * 30, torch.zeros_like(q)):
                got = _lib.host.select_mask(scaled, k, v, cu, max(lens), topk, local, init, 128 ** -0.5, 32, 16, 64)[1]
                want = ops.select_blocks(scaled, k, cu, cu, max(lens), max(lens), topk, local, init, cache_lens=held, max_cache_len=0, causal=True,
                                         return_mask=True)[1]
                assert torch.equal(got, want), (topk, local, init)
