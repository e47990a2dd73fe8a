"""The selection made by the launch that scores the blocks: the words of Stage 1, pooling and top-k one after the other, bit for bit, at the row lengths where
its registers change, with ragged and empty sequences, fewer blocks than wanted and more, none wanted, equal scores, and every size of group."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def both(q, k, v, lens, topk, local, init):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device="cuda")
    got = _lib.host.select_mask(q, k, v, cu, max(lens), topk, local, init, 128 ** -0.5, 32, 16, 64)[1]
    held = torch.zeros(len(lens), dtype=torch.int32, device="cuda")
    want = ops.select_blocks(q, k, cu, cu, max(lens), max(lens), max(topk, 1), local, init, cache_lens=held, max_cache_len=0, causal=True, return_mask=True)[1]
    if topk == 0:
        want = torch.zeros_like(want)
    assert got.shape == want.shape and torch.equal(got, want), (lens, topk, local, init)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens", [[2], [64, 1, 65], [31, 0, 47, 2048], [4096], [4097, 130], [8192], [8193], [16384], [16385], [32768], [32769]])
def test_same_words_as_apart(lens, dtype):
    gen = torch.Generator(device="cuda").manual_seed(sum(lens))
    hk = 2 if sum(lens) < 9000 else 1
    r = lambda heads: torch.randn(sum(lens), heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = r(16 * hk), r(hk), r(hk)
    for topk, local, init in ((16, 1, 1), (0, 2, 1), (64, 31, 1), (300, 0, 0), (3, 4, 2)):
        both(q, k, v, lens, topk, local, init)
    both(torch.zeros_like(q), k, v, lens, 8, 1, 1)                 # equal scores
    both(q * 30, k, v, lens, 8, 1, 1)                              # nearly all of them zero


@pytest.mark.parametrize("group, lens, hk", [(1, [700, 4300], 3), (2, [700, 4300], 3), (4, [700, 4300], 3), (8, [700, 4300], 3), (8, [16384], 1), (8, [16385], 1), (8, [32768], 1),
                                             (2, [16385, 300], 1), (4, [32768], 1)])
def test_groups(group, lens, hk):
    gen = torch.Generator(device="cuda").manual_seed(group)
    r = lambda heads: torch.randn(sum(lens), heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    both(r(hk * group), r(hk), r(hk), lens, 12, 3, 1)
