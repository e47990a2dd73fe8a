"""Selecting Stage 1 up to 10 240 tokens (one token to a wavefront) and beyond (two, in groups of 16 heads): a sequence's mask words are the same bits alone, in a launch of one form, and
beside a sequence that puts the launch in the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype, hk, group, length", [(torch.bfloat16, 2, 16, 2049), (torch.float16, 1, 16, 4097), (torch.bfloat16, 1, 16, 10240), (torch.bfloat16, 1, 16, 8191),
                                                      (torch.bfloat16, 2, 8, 6001), (torch.float16, 1, 4, 10240), (torch.bfloat16, 1, 16, 777)])
def test_alone_and_beside_a_longer_sequence(dtype, hk, group, length):
    from infllmv2_cuda_impl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(length)
    longer = 10241
    r = lambda heads: torch.randn(length + longer, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = r(hk * group), r(hk), r(hk)
    cu = lambda *at: torch.tensor(at, dtype=torch.int32, device="cuda")
    for topk in [n for n in (5, 12, 16, 64) if n < (length + 63) // 64]:         # else a row takes every column there is, which are more beside the longer one
        pick = lambda n, c, longest: _lib.host.select_mask(q[:n], k[:n], v[:n], c, longest, topk, 2, 1, 128 ** -0.5, 32, 16, 64)[1]
        alone, beside = pick(length, cu(0, length), length), pick(length + longer, cu(0, length, length + longer), longer)
        words = alone.shape[2]
        assert torch.equal(alone, beside[:, :length, :words])
        assert not beside[:, :length, words:].any()
