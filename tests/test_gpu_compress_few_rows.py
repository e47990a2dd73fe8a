"""Compressed keys of launches that leave compute units idle: half the rows to a workgroup, and a column to a thread for the wide windows.  A row
is one sum in window order in every form, so a short launch's rows are the bits of the same rows in a launch too long for it, and lie within the
rounding of the mean (2^-8 relative to the largest key, a bf16 half unit in the last place and more) of the oracle's."""
import pytest
import torch

import infllmv2_cuda_impl_amd as ops
from infllmv2_cuda_impl_amd.selection import compress_keys_pair

pytestmark = pytest.mark.gpu


def keys(n, heads, dim, dtype):
    return torch.randn((n, heads, dim), generator=torch.Generator().manual_seed(n), dtype=torch.float32).to(dtype).cuda()


def cu(*lens):
    return torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")


# two heads: 32 799 | 32 800 tokens are the last halved launch of 32 keys every 16 alone and the first that is not, 32 895 | 32 896 of 128 every 64, 10 271 | 10 272 of the pair
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,heads,dim", [(127, 2, 128), (128, 2, 128), (257, 1, 64), (1000, 3, 136), (2048, 2, 128), (10271, 2, 128), (10272, 2, 128), (10300, 2, 128), (32799, 2, 128), (32800, 2, 128), (32895, 2, 128),
                                         (32896, 2, 128)])
@pytest.mark.parametrize("window", [(32, 16), (128, 64), (192, 192), (200, 7), (96, 96), (3, 2)])
def test_rows_of_short_launches(n, heads, dim, window, dtype):
    size, stride = window
    k = keys(n, heads, dim, dtype)
    rows = max(0, (n - size) // stride + 1)
    got, lens = ops.compress_keys(k, cu(n), n, size, stride)
    assert lens.tolist() == [0, rows]
    longest = 200000                                            # the same keys first, in a launch that is sized for far more rows
    far, _ = ops.compress_keys(k, cu(n), longest, size, stride)
    assert torch.equal(got[:rows], far[:rows])
    want = torch.stack([k[j * stride:j * stride + size].double().mean(0) for j in range(min(rows, 40))]) if rows else got[:0].double()
    assert (got[:want.shape[0]].double() - want).abs().max().item() <= 2.0 ** -8 * k.abs().max().item() if rows else True
    other, other_lens = ops.compress_keys(k, cu(n), n, 128, 64)
    a, ca, b, cb = compress_keys_pair(k, cu(n), n, window, (128, 64))
    assert torch.equal(ca, lens) and torch.equal(cb, other_lens)
    assert torch.equal(a[:rows], got[:rows]) and torch.equal(b[:int(other_lens[-1])], other[:int(other_lens[-1])])
