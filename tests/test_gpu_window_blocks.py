"""The blocks of a window, written directly, are those that pooling marks +inf on a score tensor without columns and the selection then takes: bit for
bit, indices and mask, over batches, positions, rows at the edges of blocks and of mask words, and windows longer than the sequence."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # lengths, positions (None: prefill), heads, local, init, block
    ([1], None, 1, 4, 1, 64), ([64, 65, 1, 4096], None, 2, 0, 0, 64), ([4097], None, 4, 70, 3, 64), ([300, 5000], None, 1, 31, 1, 64), ([130], None, 2, 2, 5, 64),
    ([1, 1, 1], [0, 4095, 4096], 2, 8, 1, 64), ([1], [100000], 1, 31, 1, 64), ([700, 33], [64, 129], 2, 3, 2, 32), ([2000], None, 1, -1, 2, 64),
]


@pytest.mark.parametrize("lens, positions, heads, local, init, block", CASES)
def test_window_blocks(lens, positions, heads, local, init, block):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    cu = ints([sum(lens[:i]) for i in range(len(lens) + 1)])
    held, most = (ints([0] * len(lens)), 0) if positions is None else (ints(positions), max(positions))
    idx, mask = _lib.host.window_blocks(heads, sum(lens), cu, None if positions is None else held, max(lens), most, local, init, block)
    scores = torch.empty((heads, sum(lens), 0), dtype=torch.bfloat16, device="cuda")
    pooled = ops.max_pooling_1d_varlen(scores, cu, torch.zeros_like(cu), held, max(lens), 0, local, init, block_size=block, stride=16, max_cache_len=most)
    want_idx, want_mask = ops.topk_blocks(pooled, init + local + 1, return_mask=True, by_index=True, drop_unreachable=True)
    assert torch.equal(idx, want_idx) and torch.equal(mask, want_mask)
