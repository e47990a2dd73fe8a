"""Max-pooling of Stage-1 scores onto 64-token key blocks.

Operator interface of infllm_v2/max_pooling_1d.py:4-46 (fixed length) and :49-137 (packed).
Forced blocks (the first ``init_blocks`` and the query's own block plus ``local_blocks`` before
it) come out as +inf, an empty window as -inf.
"""
from __future__ import annotations

import torch

from . import _lib


def max_pooling_1d(input: torch.Tensor, cache_len: int, local_blocks: int, init_blocks: int,
                   block_size: int = 64, stride: int = 16) -> torch.Tensor:
    """input ``(num_heads, q_len, k_len)`` fp16/bf16 -> ``(num_heads, q_len, ceil((q_len+cache_len)/block_size))``."""
    assert input.dtype == torch.float16 or input.dtype == torch.bfloat16
    assert input.dim() == 3, f"Expected 3D input, got {input.dim()}D"
    return _lib.host.max_pooling_1d(input, cache_len, local_blocks, init_blocks, block_size, stride)


def max_pooling_1d_varlen(input: torch.Tensor, cu_seqlens_q: torch.Tensor, cu_seqlens_k: torch.Tensor,
                          cache_lens: torch.Tensor, max_seqlen_q: int, max_seqlen_k: int, local_blocks: int,
                          init_blocks: int, block_size: int = 64, stride: int = 16,
                          max_cache_len: int | None = None) -> torch.Tensor:
    """Packed variant: input ``(num_heads, total_q, max_seqlen_k)``; ``cache_lens`` int32 per sequence.

    Output ``(num_heads, total_q, ceil((max_seqlen_q + max(cache_lens)) / block_size))``.  Passing
    ``max_cache_len`` (an extra, optional argument) avoids the one host read of ``cache_lens``.
    """
    assert input.dtype == torch.float16 or input.dtype == torch.bfloat16
    assert cu_seqlens_q.dtype == torch.int32
    assert cu_seqlens_k.dtype == torch.int32
    assert cache_lens.dtype == torch.int32
    assert input.dim() == 3, f"Expected 3D input, got {input.dim()}D"
    batch = cu_seqlens_q.shape[0] - 1
    assert input.shape[2] == max_seqlen_k, f"max_k mismatch: {input.shape[2]} vs {max_seqlen_k}"
    assert cache_lens.shape[0] == batch, f"cache_lens batch size mismatch: {cache_lens.shape[0]} vs {batch}"
    if max_cache_len is None:
        max_cache_len = int(cache_lens.max().item()) if batch > 0 else 0
    return _lib.host.max_pooling_1d_varlen(input, cu_seqlens_q, cu_seqlens_k, cache_lens, max_seqlen_q, local_blocks, init_blocks,
                                           block_size, stride, max_cache_len)
