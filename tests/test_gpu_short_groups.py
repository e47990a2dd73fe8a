"""Stage-2 forward at the ends of sequences: a group of eight tokens that holds four or fewer shares each token's blocks out to 8, 4 or 2
wavefronts and merges their results.  Every number of tokens in the last group, rows of one and two mask words, rows with fewer blocks than
sharing wavefronts, a masked row without any key.  Against the numpy oracle with the tolerances of the forward tests."""
import numpy as np
import pytest
import torch

from oracle import infllmv2_oracle as O
from conftest import bf16_np
from test_gpu_stage2_fwd import check
from test_gpu_hybrid_walk import window_case

pytestmark = pytest.mark.gpu

CASES = [([8 + r, r], [8 + r, 600 + r], 2, 3, 4) for r in range(1, 8)] + [([1], [5000], 1, 4, 9), ([3, 2], [4500, 70], 2, 5, 6),
                                                                          ([66, 12], [2, 3], 2, 1, 1)]


@pytest.mark.parametrize("sq,sk,Hk,window,scattered", CASES)
def test_last_group(sq, sk, Hk, window, scattered):
    import infllmv2_cuda_impl_amd as ops
    dev = torch.device("cuda:0")
    q, k, v, cu_q, cu_k, idx = window_case(5, sq, sk, Hk, window, scattered, dev)
    out, lse, _ = ops.infllmv2_attn_varlen_func(q, k, v, cu_q, cu_k, max(sq), max(sk), causal=max(sq) > 1, topk_idx=idx,
                                                return_attn_probs=True)
    words, _ = O.topk_to_uint64(idx.cpu().numpy(), max(sk), 64)
    ref_o, ref_lse = O.stage2_forward(bf16_np(q), bf16_np(k), bf16_np(v), cu_q.cpu().numpy(), cu_k.cpu().numpy(), words, 128 ** -0.5,
                                      max(sq) > 1)
    check(out, lse, ref_o, ref_lse)
