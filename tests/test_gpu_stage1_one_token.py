"""Stage 1 in launches of few workgroups, whose wavefronts take one token each (two in groups of 8 heads and fewer): scores and pooled scores are,
bit for bit, those of the same sequences among so many copies that the launch takes twice as many tokens to a wavefront.  Lengths around the 8, 16 and
32 tokens of a workgroup and the 64 keys of a tile.  The mask words, too, are the same among copies; how many tokens a selecting wavefront takes depends on the
longest sequence alone (test_gpu_stage1_selecting_forms.py)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype, hk, group, lens", [
    (torch.bfloat16, 1, 16, [2]), (torch.bfloat16, 2, 16, [15, 16, 17]), (torch.float16, 1, 16, [1, 0, 9, 1040]), (torch.bfloat16, 1, 4, [1087]),
    (torch.bfloat16, 2, 16, [2049]), (torch.float16, 1, 8, [130, 4096]), (torch.bfloat16, 1, 16, [4097]), (torch.bfloat16, 1, 16, [5999]),
    (torch.bfloat16, 2, 8, [2, 31, 33]), (torch.float16, 1, 2, [8333]), (torch.bfloat16, 1, 1, [4163, 7])])
def test_as_among_many(dtype, hk, group, lens):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(sum(lens))
    r = lambda heads: torch.randn(sum(lens), heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = r(hk * group), r(hk), r(hk)
    longest = max(lens)
    tokens = 16 if group == 16 else 32
    copies = 385 // (-(-longest // tokens) * len(lens) * hk) + 1       # more than 384 workgroups of the larger kind
    cu = lambda n: torch.tensor(np.cumsum([0] + lens * n), dtype=torch.int32, device="cuda")

    def run(n):
        qn, kn, vn, c = q.repeat(n, 1, 1), k.repeat(n, 1, 1), v.repeat(n, 1, 1), cu(n)
        (fine, cu_f), (coarse, cu_c) = ops.compress_keys(kn, c, longest, 32, 16), ops.compress_keys(kn, c, longest, 128, 64)
        most = max(1, (longest - 32) // 16 + 1)
        held = torch.zeros(len(lens) * n, dtype=torch.int32, device="cuda")
        out = [ops.infllmv2_attn_stage1(qn, fine, coarse, c, cu_f, cu_c, longest, most, causal=causal) for causal in (True, False)]
        out += [ops.infllmv2_attn_stage1_pooled(qn, fine, coarse, c, cu_f, cu_c, longest, most, 3, 1, cache_lens=held, max_cache_len=0, causal=causal)
                for causal in (True, False)]
        out += [_lib.host.select_mask(qn, kn, vn, c, longest, topk, 2, 1, 128 ** -0.5, 32, 16, 64)[1] for topk in (5, 16, 64)]
        return [t[:, :sum(lens)] for t in out]

    for few, many in zip(run(1), run(copies)):
        assert torch.equal(few, many)
