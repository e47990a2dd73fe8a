"""Stage-2 forward of groups of 8 tokens whose blocks are selected by any number of the rows, one to all eight: the group walks together what five or more
of them select, and rows skip what is not theirs.  Against fp32 attention; a row's blocks at its own last key, partial groups and several mask words included."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S, group, tail", [(700, 16, 0), (64 * 70 + 3, 16, 200), (1300, 4, 0), (64 * 65, 8, 61)])
def test_every_count(S, group, tail, dtype):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    Hk, C, nblk = 2, tail or S, (S + 63) // 64
    gen = torch.Generator(device="cuda").manual_seed(S)
    rand = lambda n, heads: torch.randn(n, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = rand(C, Hk * group), rand(S, Hk), rand(S, Hk)
    pos, at = torch.arange(S - C, S, device="cuda"), torch.arange(nblk, device="cuda")
    # block j of group G is selected by (j + G) % 9 of its rows, other rows for every block; all rows select their own last block
    row = torch.arange(C, device="cuda") % 8
    count = (at[None] + torch.arange(C, device="cuda")[:, None] // 8) % 9
    chosen = ((row[:, None] * 3 + at[None] * 5) % 8 < count) | (at[None] == pos[:, None] // 64)
    chosen = (chosen & (at[None] <= pos[:, None] // 64))[None].repeat(Hk, 1, 1)
    chosen[1] ^= (torch.rand(C, nblk, generator=gen, device="cuda") < 0.1) & (at[None] < pos[:, None] // 64)
    mask = ops.blockmask_to_uint64(chosen.contiguous())[0]
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32, device="cuda")
    with torch.no_grad():
        out = attend_varlen(q, k, v, cu(C), cu(S), C, S, causal=True, topk_idx=torch.zeros(Hk, C, 64, dtype=torch.int32, device="cuda"), block_mask=mask)
    for h in range(Hk):
        for a in range(0, C, 512):
            rows = slice(a, min(C, a + 512))
            seen = chosen[h, rows].repeat_interleave(64, 1)[:, :S] & (torch.arange(S, device="cuda")[None] <= pos[rows, None])
            s = torch.einsum("tgd,sd->tgs", q[rows, group * h:group * (h + 1)].float(), k[:, h].float()) * 128 ** -0.5
            ref = torch.softmax(s.masked_fill(~seen[:, None], float("-inf")), -1) @ v[:, h].float()
            err = (out[rows, group * h:group * (h + 1)].float() - ref).abs()
            assert err.max() <= 2e-2 and err.mean() <= 1e-3, (h, a)
