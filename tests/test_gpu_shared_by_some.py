"""Stage-2 forward and dQ of groups of 8 tokens whose blocks are selected by any number of the rows, one to all eight: the group walks together what five or more
of them select, and rows skip what is not theirs.  Against fp32 attention; a row's blocks at its own last key, partial groups and several mask words included."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(700, 16, 0), (64 * 70 + 3, 16, 200), (1300, 4, 0), (64 * 65, 8, 61)]


def inputs(S, group, tail, dtype):
    import infllmv2_cuda_impl_amd as ops
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
    return q, k, v, rand(C, Hk * group), pos, chosen, mask


def attend(q, k, v, mask):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    C, S, Hk = q.shape[0], k.shape[0], k.shape[1]
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32, device="cuda")
    return attend_varlen(q, k, v, cu(C), cu(S), C, S, causal=True, topk_idx=torch.zeros(Hk, C, 64, dtype=torch.int32, device="cuda"), block_mask=mask)


def reference(q, k, v, pos, chosen, h, rows):
    """fp32 attention of some query rows of KV head h."""
    group, S = q.shape[1] // k.shape[1], k.shape[0]
    seen = chosen[h, rows].repeat_interleave(64, 1)[:, :S] & (torch.arange(S, device="cuda")[None] <= pos[rows, None])
    s = torch.einsum("tgd,sd->tgs", q[rows, group * h:group * (h + 1)], k[:, h]) * 128 ** -0.5
    return torch.softmax(s.masked_fill(~seen[:, None], float("-inf")), -1) @ v[:, h]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S, group, tail", CASES)
def test_forward(S, group, tail, dtype):
    q, k, v, _, pos, chosen, mask = inputs(S, group, tail, dtype)
    with torch.no_grad():
        out = attend(q, k, v, mask)
    for h in range(k.shape[1]):
        for a in range(0, q.shape[0], 512):
            rows = slice(a, min(q.shape[0], a + 512))
            err = (out[rows, group * h:group * (h + 1)].float() - reference(q.float(), k.float(), v.float(), pos, chosen, h, rows)).abs()
            assert err.max() <= 2e-2 and err.mean() <= 1e-3, (h, a)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S, group, tail", [CASES[0], CASES[2], CASES[3]])
def test_backward(S, group, tail, dtype):
    q, k, v, dout, pos, chosen, mask = inputs(S, group, tail, dtype)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    got = torch.autograd.grad(attend(*leaves, mask), leaves, dout)
    wide = [t.float().requires_grad_(True) for t in (q, k, v)]
    ref = torch.cat([reference(*wide, pos, chosen, h, slice(0, q.shape[0])) for h in range(k.shape[1])], 1)
    for name, a, b in zip(("dq", "dk", "dv"), got, torch.autograd.grad(ref, wide, dout.float())):
        err, scale = (a.float() - b).abs(), max(1.0, float(b.abs().max()))
        assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale, name
